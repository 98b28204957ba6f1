"""GPU parity of the kernels beside the Coulomb family (regularized
Yukawa, atan, sin-over-r, MQ, RBS-u, RBS-v, the reference's user-kernel
example) through the C ABI against the CPU oracle, which is bit-equal to
the reference's compiled kernels (test_oracle_kernels.py).  They run in
FP64 whatever precision is asked.  Bar: relative L2 <= 1e-12.
"""
import numpy as np
import pytest

from tests.helpers import KP_OTHER, other_combos, rel_l2, uniform_cube

pytestmark = pytest.mark.gpu

TOL_FP64 = 1e-12


@pytest.fixture(scope="module")
def bt():
    import barytree_amd
    barytree_amd.lib()
    return barytree_amd


@pytest.mark.parametrize("ct,k,s", other_combos())
def test_other_kernels_small(bt, oracle_mod, ct, k, s):
    print(f"case ct={ct} k={k} s={s}", flush=True)
    t, src = uniform_cube(3000, 2500, seed=700 + 10 * ct + k)
    args = (k, KP_OTHER[k], s, 1, ct, 0.7, 4, 60, 50)
    ref = oracle_mod.treecode(*t, *src, *args)
    got = bt.solve(t, src, *args)
    err = rel_l2(ref, got)
    print(f"relL2={err:.3e}", flush=True)
    assert err <= TOL_FP64
    # the mixed precision request runs these kernels in FP64
    assert np.array_equal(got, bt.solve(t, src, *args, precision=bt.PRECISION_MIXED))


@pytest.mark.parametrize("k", [4, 8, 10, 11, 12])
def test_other_kernels_cc_lists(bt, oracle_mod, k):
    print(f"case k={k}", flush=True)
    t, src = uniform_cube(12000, 12000, seed=17)
    args = (k, KP_OTHER[k], 1, 1, 3, 0.8, 2, 30, 30)
    ref = oracle_mod.treecode(*t, *src, *args)
    st = oracle_mod.last_stats()
    assert st["num_cc"] > 0
    assert rel_l2(ref, bt.solve(t, src, *args)) <= TOL_FP64


def test_other_kernels_direct_sample(bt, oracle_mod):
    t, src = uniform_cube(3000, 3000, seed=4)
    idx = np.arange(0, 3000, 7)
    for k, s in [(4, 2), (5, 1), (9, 1), (10, 1)]:
        with bt.Plan(t, src, k, KP_OTHER[k], s, 1, 1, 0.7, 4, 60, 60) as p:
            got = p.direct_sample(idx)
        ref = oracle_mod.direct(*[a[idx] for a in t], *src, k, KP_OTHER[k], s)
        assert rel_l2(ref, got) <= TOL_FP64


def test_other_kernels_reject_learned_degrees(bt):
    t, src = uniform_cube(2000, 2000, seed=2)
    with bt.Plan(t, src, 8, [1.5], 1, 1, 1, 0.7, 3, 60, 60) as p:
        with pytest.raises(RuntimeError, match="per-pair degrees"):
            p.set_pair_degrees(np.full(p.num_pairs(), 3))


@pytest.mark.parametrize("k", [4, 8, 12])
@pytest.mark.parametrize("ct,leaf", [(1, 300), (2, 33), (3, 130), (1, 7)])
def test_other_kernels_targets_equal_sources(bt, oracle_mod, k, ct, leaf):
    """Targets equal to the sources: the near field evaluates each pair of
    two leaves once for both particles.  Two particles at one point (the
    regularized kernel does not skip them, the others do), one leaf pass with
    a remainder, the one-directional form, and the mixed precision request,
    which runs in FP64."""
    rng = np.random.default_rng(10 * ct + k)
    x, y, z, q = (rng.uniform(-1, 1, 5000) for _ in range(4))
    x[40], y[40], z[40] = x[41], y[41], z[41]
    t, src = (x.copy(), y.copy(), z.copy(), q.copy()), (x, y, z, q, np.ones(5000))
    args = (k, KP_OTHER[k], 1, 1, ct, 0.7, 3, leaf, leaf)
    ref = oracle_mod.treecode(*t, *src, *args)
    with bt.Plan(t, src, *args) as p:
        st = p.stats()
        assert st["sym_ptwise"] > 0.5 * st["pp_ptwise"] and st["sym_evals"] < st["sym_ptwise"], st
        got = p.execute()
        assert np.array_equal(got, p.execute())
        p.set_symmetric(False)
        assert p.stats()["sym_ptwise"] == 0
        one = p.execute()
    assert rel_l2(ref, got) <= TOL_FP64 and rel_l2(ref, one) <= TOL_FP64
    assert np.array_equal(got, bt.solve(t, src, *args, precision=bt.PRECISION_MIXED))


@pytest.mark.parametrize("k,s", [(2, 1), (2, 2), (4, 1), (12, 1)])
@pytest.mark.parametrize("ct,leaf", [(1, 300), (2, 33), (3, 130), (1, 7)])
def test_growing_exponentials_targets_equal_sources(bt, oracle_mod, k, s, ct, leaf):
    """A negative rate (e^{|k| r}) with targets equal to the sources, in
    leaves whose counts are not multiples of 8: the places that fill the last
    step of a leaf must not bring an overflow in (zero times infinity)."""
    print(f"case k={k} s={s} ct={ct} leaf={leaf}", flush=True)
    rng = np.random.default_rng(ct + 10 * k)
    x, y, z, q = (rng.uniform(-1, 1, 3001) for _ in range(4))
    src = (x, y, z, q, rng.uniform(0.5, 1.5, 3001))
    t = tuple(a.copy() for a in src[:4])
    for rate in (-0.5, -20.0):
        args = (k, [rate, 0.1] if k == 4 else [rate], s, 1, ct, 0.7, 3, leaf, leaf)
        got = bt.solve(t, src, *args)
        assert bt.last_stats()["sym_ptwise"] > 0
        assert rel_l2(oracle_mod.treecode(*t, *src, *args), got) <= TOL_FP64, rate


@pytest.mark.parametrize("k,kp", [(8, [1.5]), (1, [0.5]), (2, [0.5]), (12, [0.5])])
def test_leaves_smaller_than_their_coordinates_spacing(bt, oracle_mod, k, kp):
    """Leaves far from the origin whose extent lies below the spacing of
    doubles at one of their coordinates: a place that fills a leaf's last step
    must not fall on a particle there."""
    y = np.array([-1.0, 0.0, 1.0, 400.0, 401.0, 402.0, 407.0]) * 1e-12
    x, z = np.full(7, 1.0e6), np.zeros(7)
    src = (x, y, z, np.arange(1.0, 8.0), np.ones(7))
    t = tuple(a.copy() for a in src[:4])
    args = (k, kp, 1, 1, 1, 0.7, 3, 2, 2)
    got = bt.solve(t, src, *args)
    assert bt.last_stats()["sym_ptwise"] > 0
    assert rel_l2(oracle_mod.treecode(*t, *src, *args), got) <= TOL_FP64


@pytest.mark.parametrize("k", [2, 4, 8, 12])
@pytest.mark.parametrize("same", [False, True])
def test_a_nan_rate_gives_nan(bt, k, same):
    """A kernel parameter that is not a number is not taken for a finite
    rate: every potential is NaN."""
    t, src = uniform_cube(700, 600, seed=k)
    if same:
        t = [a.copy() for a in src[:4]]
    got = bt.solve(t, src, k, [np.nan, 0.1] if k == 4 else [np.nan], 1, 1, 1, 0.7, 3, 100, 100)
    assert np.all(np.isnan(got))
