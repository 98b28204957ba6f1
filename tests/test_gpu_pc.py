"""FP64 particle targets against source clusters (csrc/bt_pc.hip): every grid
size, target batches around a tile of 128 targets, every kernel of r alone.
Bar: the plain-mode bar against the CPU oracle, relative L2 <= 1e-12."""
import numpy as np
import pytest

from tests.helpers import KP, rel_l2, uniform_cube

pytestmark = pytest.mark.gpu

TOL_FP64 = 1e-12


@pytest.fixture(scope="module")
def bt():
    import barytree_amd
    barytree_amd.lib()
    return barytree_amd


@pytest.mark.parametrize("deg", range(1, 13))
def test_every_grid_size(bt, oracle_mod, deg):
    """2 to 13 points per dimension: pencils that leave the four waves
    unequal shares, and clusters staged in several parts (above 1024
    points)."""
    leaf = max(20, (deg + 1) ** 3 + 10)
    rng = np.random.default_rng(deg)
    src = [rng.uniform(-1, 1, 6 * leaf) for _ in range(4)] + [rng.uniform(0.5, 1.5, 6 * leaf)]
    t = [rng.uniform(2.5, 3.0, 300) for _ in range(3)] + [rng.uniform(-1, 1, 300)]
    for k, s in ((1, 1), (1, 2), (2, 1), (3, 2)):
        args = (k, KP[k][s], s, 1, 1, 0.8, deg, leaf, 150)
        ref = oracle_mod.treecode(*t, *src, *args)
        assert oracle_mod.last_stats()["num_pc"] > 0
        assert rel_l2(ref, bt.solve(t, src, *args)) <= TOL_FP64, (k, s)


@pytest.mark.parametrize("m", [1, 63, 65, 127, 128, 129, 400])
def test_target_tiles(bt, oracle_mod, m):
    rng = np.random.default_rng(m)
    t = [rng.uniform(2.5, 3.0, m) for _ in range(3)] + [rng.uniform(-1, 1, m)]
    _, src = uniform_cube(3000, 1, seed=9)
    for k, kp, s in ((1, [0.5], 2), (2, [0.5], 2), (3, [0.05], 1), (4, [0.5, 0.1], 1), (4, [0.5, 0.1], 2),
                     (8, [1.5], 1), (12, [0.5], 1)):
        args = (k, kp, s, 1, 1, 0.8, 4, 200, 1000)
        ref = oracle_mod.treecode(*t, *src, *args)
        assert oracle_mod.last_stats()["num_pc"] > 0
        got = bt.solve(t, src, *args)
        assert rel_l2(ref, got) <= TOL_FP64, (k, s)
        if k > 3:  # these run in FP64 in either precision
            assert np.array_equal(got, bt.solve(t, src, *args, precision=bt.PRECISION_MIXED))


def test_sums_do_not_depend_on_the_tiles(bt):
    """The same batch with other targets before it (other tiles, other
    launch order) gives the same bits."""
    rng = np.random.default_rng(3)
    t = [rng.uniform(2.5, 3.0, 200) for _ in range(3)] + [rng.uniform(-1, 1, 200)]
    far = [rng.uniform(-3.0, -2.5, 500) for _ in range(3)] + [rng.uniform(-1, 1, 500)]
    _, src = uniform_cube(3000, 1, seed=9)
    args = (1, [0.5], 1, 1, 1, 0.8, 4, 200, 1000)
    both = [np.concatenate([f, a]) for f, a in zip(far, t)]
    alone = bt.solve(t, src, *args)
    assert np.array_equal(bt.solve(both, src, *args[:-1], 600)[500:], alone)
