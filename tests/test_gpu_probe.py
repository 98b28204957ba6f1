"""GPU tests of the probe library (libbt_probe.so, barytree_amd.probe): the
VALU issue-cost probe, which prices the near-field kernel's instruction mix
in bench.py, and the accuracy of the FP64 reciprocal square root every FP64
pair kernel uses (csrc/bt_rsq.h)."""
import math

import numpy as np

import pytest

pytestmark = pytest.mark.gpu


def test_probe_valu_costs_are_sane():
    from barytree_amd import probe
    p = probe.probe_valu()
    assert set(p) == set(probe.VALU_KINDS)
    for k, v in p.items():
        # a wave instruction takes between 1 and 64 cycles at 0.5-3 GHz
        assert math.isfinite(v) and 0.3 < v < 130.0, (k, v)
    # transcendentals issue no faster than an FP32 fma
    assert p["exp_f32"] >= 0.9 * p["fma_f32"] and p["rsq_f32"] >= 0.9 * p["fma_f32"]


def test_rsq64_is_within_about_one_ulp():
    """rsq64 against 1/sqrt in extended precision (x87 long double, 64-bit
    significand) over 60 decades, powers of two, values near 1 and the
    squares of the near-field's typical distances."""
    from barytree_amd import probe
    rng = np.random.default_rng(5)
    x = np.concatenate([
        10.0 ** rng.uniform(-30, 30, 200_000),
        2.0 ** np.arange(-200, 201).astype(np.float64),
        1.0 + rng.uniform(-1e-6, 1e-6, 10_000),
        rng.uniform(0.0, 1.0, 100_000) ** 2 + 1e-300,
    ])
    y = probe.rsq64(x)
    ref = 1.0 / np.sqrt(x.astype(np.longdouble))
    assert np.finfo(np.longdouble).nmant >= 63, "needs an extended-precision long double"
    ulps = np.abs(y.astype(np.longdouble) - ref) / np.spacing(ref.astype(np.float64))
    print(f"rsq64: max error {float(ulps.max()):.3f} ulp, mean {float(ulps.mean()):.3f} ulp", flush=True)
    assert float(ulps.max()) <= 1.5
    # zero and infinity give NaN (callers skip coincident points by a select)
    assert np.all(np.isnan(probe.rsq64(np.array([0.0, np.inf]))))


ULP1 = 2.0 ** -52


@pytest.mark.parametrize("k", [1e-6, 0.5, 7.3, 400.0, 0.0, -0.7])
def test_exp_table_form_is_within_two_ulp_and_the_argument_rounding(k):
    """exp_neg against extended precision over [0, 746/k]: table entry (the
    library's exp2, 1 ulp), polynomial, product and scaling stay within two
    ulp, and c's rounding moves k x by a relative 2^-53.  Past the clamp the
    result is 0; where the result is subnormal its spacing is the least
    subnormal."""
    from barytree_amd import probe
    rng = np.random.default_rng(3)
    top = 740.0 / abs(k) if k else 1e3
    x = np.concatenate([rng.uniform(0, top, 200_000), top * 10.0 ** rng.uniform(-18, 0, 200_000),
                        [0.0, top], np.arange(300) * (np.log(2) / 256 / (abs(k) or 1))])
    x = x[abs(k) * x <= 700] if k < 0 else x
    y = probe.exp_neg(k, x).astype(np.longdouble)
    ref = np.exp(-np.longdouble(k) * x.astype(np.longdouble))
    bar = 2 * np.spacing(ref.astype(np.float64)) + np.abs(k * x) * 2.0 ** -53 * ref * 1.01
    assert np.all(np.abs(y - ref) <= bar), float((np.abs(y - ref) / bar).max())
    if k > 0:
        assert np.all(probe.exp_neg(k, np.array([760.0 / k, 1e300, np.inf])) == 0.0)
    if k == 0.0:
        assert np.all(y == 1.0)


@pytest.mark.parametrize("k", [1e-3, 1.5, 300.0, 1e9, 0.0, -2.0])
def test_sin_table_form_is_within_two_ulp_of_one(k):
    """sin_kr against extended precision, to arguments of 1e12 (k = 1e9: its
    own limit, the library beyond it): table, polynomials and product stay
    within 2 ulp of 1, near 0 within 2 ulp of the result.  x87 long double
    reduces its argument with a 66-bit pi, so the reference reduces first
    with pi in two parts."""
    from barytree_amd import probe
    rng = np.random.default_rng(4)
    x = np.concatenate([rng.uniform(0, 10.0, 200_000), 10.0 ** rng.uniform(-12, 3, 100_000), [0.0, 1.0]])
    y = probe.sin_kr(k, x).astype(np.longdouble)
    a = np.longdouble(k) * x.astype(np.longdouble)
    two_pi = np.longdouble("6.283185307179586476925286766559")
    if abs(k) <= 300.0:
        n = np.rint(a / two_pi)
        hi = np.longdouble(6.28318530717958623199592)       # the double
        lo = np.longdouble("2.449293598294706414e-16")
        ref = np.sin((a - n * hi) - n * lo)
        # n hi and a are rounded to 64 bits: 2^-64 of them
        bar = 2 * ULP1 * np.minimum(1.0, np.maximum(np.abs(ref) * 1.0, 2.0 ** -1000)) + np.abs(a) * 2.0 ** -62
        near = np.abs(a) < 1.0
        assert np.all(np.abs(y - ref)[near] <= bar[near]), float((np.abs(y - ref) / bar)[near].max())
        assert np.all(np.abs(y - ref) <= 2 * ULP1 + np.abs(a) * 2.0 ** -62)
    else:
        # long arguments: the same sine as the library's of the rounded product
        assert np.all(np.abs(y) <= 1.0 + 2 * ULP1)
        ref = np.sin((np.float64(k) * x))
        assert np.all(np.abs(y - ref) <= 4 * ULP1 + np.abs(a) * 2.0 ** -52)
    assert np.all(np.isnan(probe.sin_kr(1.5, np.array([np.nan]))))


def test_table_forms_of_a_nan_rate_are_nan():
    """A rate that is not a number gives NaN, as the library's functions do."""
    from barytree_amd import probe
    x = np.array([0.0, 1e-3, 1.0, 1e300, np.inf])
    assert np.all(np.isnan(probe.exp_neg(np.nan, x)))
    assert np.all(np.isnan(probe.sin_kr(np.nan, x)))
