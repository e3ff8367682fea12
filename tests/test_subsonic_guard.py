"""The sampler's certainty test (surely_below, hfv_physics.hpp): where it holds, the sign of v - a y for the computed
root or power y is the sign of -a.  Restated with numpy in the kernel's operation order, FP32 and FP64, over random
states and states next to the decision."""
import numpy as np
import pytest


def surely_below(v, a, num, den):
    t = v.dtype.type
    lim, x = np.abs(a) * num, np.abs(v) * den
    return (x < t(0.9999) * lim) & (lim > t(1e-30)) & (lim < t(1e30)) & (x < t(1e30))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("gamma", [1.0001, 1.1, 1.4, 5.0 / 3.0, 3.0])
def test_certain_signs(dtype, gamma):
    rng = np.random.default_rng(11)
    n = 400_000
    t = dtype
    e = t(0.5 * (gamma - 1.0) / gamma)
    span = 30.0 if dtype == np.float64 else 12.0
    p = np.exp(rng.uniform(-span, span, n)).astype(t)
    a = (np.exp(rng.uniform(-span, span, n)) * rng.choice([-1.0, 1.0], n)).astype(t)
    near = 1.0 + rng.choice([-1.0, 1.0], n) * np.exp(rng.uniform(np.log(1e-9), 0.0, n))
    with np.errstate(all="ignore"):
        # rarefactions: star.p / p in (0, 1], many of them next to 1
        q = (1.0 - np.exp(rng.uniform(np.log(1e-16), np.log(1.0 - 1e-6), n))).astype(t)
        ps = np.minimum(p * q, p)
        v = (a.astype(np.float64) * (ps / p) * near).astype(t)
        sure = surely_below(v, a, ps, p)
        tail = v - a * np.power(ps / p, e)
        assert sure.mean() > 0.2
        assert np.array_equal(np.sign(tail[sure]), -np.sign(a[sure]))
        # shocks: star.p / p above 1
        ratio = (1.0 + np.exp(rng.uniform(np.log(1e-16), np.log(1e6), n))).astype(t)
        v = (a.astype(np.float64) * near).astype(t)
        sure = surely_below(v, a, t(1), t(1))
        speed = v - a * np.sqrt(t(0.5) * t((gamma + 1.0) / gamma) * ratio + e)
        assert sure.mean() > 0.2
        assert np.array_equal(np.sign(speed[sure]), -np.sign(a[sure]))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_edges_are_not_certain(dtype):
    t = dtype
    for v, a, num, den in ((0, 0, 1, 1), (1, 1, 1, 1), (np.nan, 1, 1, 1), (0, np.nan, 1, 1), (0, 1, np.nan, 1),
                           (0, 1, -1, -1), (0, 1, 0, 0), (0, np.inf, 1, 1), (np.inf, 1, 1, 1), (0, 1e-20, 1e-20, 1)):
        with np.errstate(all="ignore"):
            assert not surely_below(t(v), t(a), t(num), t(den)), (v, a, num, den)
