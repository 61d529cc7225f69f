"""The Gumbel sampler's bound (rl_gumbel_kernels.hpp, gumbel_bound), as a method: from the high word alone it
is never below the draw's g = -ln(-ln u) by more than the slack of bound_floor (2e-3, less 1e-3 of it for
what is sure), and above it by at most 1e-3 except at the ends of the range, where what is sure is not taken
from it. numpy's f32 logarithm stands in for the hardware's (both within about an ulp)."""
import numpy as np
import pytest


def bound(hi):
    f = np.float32
    with np.errstate(divide="ignore"):
        ta = (f(32) - np.log2(hi.astype(f) + f(1))).astype(f)
        d = ((~hi).astype(f) * f(2.0 ** -32)).astype(f)
        l2e = f(1.44269504088896340736)
        tb = (d * (d * f(0.5) * l2e + l2e)).astype(f)
        t2 = np.where(hi >= np.uint32(0xF8000000), tb, ta)
        return (np.log2(t2).astype(f) * f(-0.69314718055994530942) + f(0.36651292058166432701)).astype(f)


def g_of(hi, lo):
    k = (hi.astype(np.uint64) << np.uint64(21)) | (lo.astype(np.uint64) >> np.uint64(11))
    with np.errstate(divide="ignore"):
        return -np.log(-np.log((k.astype(np.float64) + 0.5) * 2.0 ** -53))


def test_bound_over_the_range_of_the_high_word():
    rng = np.random.default_rng(1)
    ends = np.arange(1 << 17, dtype=np.uint64)
    hi = np.concatenate([rng.integers(0, 1 << 32, 1_000_000, dtype=np.uint64), ends, (1 << 32) - 1 - ends,
                         np.uint64(0xF8000000) + ends - np.uint64(1 << 16)]).astype(np.uint32)
    for lo in (np.zeros_like(hi), np.full_like(hi, 0xFFFFFFFF), rng.integers(0, 1 << 32, hi.size, dtype=np.uint64).astype(np.uint32)):
        g, b = g_of(hi, lo), bound(hi).astype(np.float64)
        assert np.all(b >= g - 5e-4)
        sure = (hi >= np.uint32(0x1000)) & (hi < np.uint32(0xFFFF0000))
        assert np.all(b[sure] <= g[sure] + 1e-3)
    assert bound(np.array([0xFFFFFFFF], np.uint32))[0] == np.inf


# The bound with the logit's share: x inv_tau + bound(hi), inv_tau NaN where 1 / tau overflows in f32 (the
# host's rule). An element may be skipped only where its bound is below bound_floor of its own value:
# below any floor that a larger one sets.
@pytest.mark.parametrize("tau", [0.0, 1e-45, 1e-40, 2.9387e-39, 2.9388e-39, 1e-37, 1e-20, 0.6, 3.0, 1e20, 3e38])
def test_no_element_is_skipped_beside_itself(tau):
    f = np.float32
    rng = np.random.default_rng(2)
    tau = f(tau)
    hi = rng.integers(1 << 16, (1 << 32) - (1 << 16), 200_000, dtype=np.uint64).astype(np.uint32)
    x = (rng.normal(0, 3, hi.size) * 10.0 ** rng.uniform(-44, 30, hi.size)).astype(f)
    x[:1000] = 0.0
    with np.errstate(all="ignore"):
        near_one = (rng.normal(0, 3, hi.size).astype(f) * tau).astype(f)  # quotients of a logit's size
        x[1000:100_000] = near_one[1000:100_000]
        inv = f(1) / tau
        if not np.isfinite(inv):
            inv = f(np.nan)
        z = (x / tau).astype(f)
        a = (z + g_of(hi, np.zeros_like(hi)).astype(f)).astype(f)
        b = (x * inv + bound(hi)).astype(f)
        screen = a - np.maximum(f(1e-3), np.abs(a) * f(2.0 ** -20))
        floor = np.fmin(screen - np.maximum(f(2e-3), np.abs(a) * f(2.0 ** -20)), f(3e38))
    candidate = ~np.isnan(z) & (z > -np.inf)
    assert not np.any(candidate & (b < floor))
