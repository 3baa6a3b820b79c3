"""The append's quotients without IEEE division (csrc/kv_quant.h), restated with
exact fused multiply-adds on the CPU: an element's x / scale by a reciprocal and
one residual step rounds to the same code as the IEEE quotient does, and amax / 7,
/ 15 and / 127 are the IEEE quotients themselves.  A sample of what was compared
once in full (every mantissa of the scale): 1000 scales, reciprocals up to 2 ulps
off, every rounding threshold and the values within 4 ulps of it."""
import numpy as np
import pytest

F, L = np.float32, np.longdouble


def fma(a, b, c):
    """a b + c rounded once: the product is exact in 64 bits of mantissa."""
    return (a.astype(L) * b.astype(L) + c.astype(L)).astype(F)


def ulps(x, n):
    return (x.view(np.int32) + np.int32(n)).view(F)


@pytest.mark.parametrize("rcp_off", [-2, -1, 0, 1, 2])
def test_codes_are_those_of_the_ieee_quotient(rcp_off):
    g = np.random.default_rng(rcp_off + 10)
    scale = (g.integers(0, 1 << 23, 1000, dtype=np.int32) | np.int32(127 << 23)).view(F)
    scale[:4] = F(1), ulps(F([2]), -1)[0], ulps(F([1]), 1)[0], F(1.5)
    y0 = ulps((L(1) / scale.astype(L)).astype(F), rcp_off)
    y = fma(fma(-scale, y0, np.ones_like(y0)), y0, y0)
    half = np.arange(1, 129, dtype=F) - F(0.5)
    at = (half[None, :] * scale[:, None]).astype(F)                    # the thresholds
    s, r = (np.broadcast_to(a[:, None], at.shape) for a in (scale, y))
    for off in range(-4, 5):
        x = ulps(np.ascontiguousarray(at), off)
        q0 = (x * r).astype(F)
        t = fma(fma(-q0, s, x), r, q0)
        assert np.array_equal(np.floor(t + F(0.5)), np.floor((x / s).astype(F) + F(0.5))), off


@pytest.mark.parametrize("c", [7, 15, 127])
def test_constant_divisors_are_exact_for_every_mantissa(c):
    for part in np.split(np.arange(1 << 23, dtype=np.int32), 16):
        x = (part | np.int32(127 << 23)).view(F)
        rc = np.full_like(x, F(1) / F(c))
        q0 = (x * rc).astype(F)
        got = fma(fma(-q0, np.full_like(x, F(c)), x), rc, q0)
        assert np.array_equal(got, (x / F(c)).astype(F))
