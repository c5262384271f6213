"""The quotient and square root steps of the integration (div_nr, recip_nr and
sqrt_nr in dynamap_amd/csrc/volume.hip) against correct rounding, restated in
extended precision: every mantissa of the divisor and of the radicand, with the
hardware's reciprocal and reciprocal square root taken as the rounded value and
one unit in the last place to either side (v_rcp_f32 and v_rsq_f32 are within
one)."""
import numpy as np
import pytest

F, X = np.float32, np.longdouble
pytestmark = pytest.mark.skipif(np.finfo(X).nmant < 63, reason="needs an extended long double")
N = 1 << 23


def fma(a, b, c):
    # a * b is exact in 64 bits; the sum is rounded once to 64 and once to 24,
    # which differs from one rounding only on ties that these values do not meet
    return (a.astype(X) * b.astype(X) + c.astype(X)).astype(F)


def ulp(x, n):
    return (x.view(np.int32) + np.int32(n)).view(F)


def mantissas(seed, lo, hi):
    e = np.random.default_rng(seed + 20).integers(lo, hi, N)
    return np.ldexp((1 + np.arange(N, dtype=np.float64) / N), e).astype(F)


@pytest.mark.parametrize("off", [-1, 0, 1])
def test_quotient(off):
    rng = np.random.default_rng(off + 5)
    b = mantissas(off, -40, 41)
    a = rng.permutation(mantissas(off + 3, -40, 41)) * rng.choice(np.array([-1, 1], F), N)
    r = ulp((X(1) / b.astype(X)).astype(F), off)
    r = fma(fma(-b, r, np.ones(1, F)), r, r)
    q = a * r
    q = fma(fma(-q, b, a), r, q)
    q = fma(fma(-q, b, a), r, q)
    np.testing.assert_array_equal(q, a / b)


# Weights: divisors 1 to 256, the sums of any mantissa.
def test_quotient_by_weights():
    rng = np.random.default_rng(2)
    b = rng.integers(1, 257, N).astype(F)
    a = rng.permutation(mantissas(7, -40, 8))
    r = ulp((X(1) / b.astype(X)).astype(F), 0)
    r = fma(fma(-b, r, np.ones(1, F)), r, r)
    q = a * r
    q = fma(fma(-q, b, a), r, q)
    q = fma(fma(-q, b, a), r, q)
    np.testing.assert_array_equal(q, a / b)


@pytest.mark.parametrize("odd", [0, 1])
@pytest.mark.parametrize("off", [-1, 0, 1])
def test_square_root(off, odd):
    x = mantissas(off + 11, -40, 41)
    x = np.ldexp(np.frexp(x)[0], 2 * (np.frexp(x)[1] // 2) + odd).astype(F)
    r = ulp((X(1) / np.sqrt(x.astype(X))).astype(F), off)
    g, h = x * r, F(0.5) * r
    e = fma(-h, g, np.full(1, 0.5, F))
    g, h = fma(g, e, g), fma(h, e, h)
    np.testing.assert_array_equal(fma(fma(-g, g, x), h, g), np.sqrt(x))


# The numerator may be far smaller than the stated range where the quotient is
# added to the principal point: a pixel is the same for every quotient below half
# a unit in the last place of any pixel coordinate, and 0 stays 0.
@pytest.mark.parametrize("c", [0.0, -0.5, 0.5, 319.5])
def test_tiny_numerators_keep_the_pixel(c):
    half = np.uint32(0x3effffff).view(F)
    a = np.concatenate([F([0.0, 1e-45, 1e-40, 1e-38]), np.ldexp(1.0, np.arange(-149, -39)).astype(F)])
    a = np.concatenate([a, -a])
    for z in F([2.0 ** -14, 0.3, 5.0, 2.0 ** 20]):
        r = (X(1) / X(z)).astype(F)
        q = a * r
        q = fma(fma(-q, np.full(1, z), a), np.full(1, r), q)
        q = fma(fma(-q, np.full(1, z), a), np.full(1, r), q)
        s = (q + F(c)) + half
        x = (a / z) + F(c)
        want = np.where(x > -0.5, np.floor(x.astype(np.float64) + 0.5), -1)  # half away from zero, all below as one
        np.testing.assert_array_equal(np.where(s >= 0, np.trunc(s), -1), want)
