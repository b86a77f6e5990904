"""The apply of add_rms_norm_stats in fp32 operations (csrc/add_rms_norm.hip) against the
fp64 model: rd(x * rstd) from the two floats around rstd, and m * gamma + beta as one
rounding of the exact sum. Both must give the fp64 model's bits wherever they are used."""
from fractions import Fraction

import numpy as np
import pytest

from oracle.bf16 import bits_to_f32
from oracle.rmsnorm import rd


def _values(rng, n, dtype):
    """dtype values over their whole range, zeros of both signs and denormals among them"""
    if dtype == "bf16":
        b = rng.integers(0, 1 << 16, size=n).astype(np.uint16)
        b[:4] = [0, 0x8000, 1, 0x8001]
        v = bits_to_f32(b)
    else:
        b = rng.integers(0, 1 << 16, size=n).astype(np.uint16)
        b[:4] = [0, 0x8000, 1, 0x8001]
        v = b.view(np.float16).astype(np.float32)
    return np.where(np.isfinite(v), v, np.float32(1))


def _around(rstd):
    n = rstd.astype(np.float32)
    below = n.astype(np.float64) < rstd
    return (np.where(below, n, np.nextafter(n, np.float32(0))),
            np.where(below, np.nextafter(n, np.float32(np.inf)), n))


def _near_ties(rng, x, dtype):
    """rstd whose fp64 product with x lies within a few 2^-52 of the fp32 midpoint beside
    a tie of the dtype, on either side"""
    keep = 8 if dtype == "bf16" else 11
    t = 1.0 + (2 * rng.integers(0, 1 << (keep - 1), size=x.size) + 1) * 2.0 ** -keep
    t = t + rng.choice([-1.0, 0.0, 1.0], size=x.size) * 2.0 ** -24 + rng.integers(-3, 4, size=x.size) * 2.0 ** -52
    return t / np.abs(x)


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_product_from_the_floats_around_rstd(dtype):
    rng = np.random.default_rng(7)
    n = 400000
    x = _values(rng, n, dtype)
    with np.errstate(over="ignore", under="ignore", invalid="ignore"):
        tie_x = rng.integers(0x3F80, 0x4000, size=n).astype(np.uint16)
        tie_x = bits_to_f32(tie_x) if dtype == "bf16" else 1 + rng.integers(0, 1024, size=n).astype(np.float32) / 1024
        for xs, rstd in ((x, np.exp2(rng.uniform(-20, 20, size=n))), (tie_x, _near_ties(rng, tie_x, dtype))):
            lo, hi = _around(rstd)
            a = rd((xs * lo).astype(np.float64), dtype)
            b = rd((xs * hi).astype(np.float64), dtype)
            want = rd(xs.astype(np.float64) * rstd, dtype)
            same = (a == b) & (np.signbit(a) == np.signbit(b))
            assert (lo.astype(np.float64) <= rstd).all() and (rstd <= hi.astype(np.float64)).all()
            assert np.array_equal(a[same], want[same]) and np.array_equal(np.signbit(a[same]), np.signbit(want[same]))
        assert (~same).sum() > n // 4  # the near-tie products reach the fp64 form


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_one_rounding_of_the_exact_sum(dtype):
    """fp32(m * gamma + beta) of the exact sum == fp32(fp64 sum), on values whose parts lie
    far apart, cancel, or meet at an fp32 midpoint."""
    rng = np.random.default_rng(11)
    n = 20000
    m, g, b = (_values(rng, n, dtype).astype(np.float64) for _ in range(3))
    scale = np.exp2(rng.integers(-60, 2, size=n).astype(np.float64))
    with np.errstate(over="ignore"):
        near = rd(-m * g * rng.choice([1.0, 1 + 2.0 ** -7, 2.0 ** -30, 2.0 ** 30], size=n) * scale, dtype)
    b = np.where(rng.random(n) < 0.7, near, b)
    with np.errstate(over="ignore"):
        want = (m * g + b).astype(np.float32)
    ok = np.isfinite(want) & np.isfinite(b)
    for i in np.flatnonzero(ok)[:8000]:
        exact = Fraction(m[i]) * Fraction(g[i]) + Fraction(b[i])
        assert _rne32(exact) == Fraction(float(want[i])), (m[i], g[i], b[i])


def _rne32(x):
    """x rounded once to the fp32 grid (denormals included), ties to even"""
    if x == 0:
        return x
    a = abs(x)
    e = a.numerator.bit_length() - a.denominator.bit_length()
    if Fraction(2) ** e > a:
        e -= 1
    step = Fraction(2) ** (max(e, -126) - 23)
    q = round(a / step) * step  # Fraction rounds half to even
    return q if x > 0 else -q
