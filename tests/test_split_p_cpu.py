"""The suffix kernels' P operand on the matrix cores: p (fp32, 0 <= p <= 2^8 after
the lazy running max) enters the bf16 MFMA as two terms, hi = p truncated to bf16
and lo = p - hi rounded to bf16 (csrc/suffix_decode.hip, the window step), or, in the
fused kernel above 4 heads per group and in stage 1's decode form, as three
truncated terms. What is left after the first is kept at min(p, 2^-100) or above, so
that no term of a p > 0 is 0 (an infinite V element times 0 would be NaN).
The kernel's contract is fp32-P precision: |hi + lo - p| <= 2^-16 p, so that the
value MFMA sums p * v to within fp32-level error of the unquantised oracle.

The bound follows from hi keeping p's top 8 significand bits (|p - hi| < 2^-7 p,
and p - hi is exact in fp32) and lo's RNE to 8 bits (error <= 2^-9 |p - hi|).
These checks pin it on random and adversarial values with the oracle's own RNE
(oracle/bf16.py, itself pinned against torch), and show the two plausible
mistakes miss it: hi alone (bf16 P) and a truncated lo term."""
import numpy as np

from oracle.bf16 import bits_to_f32, round_bf16


def _hi(p):
    return (p.astype(np.float32).view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)


def _split(p, lo_round=True):
    p = p.astype(np.float32)
    hi = _hi(p)
    d = (p - hi).astype(np.float32)  # exact: hi is p with its low 16 bits cleared
    lo = round_bf16(d) if lo_round else _hi(d)
    return hi, lo


def _p_values():
    rng = np.random.default_rng(0)
    p = np.concatenate([
        np.exp2(-rng.uniform(0, 60, 200000)),              # exp2(s - m) after the running max
        rng.uniform(0, 256, 100000),                        # up to 2^kTau above the max's reference
        np.float32(1.0) + np.arange(1, 4096, dtype=np.float32) * np.float32(2.0 ** -23),  # low bits set
        bits_to_f32(np.arange(0x3F80, 0x4380, dtype=np.uint16)),                            # exact bf16 values
        np.array([0.0, 2.0 ** -126, 255.99998, 256.0], dtype=np.float32),
    ]).astype(np.float32)
    return p


def test_difference_is_exact_in_fp32():
    p = _p_values()
    hi = _hi(p)
    d32 = (p - hi).astype(np.float32)
    np.testing.assert_array_equal(d32.astype(np.float64), p.astype(np.float64) - hi.astype(np.float64))


def test_hi_plus_lo_within_2_pow_minus_16():
    p = _p_values()
    hi, lo = _split(p)
    err = np.abs(hi.astype(np.float64) + lo.astype(np.float64) - p.astype(np.float64))
    assert np.all(err <= 2.0 ** -16 * p.astype(np.float64)), (err / np.maximum(p, 1e-300)).max()
    # exact bf16 values split into (p, 0)
    b = bits_to_f32(np.arange(0x3F80, 0x4380, dtype=np.uint16))
    hb, lb = _split(b)
    assert np.array_equal(hb, b) and not lb.any()


def test_plausible_mistakes_miss_the_bound():
    p = _p_values()
    pos = p > 0
    # bf16 P alone (hi only, or p rounded once): errors up to 2^-8 p
    hi, _ = _split(p)
    rel_hi = np.abs(hi.astype(np.float64) - p)[pos] / p[pos]
    rel_rne = np.abs(round_bf16(p).astype(np.float64) - p)[pos] / p[pos]
    assert rel_hi.max() > 2.0 ** -16 and rel_rne.max() > 2.0 ** -16
    # a truncated lo term (not rounded) doubles lo's error bound: 2^-16 is exceeded
    h2, l2 = _split(p, lo_round=False)
    rel_trunc = np.abs(h2.astype(np.float64) + l2.astype(np.float64) - p)[pos] / p[pos]
    assert rel_trunc.max() > 2.0 ** -16


FLOOR = np.float32(2.0 ** -100)


def _rest(p):
    """median(p - hi, p, 2^-100) as the kernel has it"""
    d = (p - _hi(p)).astype(np.float32)
    return np.maximum(d, np.minimum(p, FLOOR))


def _terms3(p):
    r = _rest(p)
    c = np.float64(1.0) + 2.0 ** -23  # one fma: the exact product and difference, rounded once
    lo = _hi((r.astype(np.float64) * c - _hi(r).astype(np.float64)).astype(np.float32))
    # lo is halved through its exponent field, one half per half of the operand
    half = np.where(lo > 0, (lo.view(np.uint32) - np.uint32(1 << 23)).view(np.float32), np.float32(0))
    return _hi(p), _hi(r), half


def test_floored_two_terms_keep_the_bound_and_their_sign():
    p = _p_values()
    hi, lo = _hi(p), round_bf16(_rest(p))
    err = np.abs(hi.astype(np.float64) + lo.astype(np.float64) - p.astype(np.float64))
    assert np.all(err <= 2.0 ** -16 * p.astype(np.float64) + 2.0 ** -100 * (p > 0))
    pos = p > 0
    assert (hi[pos] > 0).all() and (lo[pos] > 0).all() and not hi[~pos].any() and not lo[~pos].any()
    # unchanged by the floor wherever p is not a bf16 value
    old = _split(p)[1]
    changed = lo != old
    assert not old[changed].any()


def test_three_terms_hold_fp32():
    p = _p_values()
    hi, mid, half = (t.astype(np.float64) for t in _terms3(p))
    err = np.abs(hi + mid + 2 * half - p.astype(np.float64))
    # 2^-23 of the rest (< 2^-7 p) and the floor
    assert np.all(err <= 2.0 ** -30 * p.astype(np.float64) + 2.0 ** -99 * (p > 0)), err.max()
    pos = p >= np.float32(2.0 ** -125)
    assert (hi[pos] > 0).all() and (mid[pos] > 0).all() and (half[pos] > 0).all()
    assert not hi[p == 0].any() and not mid[p == 0].any() and not half[p == 0].any()
