"""The two arithmetic shortcuts of the threshold rows (csrc/sdx_thr.hip), restated and
compared with what they stand for: the fixed-point exp formed from the mantissa and the
exponent by one shift, and x / T by two FMA steps from 1 / T."""
from fractions import Fraction

import numpy as np

from oracle import numerics as N


def _exp62(d):
    """thr_exp62 in numpy fp32 / float64, step by step."""
    dd = np.maximum(d, np.float32(-43.5)).astype(np.float64)
    kf = np.floor(dd * float.fromhex("0x1.71547652b82fep+0"))
    r = np.maximum((dd - kf * float.fromhex("0x1.62e42fefa39efp-1")).astype(np.float32),
                   np.float32(0))
    p = N.exp_det_poly(r)
    mant = np.minimum(p, np.float32(2)).view(np.uint32) - np.uint32(0x3F000000)
    hi = (mant << np.uint32(7)).astype(np.uint64) << np.uint64(32)
    return hi >> (-kf).astype(np.uint64)


def test_fixed_point_exp_by_one_shift():
    rng = np.random.default_rng(0)
    k = np.arange(0, 160) * -np.log(2.0)
    edges = np.concatenate([k, k / 2, np.arange(0, 111), [43.5, 43.49999, 43.50001, 42.975]])
    edges = (-np.abs(edges)).astype(np.float32)
    near = np.concatenate([np.nextafter(edges, np.float32(s)) for s in (-200, 0)])
    tiny = -np.exp(rng.uniform(-100, 0, 1 << 16)).astype(np.float32)
    d = np.concatenate([edges, near, tiny, -rng.uniform(0, 110, 1 << 20).astype(np.float32)])
    d = np.minimum(d, np.float32(0))
    ref = np.asarray(N.fixed62(N.exp_det(d)), np.uint64)
    assert np.array_equal(_exp62(d), ref)


def _rn(v):
    """A Fraction rounded to the nearest fp32 (ties to even; normal range)."""
    if v == 0:
        return Fraction(0)
    e = 0
    a = abs(v)
    while a >= 2:
        a, e = a / 2, e + 1
    while a < 1:
        a, e = a * 2, e - 1
    n = a * (1 << 23)
    q = n.numerator // n.denominator
    rest = n - q
    if rest > Fraction(1, 2) or (rest == Fraction(1, 2) and q % 2 == 1):
        q += 1
    return (1 if v > 0 else -1) * Fraction(q, 1 << 23) * Fraction(2) ** e


def test_division_by_two_fma_steps():
    """Correctly rounded wherever the kernel uses it, at ordinary temperatures and at
    mantissas next to the ends of their range."""
    rng = np.random.default_rng(1)
    ts = [np.float32(t) for t in (0.6, 0.7, 0.8, 0.9, 1.1, 1.3, 1e-3, 3.0, 4e5)]
    ts += list(np.array([0x3F800001, 0x3FFFFFFF, 0x3FFFFFFE, 0x35800001, 0x497FFFFF],
                        np.uint32).view(np.float32))
    for T in ts:
        t, rt = Fraction(float(T)), _rn(1 / Fraction(float(T)))
        bits = rng.integers(0, 1 << 23, 60).astype(np.uint32)
        bits = np.concatenate([bits, np.array([0, 1, (1 << 23) - 1, (1 << 23) - 2], np.uint32)])
        for x in (bits | np.uint32(130 << 23)).view(np.float32):
            v = Fraction(float(x))
            q = _rn(v * rt)
            for _ in range(2):
                q = _rn(_rn(v - t * q) * rt + q)
            assert q == _rn(v / t), (float(T), float(x))
