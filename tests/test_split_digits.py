"""The split form's digit bounds (steppe_amd/csrc/f2_split.hip, stage_entry and balanced48),
restated in numpy from the kernel's own steps and checked against what the scheme needs:

* q' = q - 1/2 and w = -(q~^2 - h)/2 as 48-bit integers in six balanced 8-bit digits:
  |d_0| <= 64, every other digit in [-128, 127], |q~ - q'| <= 2^-48, |w~ - w| <= 2^-48;
* the first w byte of an observed entry, W_0 + 96, has bit 6 set and bit 7 clear, so the flag
  V = -128 v is its bit 6 moved up;
* 16,384 SNPs keep every int32 level sum below 2^31, and the combined levels are exact in
  64-bit integers and in a double;
* the sum of the levels, with W_0's offset taken back from the pair count, is the estimator up
  to the digits' truncation and the dropped products.

Counts run over every population size of the panels (n = 1 .. 16383) with edge cases
(q = 0, 1/2, 1 and q = 1/256-style values with short binary expansions).
"""
from fractions import Fraction

import numpy as np

OFFSET = 96                # W_0' - W_0
SEGMENT = 512 * 32         # SNPs summed in int32


def _balanced(x):
    """Digits 0 (most significant) to 5 of round-to-even(x), by balanced48's bytes."""
    bits = (x + 1.5 * 2.0 ** 52).view(np.uint64)
    b = (bits + np.uint64(0x8080808080)) ^ np.uint64(0x8080808080)
    return [((b >> np.uint64(8 * (5 - k))) & np.uint64(0xFF)).astype(np.uint8).view(np.int8).astype(np.int64)
            for k in range(6)]


def _entry(a, n):
    """(d, W, q, w) of observed entries, as stage_entry forms them (W without its offset)."""
    q = a / (2.0 * n)
    h = q * (1.0 - q) / np.maximum(n - 1.0, 1.0)
    assert (h >= 0).all()
    x = (q - 0.5) * 2.0 ** 47
    qt = ((x + 1.5 * 2.0 ** 52) - 1.5 * 2.0 ** 52) * 2.0 ** -47
    y = qt * qt - h
    return _balanced(x), _balanced(y * 2.0 ** 46), q, -0.5 * y


def _value(d):
    return sum(dk << (8 * (5 - k)) for k, dk in enumerate(d))


def _counts(size=1_000_000):
    rng = np.random.default_rng(7)
    n = rng.integers(1, 16384, size).astype(np.float64)
    a = np.minimum(np.floor(rng.random(n.size) * (2 * n + 1)), 2 * n)
    edge_n = np.array([1, 1, 1, 2, 2, 128, 128, 16383, 16383, 16383, 256, 512], np.float64)
    edge_a = np.array([0, 1, 2, 1, 3, 1, 255, 0, 16383, 32766, 1, 3], np.float64)
    return np.concatenate([edge_a, a]), np.concatenate([edge_n, n])


def test_q_digits():
    d, _, q, _ = _entry(*_counts())
    assert np.abs(d[0]).max() <= 64
    err = np.abs(_value(d) * 2.0 ** -47 - (q - 0.5))
    assert err.max() <= 2.0 ** -48
    # (against q itself, the subtraction's rounding of at most 2^-55 comes on top)
    for i in np.argsort(err)[-20:]:
        exact = Fraction(float(q[i])) - Fraction(1, 2)
        assert abs(Fraction(int(_value(d)[i]), 2 ** 47) - exact) <= Fraction(1, 2 ** 48) + Fraction(1, 2 ** 55)


def test_w_digits_and_the_flag():
    _, W, _, w = _entry(*_counts())
    byte = W[0] + OFFSET
    assert byte.min() >= 79 and byte.max() <= 113
    assert ((byte & 0x40) == 0x40).all() and ((byte & 0x80) == 0).all()
    assert (((byte << 1) & 0x80).astype(np.uint8).view(np.int8) == -128).all() and (0 << 1) & 0x80 == 0
    # w~ = -128 sum_k W_k 2^(-14 - 8 k)
    exact = [Fraction(-int(v), 2 ** 47) for v in _value(W)[:20]]
    got = -_value(W) * 2.0 ** -47
    assert all(Fraction(float(g)) == e for g, e in zip(got, exact))
    err = np.abs(got - w)
    assert err.max() <= 2.0 ** -48
    for i in np.argsort(err)[-20:]:
        assert abs(Fraction(-int(_value(W)[i]), 2 ** 47) - Fraction(float(w[i]))) <= Fraction(1, 2 ** 48)


def test_level_sums_fit_int32():
    d, W, _, _ = _entry(*_counts())
    m = [int(np.abs(x).max()) for x in d]
    W[0] = W[0] + OFFSET
    growth = [sum(m[k] * m[t - k] for k in range(t + 1)) + 2 * 128 * int(np.abs(W[t]).max()) for t in range(6)]
    assert max(growth) == growth[5] <= 114_688
    assert all(SEGMENT * g < 2 ** 31 for g in growth)
    # the epilogue's upper and lower halves, exact in a double
    level = [SEGMENT * g for g in growth]
    level[0] += 2 * 128 * OFFSET * SEGMENT
    assert (level[0] << 16) + (level[1] << 8) + level[2] < 2 ** 53
    assert (level[3] << 16) + (level[4] << 8) + level[5] < 2 ** 53


def test_levels_recombine_to_the_estimator():
    # a block of 3 segments, two populations with missing entries: levels summed in integers,
    # W_0's offset taken back in shares of the pair count
    rng = np.random.default_rng(3)
    M = 2 * SEGMENT + 77
    ent, v = [], []
    for _ in range(2):
        n = rng.integers(1, 60, M).astype(np.float64)
        ent.append(_entry(np.floor(rng.random(M) * (2 * n + 1)), n))
        v.append((rng.random(M) < np.where(np.arange(M) < SEGMENT, 0.3, 0.95)).astype(np.int64))
    (di, Wi, qi, wi), (dj, Wj, qj, wj) = ent
    vi, vj = v
    steps = -(-M // 64) * 2                       # blocks are padded to 64 SNPs
    pairs = int((vi * vj).sum())
    num = Fraction(0)
    for s0 in range(0, steps, 512):
        s1 = min(s0 + 512, steps)
        at = slice(32 * s0, min(32 * s1, M))
        L = []
        for t in range(6):
            x = sum((di[k] * dj[t - k] * vi * vj)[at].sum() for k in range(t + 1))
            wt, wu = (Wi[t] + (OFFSET if t == 0 else 0)) * vi, (Wj[t] + (OFFSET if t == 0 else 0)) * vj
            L.append(int(x + (-128 * vj * wt)[at].sum() + (-128 * vi * wu)[at].sum()))
            assert abs(L[-1]) < 2 ** 31
        L[0] += 2 * 128 * OFFSET * (pairs * s1 // steps - pairs * s0 // steps)
        hi, lo = (L[0] << 16) + (L[1] << 8) + L[2], (L[3] << 16) + (L[4] << 8) + L[5]
        num += -2 * (Fraction(hi, 2 ** 30) + Fraction(lo, 2 ** 54))
    want = Fraction(0)
    both = np.flatnonzero(vi * vj)
    for s in both:
        x, y = Fraction(float(qi[s])) - Fraction(1, 2), Fraction(float(qj[s])) - Fraction(1, 2)
        want += -2 * (x * y + Fraction(float(wi[s])) + Fraction(float(wj[s])))
    # per SNP: two digit truncations of at most 2^-48 on each operand and products k + l >= 6
    assert abs(num - want) <= len(both) * Fraction(1, 2 ** 43)
    print(f"  {len(both)} pairs: off by {float(abs(num - want)) / len(both):.1e} a pair")
