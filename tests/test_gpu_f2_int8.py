"""The split form's int8 contraction where its shape can go wrong: blocks longer than the
16,384 SNPs that fit its int32 levels (summed in segments whose shares of W_0's offset have
to add up), blocks of one K-step pair, empty blocks in every position, and the sub-tile
deal of diagonal and partial 128-row tiles.

Bars: pair counts exact; f2 within 1e-9 of the long-double oracle (floor 1e-6, or the
tiny-block floor of test_gpu_decode_f2 where blocks hold a few SNPs), the form's stated
precision.
"""
import numpy as np
import pytest

from steppe_amd import _core
from test_gpu_decode_f2 import F2_FLOOR_TINY_BLOCKS, _f2_qvn_gpu, _rel_err

pytestmark = pytest.mark.gpu

SPLIT = _core.STP_PREC_SPLIT_BF16


def _qvn(P, M, seed, missing=0.1):
    rng = np.random.default_rng(seed)
    n = rng.integers(1, 120, (P, M)).astype(np.float64)
    q = np.round(rng.random((P, M)) * 2 * n) / (2 * n)
    q[: P // 3] = np.round(q[: P // 3])            # fixed SNPs: the digits' extremes
    v = (rng.random((P, M)) >= missing).astype(np.float64)
    return q * v, v, n * v


@pytest.mark.parametrize("length", [16383, 16384, 16385, 32768 + 7, 50001])
def test_blocks_longer_than_a_segment(engine, cref, length):
    P = 9
    q, v, n = _qvn(P, length + 900, seed=length)
    bid = np.repeat(np.array([0, 1, 2], np.int32), [400, length, 500])
    f2, vp, _ = _f2_qvn_gpu(engine, q, v, n, bid, 3, SPLIT)
    fr, vr, _ = cref.f2_blocks(q, v, n, bid, 3)
    assert np.array_equal(vp, vr)
    err = _rel_err(f2, fr)
    print(f"  block of {length}: {err:.2e}", flush=True)
    assert err <= 1e-9
    assert np.array_equal(f2, f2.transpose(1, 0, 2))


@pytest.mark.parametrize("P", [1, 32, 33, 64, 65, 96, 97, 128, 129, 161, 200, 225])
@pytest.mark.parametrize("prec", [SPLIT, _core.STP_PREC_FP64])
def test_sub_tile_deal(engine, cref, P, prec):
    # one to two 128-row tiles with every number of 32-row groups; K-steps 2, 4, 6, ...
    sizes = [1, 33, 64, 65, 130, 300]
    q, v, n = _qvn(P, sum(sizes), seed=P)
    bid = np.repeat(np.arange(len(sizes), dtype=np.int32), sizes)
    f2, vp, _ = _f2_qvn_gpu(engine, q, v, n, bid, len(sizes), prec)
    fr, vr, _ = cref.f2_blocks(q, v, n, bid, len(sizes))
    assert np.array_equal(vp, vr)
    assert _rel_err(f2, fr, F2_FLOOR_TINY_BLOCKS) <= 1e-9


@pytest.mark.parametrize("ids,n_block", [([1, 1, 3], 5), ([0, 2], 3), ([4], 5)])
def test_empty_blocks(engine, cref, ids, n_block):
    # blocks without a SNP first, between and last: zero f2 and zero pairs
    P = 40
    bid = np.repeat(np.array(ids, np.int32), 70)
    q, v, n = _qvn(P, len(bid), seed=n_block)
    f2, vp, bs = _f2_qvn_gpu(engine, q, v, n, bid, n_block, SPLIT)
    fr, vr, br = cref.f2_blocks(q, v, n, bid, n_block)
    assert np.array_equal(vp, vr) and np.array_equal(bs, br)
    for b in range(n_block):
        if b not in ids:
            assert not f2[:, :, b].any() and not vp[:, :, b].any()
    assert _rel_err(f2, fr, F2_FLOOR_TINY_BLOCKS) <= 1e-9


def test_frequencies_outside_the_unit_interval_count_as_missing(engine):
    # a frequency that is not one (or not a number) drops its entry, as with V = 0
    q, v, n = _qvn(20, 512, seed=3, missing=0.0)
    bid = np.zeros(512, np.int32)
    bad_q, ok_v = q.copy(), v.copy()
    for k, x in enumerate([1.5, -0.25, np.nan, np.inf, -np.inf]):
        bad_q[k, 10 * k:10 * k + 7] = x
        ok_v[k, 10 * k:10 * k + 7] = 0.0
    want = _f2_qvn_gpu(engine, q, ok_v, n, bid, 1, SPLIT)
    tau_free = np.abs(want[0]) >= 1e-4     # smaller entries are recomputed from the input as given
    got = _f2_qvn_gpu(engine, bad_q, v, n, bid, 1, SPLIT)
    assert np.array_equal(got[1], want[1])
    assert np.array_equal(got[0][tau_free], want[0][tau_free])
