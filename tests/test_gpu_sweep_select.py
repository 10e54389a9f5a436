"""Sweeps whose launches leave more hits than the device-side selection's threshold (32,768
and twice top_k), against the same sweep where no launch does (a top_k of everything, or
small launches): the kept rows must be the same, bit for bit, ties included."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

FIELDS = ("keys", "est", "se", "z", "p")


def _handle(P, nb=40, seed=5, twins=0):
    from steppe_amd import _core
    rng = np.random.default_rng(seed)
    q = rng.random((P, 1, 60)) * 0.8 + 0.1 + 0.05 * rng.standard_normal((P, nb, 60))
    for i in range(twins):                  # copies of a population: statistics with equal |z|
        q[P - 1 - i] = q[i]
    f2 = np.asfortranarray(((q[:, None] - q[None]) ** 2).mean(-1))
    return _core.upload_f2(f2, None, rng.integers(50, 90, nb).astype(np.int32), [f"p{i:03d}" for i in range(P)])


@pytest.mark.parametrize("k,P,method,twins", [(4, 40, "gram", 0), (4, 40, "direct", 0), (4, 34, "gram", 3),
                                              (3, 64, "direct", 0), (3, 64, "direct", 4)])
def test_selected_rows_are_the_strongest(k, P, method, twins):
    from steppe_amd import _core
    h = _handle(P, twins=twins)
    total = math.comb(P, k)
    assert total > 1 << 15
    whole = _core.run_fstat_sweep(h, k, min_z=0.0, top_k=total, method=method)   # 2 top_k > hits: no selection
    n = len(whole["z"])
    for top_k in (1, 2, 100, 16384, 16385, n // 2 - 1):
        d = _core.run_fstat_sweep(h, k, min_z=0.0, top_k=top_k, method=method)
        for f in FIELDS:
            assert np.array_equal(d[f], whole[f][:top_k]), (f, top_k)


def test_selection_across_launches(monkeypatch):
    from steppe_amd import _core
    h = _handle(70)
    whole = _core.run_fstat_sweep(h, 3, min_z=0.0, top_k=500, method="direct")
    monkeypatch.setenv("STEPPE_FSTAT_CHUNK", "40000")   # 54,740 triples: one launch selects, one does not
    d = _core.run_fstat_sweep(h, 3, min_z=0.0, top_k=500, method="direct")
    for f in FIELDS:
        assert np.array_equal(d[f], whole[f]), f


def _four_kinds(P=64, nb=40, seed=9):
    """Copies of four populations, 16 of each: the 65,536 quartets with one of each kind share
    three values of |z|, to rounding."""
    from steppe_amd import _core
    rng = np.random.default_rng(seed)
    q = rng.random((4, 1, 60)) * 0.8 + 0.1 + 0.05 * rng.standard_normal((4, nb, 60))
    q = q[rng.permutation(np.arange(P) % 4)]
    f2 = np.asfortranarray(((q[:, None] - q[None]) ** 2).mean(-1))
    return _core.upload_f2(f2, None, rng.integers(50, 90, nb).astype(np.int32), [f"p{i:03d}" for i in range(P)])


@pytest.mark.parametrize("method", ["gram", "direct"])
def test_more_equal_hits_than_the_selection_holds(method):
    from steppe_amd import _core
    h = _four_kinds()
    total = math.comb(64, 4)
    whole = _core.run_fstat_sweep(h, 4, min_z=0.0, top_k=total, method=method)
    az = np.abs(whole["z"])
    for top_k in (1, 100, 1500):
        # hits of the K-th hit's bin and above: more than 2 K and the spare 4096
        assert (az >= az[top_k - 1] * (1 - 1e-9)).sum() > 2 * top_k + 4096
        d = _core.run_fstat_sweep(h, 4, min_z=0.0, top_k=top_k, method=method)
        for f in FIELDS:
            assert np.array_equal(d[f], whole[f][:top_k]), (f, top_k)


def test_selection_memory():
    # a sweep's memory follows from its hits; the selection adds what is kept, not all hits again
    from steppe_amd import _core
    h = _handle(100)
    total = math.comb(100, 4)
    assert len(_core.run_fstat_sweep(h, 4, min_z=1e9)["z"]) == 0     # room for every hit, none found
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    assert len(_core.run_fstat_sweep(h, 4, min_z=0.0, top_k=100)["z"]) == 100
    grown = before - torch.cuda.mem_get_info()[0]
    print(f"{total} hits of 32 bytes, 100 kept: {grown / 2 ** 20:.1f} MiB more", flush=True)
    assert grown <= 8 << 20
