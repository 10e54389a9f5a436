"""Sweeps whose launches leave more hits than the device-side selection's threshold (32,768
and twice top_k), against the same sweep where no launch does (a top_k of everything, or
small launches): the kept rows must be the same, bit for bit, ties included."""
import math

import numpy as np
import pytest

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
