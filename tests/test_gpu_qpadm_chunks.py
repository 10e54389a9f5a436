"""Device memory and chunks of a qpAdm call over many models."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _tensor(P, nb, seed=11):
    rng = np.random.default_rng(seed)
    q = np.clip(rng.random((P, 1, 80)) * 0.6 + 0.2 + 0.08 * rng.standard_normal((P, nb, 80)), 0.0, 1.0)
    f2 = np.asfortranarray(((q[:, None] - q[None]) ** 2).mean(-1))
    return f2, rng.integers(50, 90, nb).astype(np.int32)


def test_memory_of_a_fleet():
    # a call keeps each model's setup results (X, LOO, Qinv, totals) and its refits' weights, once
    from steppe_amd import _core
    n, nb, nl, nr = 2000, 700, 2, 3
    f2, bs = _tensor(12, nb)
    rng = np.random.default_rng(1)
    models = [(int(p[0]), [int(x) for x in p[1:1 + nl]], [int(x) for x in p[1 + nl:2 + nl + nr]])
              for p in (rng.permutation(12) for _ in range(n))]
    h = _core.upload_f2(f2, None, bs, [f"p{i}" for i in range(12)])
    _core.qpadm_models(h, models[:1])
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    _core.qpadm_models(h, models)
    grown = before - torch.cuda.mem_get_info()[0]
    m = nl * nr
    kept = 8.0 * n * (2 * m * nb + m * m + 2 * m + 8 * nb)
    print(f"{n} models: {grown / 2 ** 20:.0f} MiB more, {kept / 2 ** 20:.0f} MiB of results", flush=True)
    # beside them a fit table, a model and a record each (under 8 KiB) and allocation granules
    assert grown <= kept + 8192 * n + (16 << 20)


def _mixed(n, P, seed=4):
    """Models of every refit kernel: 1-5 sources in the row form's instances, 6-7 sources and
    more right populations with a wavefront a fit, and one beyond 64 entries."""
    rng = np.random.default_rng(seed)
    shapes = [(1, 3), (2, 2), (2, 9), (2, 14), (3, 5), (3, 11), (3, 16), (4, 8), (4, 12), (5, 6), (5, 12), (6, 7),
              (7, 9), (2, 20), (6, 12)]
    out = []
    for i in range(n):
        nl, nr = shapes[i % len(shapes)]
        p = [int(x) for x in rng.permutation(P)]
        out.append((p[0], p[1:1 + nl], p[1 + nl:2 + nl + nr]))
    return out


@pytest.mark.parametrize("jackknife", ["all", "feasible", "none"])
def test_chunks_give_the_same_fits(monkeypatch, jackknife):
    # a call cut into chunks re-uses every workspace: the records are the uncut call's bytes
    from steppe_amd import _core
    f2, bs = _tensor(30, 45)
    h = _core.upload_f2(f2, None, bs, [f"p{i}" for i in range(30)])
    models = _mixed(47, 30)
    monkeypatch.delenv("STEPPE_QPADM_CHUNK", raising=False)
    whole = [bytes(r) for r in _core.qpadm_models(h, models, jackknife=jackknife, raw=True)]
    assert len({r for r in whole}) == len(models)
    for chunk in (1, 7, 23, 46):
        monkeypatch.setenv("STEPPE_QPADM_CHUNK", str(chunk))
        got = [bytes(r) for r in _core.qpadm_models(h, models, jackknife=jackknife, raw=True)]
        assert got == whole, chunk
