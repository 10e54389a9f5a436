"""Leave-one-block-out refits with eight or sixteen lanes a fit, at the edges of their shapes:
right populations at and around the kernel instances' limits (8, 12, 16 columns), the fewest
that a model may have, block counts around the sixteen and thirty-two fits of a workgroup and
of a whole genome, against the oracle with the bounds of test_gpu_qpadm, and against the form
with a wavefront a fit, bit for bit."""
import numpy as np
import pytest

from test_gpu_qpadm import check_fields, compare, merge

pytestmark = pytest.mark.gpu

# sources -> right - 1
SHAPES = {2: (1, 2, 7, 8, 9, 12, 13, 16), 3: (2, 3, 8, 9, 12, 13, 16), 4: (3, 4, 8, 9, 12, 13, 16),
          5: (4, 5, 8, 9, 12)}


def _tensor(nb, seed=3):
    """A target (0) mixed from five sources (1-5) and 17 right populations related to them, so
    that every model of a few sources is well determined."""
    rng = np.random.default_rng(seed)
    src = rng.random((5, nb, 400)) * 0.6 + 0.2
    right = np.einsum("rs,sbk->rbk", rng.dirichlet(np.full(5, 0.4), 17), src) + 0.05 * rng.standard_normal((17, nb, 400))
    target = np.einsum("s,sbk->bk", [0.3, 0.25, 0.2, 0.15, 0.1], src) + 0.02 * rng.standard_normal((nb, 400))
    q = np.concatenate([target[None], src, right])
    f2 = ((q[:, None] - q[None]) ** 2).mean(-1)
    return np.asfortranarray(f2), rng.integers(20, 90, nb).astype(np.int32)


@pytest.mark.parametrize("nb", [2, 16, 17, 41, 700])
def test_refits_at_shape_edges(cref, nb):
    from steppe_amd import _core
    f2, bs = _tensor(nb)
    h = _core.upload_f2(f2, None, bs, [f"p{i}" for i in range(f2.shape[0])])
    models = [(0, list(range(1, 1 + nl)), list(range(6, 7 + nr))) for nl, cols in SHAPES.items() for nr in cols]
    res = _core.qpadm_models(h, models)
    worst = {}
    for (t, left, right), d in zip(models, res):
        o = cref.qpadm(f2, None, bs, t, left, right)
        merge(worst, compare(d, o, f"nb {nb}, {len(left)} sources, {len(right)} right"))
        # the same model alone, and without refits, gives the same fit
        one = _core.run_qpadm(h, t, left, right)
        assert one["weight"] == d["weight"] and one["se"] == d["se"]
        bare = _core.qpadm_models(h, [(t, left, right)], jackknife="none")[0]
        assert bare["weight"] == d["weight"] and bare["chisq"] == d["chisq"]
    check_fields(worst, f"{len(models)} shapes, {nb} blocks")


def _near_degenerate(nb, seed=8):
    """The same populations with the second source a copy of the first but for noise of 1e-6 and
    two equal right populations: refits whose pivots are rounding, or exactly zero."""
    rng = np.random.default_rng(seed)
    q = rng.random((23, nb, 50)) * 0.8 + 0.1
    q[2] = q[1] + 1e-6 * rng.standard_normal((nb, 50))
    q[8] = q[7]
    f2 = ((q[:, None] - q[None]) ** 2).mean(-1)
    return np.asfortranarray(f2), rng.integers(20, 90, nb).astype(np.int32)


@pytest.mark.parametrize("tensor", [_tensor, _near_degenerate])
@pytest.mark.parametrize("nb", [2, 3, 33, 500])
def test_both_refit_forms_same_bits(monkeypatch, tensor, nb):
    # few lanes a fit and a wavefront a fit, over every shape of the former: the same records
    from steppe_amd import _core
    f2, bs = tensor(nb)
    h = _core.upload_f2(f2, None, bs, [f"p{i}" for i in range(f2.shape[0])])
    models = [(0, list(range(1, 1 + nl)), list(range(6, 6 + nr + 1)))
              for nl in SHAPES for nr in range(nl - 1 or 1, 17) if nl * nr <= 64]
    for options in ({}, {"jackknife": "feasible"}, {"als_iterations": 1}, {"fudge": 0.0}):
        monkeypatch.delenv("STEPPE_QPADM_REFITS", raising=False)
        few = [bytes(r) for r in _core.qpadm_models(h, models, raw=True, **options)]
        monkeypatch.setenv("STEPPE_QPADM_REFITS", "wave")
        wave = [bytes(r) for r in _core.qpadm_models(h, models, raw=True, **options)]
        off = [(len(m[1]), len(m[2]) - 1) for m, a, b in zip(models, few, wave) if a != b]
        print(f"  {tensor.__name__} nb {nb} {options}: {len(models)} models, differing {off}", flush=True)
        assert not off
