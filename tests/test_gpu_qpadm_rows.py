"""Leave-one-block-out refits with sixteen lanes a fit, at the edges of their shapes: right
populations at and around the kernel instances' limits (8, 12, 16 columns), the fewest that a
model may have, block counts around the sixteen fits of a workgroup, against the oracle with
the bounds of test_gpu_qpadm."""
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


@pytest.mark.parametrize("nb", [2, 16, 17, 41])
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
    check_fields(worst, f"{len(models)} shapes, {nb} blocks")
