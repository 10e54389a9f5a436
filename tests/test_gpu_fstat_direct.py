"""A few f4 / f3 of a large tensor are read in place, many from the transposed copy: the same
statistics in either batch must be the same bits, at block counts around a wavefront's 64
values a lane step and the widths cached per lane, with dropped blocks, on both sides of the
size where the route changes."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _stats(h, width, idx):
    from steppe_amd import _core
    n = len(idx)
    out = np.empty((4, n))
    idx = np.ascontiguousarray(idx, np.int32)
    p = [C.c_void_p(x.ctypes.data) for x in (idx, *out)]
    f = _core.lib().stp_f4 if width == 4 else _core.lib().stp_f3
    _core.check(f(_core.Context.get(0).h, h.raw, p[0], n, *p[1:]))
    return out


@pytest.mark.parametrize("width", [3, 4])
@pytest.mark.parametrize("P,nb", [(7, 5), (48, 1), (48, 64), (48, 65), (49, 129), (64, 700), (31, 2049)])
def test_in_place_and_transposed_agree(width, P, nb):
    from steppe_amd import _core
    rng = np.random.default_rng(P + nb)
    f2 = rng.random((P, P, nb)) * 0.1
    f2 = np.asfortranarray(f2 + f2.transpose(1, 0, 2))
    vpair = np.asfortranarray(np.full((P, P, nb), 50.0))
    for b in range(2, nb, 9):               # blocks that miss a population are dropped
        vpair[b % P, :, b] = vpair[:, b % P, b] = 0.0
    h = _core.upload_f2(f2, vpair, rng.integers(20, 90, nb).astype(np.int32), [f"p{i}" for i in range(P)])
    line = P * P // (8 * width)             # the most statistics that are read in place
    many = np.array([rng.permutation(P)[:width] for _ in range(line + 40)], np.int32)
    want = _stats(h, width, many)
    for n in {1, 2, line, line + 1}:
        if n >= 1:
            got = _stats(h, width, many[:n])
            assert np.array_equal(got, want[:, :n], equal_nan=True), (n, line)
