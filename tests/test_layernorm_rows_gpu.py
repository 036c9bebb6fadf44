"""nn::layernorm's row and column kernels at the edges of their splits, bit for bit against the oracle: rows at and
around the chains' 16-element blocks and the longest row a workgroup holds with either slot count, row counts around the
column kernel's 192-row chunks (fewer chunks than its load ring, whole rounds and remainders), aligned and not. Each sum
is a chain in a fixed order, so the tolerance is zero."""
import numpy as np
import pytest

from helpers import assert_same
from nnh import synth

pytestmark = pytest.mark.gpu

EPS = 1e-5


@pytest.mark.parametrize("R,D", [(1025, 16), (1152, 20), (1153, 5), (1343, 36), (1344, 64), (1345, 1), (1729, 100), (3, 8192),
                                 (2, 8193), (2, 8196), (1, 16384), (2, 16383), (1, 16385), (33, 255), (1030, 300)])
def test_rows_and_columns(gpu, oracle, R, D):
    import torch

    import nnh
    x, g = synth.normal(31, (R, D)), synth.normal(32, (R, D))
    gm, bt = synth.normal(33, (D,)), synth.normal(34, (D,))
    old = synth.normal(35, (R, D)), synth.normal(36, (D,)), synth.normal(37, (D,))
    y0, mean0, inv0 = oracle.layernorm_forward(x, gm, bt, EPS)

    def place(a, off):  # off floats past a 16-byte boundary
        t = torch.empty(a.size + off, device="cuda")
        t[off:] = torch.from_numpy(np.ascontiguousarray(a).ravel()).cuda()
        return t[off:].view(a.shape)

    for off in (0, 1):
        xd, gd, gmd, btd = (place(a, off) for a in (x, g, gm, bt))
        y, mean, inv = nnh.layernorm_forward(xd, gmd, btd, EPS)
        for got, want, what in ((y, y0, "y"), (mean, mean0, "mean"), (inv, inv0, "inv_std")):
            assert_same(got.cpu().numpy(), want.reshape(got.shape), (what, R, D, off))
        for first in (True, False):
            want = oracle.layernorm_backward(g, x, gm, mean0, inv0, old[0], first, old[1], first, old[2], first)
            for parts in ((1, 1, 1), (1, 0, 0), (0, 1, 1)):
                got = [place(a, off) if p else None for a, p in zip(old, parts)]
                nnh.layernorm_backward(gd, xd, gmd, mean, inv, dx=got[0], dx_first=first, dgamma=got[1], dgamma_first=first,
                                       dbeta=got[2], dbeta_first=first)
                for t, w, what in zip(got, want, ("dx", "dgamma", "dbeta")):
                    if t is not None:
                        assert_same(t.cpu().numpy(), w, (what, R, D, off, first, parts))
