"""nn::batchnorm's row sums at the edges of their split, bit for bit against the oracle: row lengths around the eight
partials' tail and the 2304-element chunk (one chunk, a whole one, one and a tail, two and a rest), sample counts around
the four rows of a workgroup and the sixteen-wide blocks of the channel sums, aligned rows and not, with and without the
folded ReLU's flags. Every sum runs in a fixed order, so the tolerance is zero."""
import numpy as np
import pytest

from helpers import assert_same
from nnh import synth

pytestmark = pytest.mark.gpu

EPS = 1e-5


@pytest.mark.parametrize("N,C,S", [(1, 1, 1), (3, 2, 7), (4, 3, 8), (5, 2, 12), (17, 2, 36), (33, 1, 100), (4, 1, 2303), (6, 2, 2304),
                                   (2, 1, 2305), (3, 1, 2312), (5, 1, 4608), (2, 2, 4613), (1, 1, 7004)])
@pytest.mark.parametrize("relu", [False, True])
def test_row_sums(gpu, oracle, N, C, S, relu):
    import torch

    import nnh
    x, g = synth.normal(51, (N, C, S)), synth.normal(52, (N, C, S))
    w, b = synth.normal(53, (C,)), synth.normal(54, (C,))
    fwd = oracle.batchnorm_forward(x, w, b, EPS, relu)
    y0, alive0, mean0, var0, inv0 = fwd
    dx0, dw0, db0 = oracle.batchnorm_backward(g, x, alive0 if relu else None, w, mean0, inv0)

    def place(a, off):  # off floats past a 16-byte boundary
        t = torch.empty(a.size + off, device="cuda")
        t[off:] = torch.from_numpy(np.ascontiguousarray(a).ravel()).cuda()
        return t[off:].view(a.shape)

    for off in (0, 1):
        xd, gd, wd, bd = (place(a, off) for a in (x, g, w, b))
        y, alive, mean, var, inv = nnh.batchnorm_forward(xd, wd, bd, EPS, fuse_relu=relu)
        for got, want, what in ((y, y0, "y"), (mean, mean0, "mean"), (var, var0, "var"), (inv, inv0, "inv_std")):
            assert_same(got.cpu().numpy(), want.reshape(got.shape), (what, N, C, S, off))
        dx, dw, db = torch.empty_like(xd), torch.empty_like(wd), torch.empty_like(bd)
        nnh.batchnorm_backward(gd, xd, alive, wd, mean, inv, dx=dx, dw=dw, db=db)
        for got, want, what in ((dx, dx0, "dx"), (dw, dw0, "dw"), (db, db0, "db")):
            assert_same(got.cpu().numpy(), want.reshape(got.shape), (what, N, C, S, off))
