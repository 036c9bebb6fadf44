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


@pytest.mark.parametrize("N,C,S", [(1, 256, 1), (31, 256, 8), (32, 257, 5), (33, 128, 7), (65, 90, 127), (32, 256, 128),
                                   (40, 52, 129), (9, 128, 256), (8, 256, 768), (7, 256, 769), (17, 90, 1000), (9, 130, 1024),
                                   (9, 130, 1025)])
@pytest.mark.parametrize("relu", [False, True])
def test_short_row_sums(gpu, oracle, N, C, S, relu):
    """Enough short rows to go 32 or 8 to a workgroup: lengths and counts around both."""
    test_row_sums(gpu, oracle, N, C, S, relu)


@pytest.mark.parametrize("N,C,S", [(512, 2, 16), (513, 3, 8), (513, 2, 7), (600, 1, 20), (2049, 2, 4)])
@pytest.mark.parametrize("relu", [False, True])
def test_many_samples(gpu, oracle, N, C, S, relu):
    """Sample counts on both sides of where dx loads its elements after the channel's sums, whole chunks and remainders."""
    test_row_sums(gpu, oracle, N, C, S, relu)


def test_more_rows_than_one_launch_takes(gpu):
    """40 x 2^23 rows of one element: the row sums take 2^24 workgroups, more than the 2^32 - 1 work-items of a launch. The
    reference is the same sums in order, channel-wise."""
    import torch

    import nnh
    N, C = 40, 1 << 23
    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.empty(N, C, device="cuda").normal_(generator=gen)
    w, b = (torch.empty(C, device="cuda").normal_(generator=gen) for _ in range(2))
    y, _, mean, var, inv = nnh.batchnorm_forward(x, w, b, EPS)
    s, q = (torch.zeros(C, dtype=torch.float64, device="cuda") for _ in range(2))
    for n in range(N):
        s += x[n].double()
    assert torch.equal(mean, (s / N).float())
    for n in range(N):
        d = x[n] - mean
        q += (d * d).double()
    assert torch.equal(var, (q / N).float())
    assert torch.equal(y, (x - mean) * (w * inv) + b)
    del y, d
    g = torch.empty(N, C, device="cuda").normal_(generator=gen)
    dw, db = torch.empty_like(w), torch.empty_like(b)
    nnh.batchnorm_backward(g, x, None, w, mean, inv, dw=dw, db=db)
    s.zero_()
    q.zero_()
    for n in range(N):
        s += g[n].double()
        q += (g[n] * (x[n] - mean)).double()
    assert torch.equal(db, s.float() + 0.0)
    assert torch.equal(dw, (q * inv.double()).float() + 0.0)
