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


@pytest.mark.parametrize("R,D", [(1, 4096), (17, 4095), (9, 4100), (1024, 4096), (1025, 4097), (200, 140), (1200, 300), (1030, 16380)])
def test_wide_columns(gpu, oracle, R, D):
    """Column sums alone on both sides of where a thread takes a column, and column blocks that do and do not divide by
    eight."""
    test_rows_and_columns(gpu, oracle, R, D)


@pytest.mark.parametrize("R,D", [(1, 1), (255, 1), (256, 1), (257, 2), (1025, 3), (511, 4), (513, 8), (129, 16), (300, 9), (151, 27),
                                 (65, 60), (33, 64), (31, 65), (63, 68), (5, 1000), (3, 2047), (3, 2048), (2, 2049), (4100, 25)])
def test_short_rows(gpu, oracle, R, D):
    """Rows around those that go up to 256 to a workgroup of 2048 floats, full workgroups and a last row alone."""
    test_rows_and_columns(gpu, oracle, R, D)


def test_more_rows_than_32_a_workgroup_take(gpu):
    """2^29 + 3 rows of two: with 32 rows a workgroup more than the 2^32 - 1 work-items of a launch. Rows at both ends and on
    either side of 2^29 against the same arithmetic."""
    import torch

    import nnh
    R = (1 << 29) + 3
    x = torch.empty(R, 2, device="cuda").uniform_(-1, 1, generator=torch.Generator(device="cuda").manual_seed(6))
    gm, bt = torch.tensor([1.5, -0.75], device="cuda"), torch.tensor([0.25, 2.0], device="cuda")
    y, mean, inv = nnh.layernorm_forward(x, gm, bt, EPS)
    for r0, r1 in ((0, 1 << 16), ((1 << 29) - (1 << 16), R)):
        xs = x[r0:r1].cpu().numpy()
        mu = (xs[:, 0] + xs[:, 1]) / np.float32(2)
        d = xs - mu[:, None]
        iv = np.float32(1) / np.sqrt((d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) / np.float32(2) + np.float32(EPS))
        want = d * iv[:, None] * gm.cpu().numpy() + bt.cpu().numpy()
        for got, ref, what in ((mean, mu, "mean"), (inv, iv, "inv_std"), (y, want, "y")):
            assert_same(got[r0:r1].cpu().numpy(), ref, (what, r0))
    # the gradient of the same rows: more workgroups than one launch takes
    g = torch.empty(R, 2, device="cuda").uniform_(-1, 1, generator=torch.Generator(device="cuda").manual_seed(7))
    dx = y.zero_()
    nnh.layernorm_backward(g, x, gm, mean, inv, dx=dx)
    two = np.float32(2)
    for r0, r1 in ((0, 1 << 16), ((1 << 29) - (1 << 20), (1 << 29) - (1 << 19)), ((1 << 29) - (1 << 16), R)):
        xs, gs, mu, iv = (t[r0:r1].cpu().numpy() for t in (x, g, mean, inv))
        xh, dh = (xs - mu[:, None]) * iv[:, None], gs * gm.cpu().numpy()
        sa = np.float32(0) + dh[:, 0] + dh[:, 1]
        p = dh * xh
        sb = np.float32(0) + p[:, 0] + p[:, 1]
        want = (iv / two)[:, None] * (two * dh - sa[:, None] - xh * sb[:, None])
        assert_same(dx[r0:r1].cpu().numpy(), want + np.float32(0), ("dx", r0))
