"""The bias gradient of a three-dimensional gradient (two ordered sums) at the edges of its kernels: axis-0 counts around
the sixteen loads in flight, axis-1 counts around the 256 threads, the 32-wide blocks of the second sum and the largest the
kernel takes, aligned quads of columns and not. The sums are chains in a fixed order, so the tolerance is zero."""
import numpy as np
import pytest

from helpers import assert_same
from nnh import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r0,r1,n", [(1, 1, 4), (15, 255, 8), (16, 256, 36), (17, 257, 4), (33, 512, 20), (5, 31, 6), (3, 33, 68),
                                     (32, 64, 5)])
@pytest.mark.parametrize("first", [True, False])
def test_two_axis_bias_gradient(gpu, oracle, r0, r1, n, first):
    import torch

    import nnh
    g, old = synth.normal(41, (r0, r1, n)), synth.normal(42, (n,))
    s = oracle.sum_axis0(oracle.sum_axis0(g))
    want = s + np.float32(0.0) if first else old + s
    for off in (0, 1):  # off floats past a 16-byte boundary
        buf = torch.empty(g.size + off, device="cuda")
        buf[off:] = torch.from_numpy(g.ravel()).cuda()
        db = torch.from_numpy(old).cuda()
        x, w = torch.zeros(r0, r1, 4, device="cuda"), torch.zeros(n, 4, device="cuda")
        nnh.linear_backward(buf[off:].view(r0, r1, n), x, w, db=db, db_first=first)
        assert_same(db.cpu().numpy(), want, (r0, r1, n, first, off))


@pytest.mark.parametrize("r0,r1,n", [(1, 2, 2996), (14, 5, 3000), (23, 3, 3004), (17, 123, 3004), (18, 3, 3004), (7, 124, 3004),
                                     (31, 64, 12), (46, 130, 4184), (46, 140, 3596), (8, 24, 512)])
@pytest.mark.parametrize("first", [True, False])
def test_two_axis_bias_gradient_routes(gpu, oracle, r0, r1, n, first):
    """Both sides of where four columns a workgroup are taken, and every count of a last batch of loads."""
    test_two_axis_bias_gradient(gpu, oracle, r0, r1, n, first)


def test_more_columns_than_one_launch_takes_by_four(gpu):
    """2^26 columns, four of them a workgroup, would be 2^32 work-items."""
    import torch

    import nnh
    r0, n = 18, 1 << 26
    g = torch.empty(r0, 1, n, device="cuda").uniform_(-1, 1, generator=torch.Generator(device="cuda").manual_seed(9))
    x, w = torch.zeros(r0, 1, 1, device="cuda"), torch.zeros(n, 1, device="cuda")
    db = torch.empty(n, device="cuda")
    nnh.linear_backward(g, x, w, db=db)
    want = torch.zeros(n, device="cuda")
    for i in range(r0):
        want += g[i, 0]
    assert torch.equal(db, want)
