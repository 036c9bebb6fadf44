"""The ring GEMM (gemm_ring.hpp) where it can go wrong, bit for bit against the oracle: every tile shape forced at one
row and column below, at and past its tile, depths around its stages (fewer stages than the ring holds, a partial last
stage of every remainder class, the accumulate point at 256), 16-byte and 4-byte loads; and, through its own route, row
sums, the GELU epilogue and batches. The outputs are whole sums in a fixed order, so the tolerance is zero."""
import numpy as np
import pytest

from helpers import SENTINEL, Problem, assert_same, gpu_sgemm, oracle_sgemm
from nnh import synth

pytestmark = pytest.mark.gpu


def ring_configs():
    import nnh
    return {nm: i for i, nm in enumerate(nnh.gemm_configs()) if nm.startswith("ring ")}


def host(t):
    import torch
    torch.cuda.synchronize()
    return t.cpu().numpy()


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_ring_edges(gpu, oracle, ta, tb):
    seed = 91000
    for name, cfg in ring_configs().items():
        bm, bn = (int(v) for v in name.split()[1].split("_")[0].split("x"))
        # (m, n, k, pad): pad 0 with sizes a multiple of four takes 16-byte loads, the others one float a lane
        for m, n, k, pad in ((bm, bn, 32, 0), (bm + 4, bn - 4, 100, 0), (bm - 1, bn + 1, 33, 0), (4, 8, 4, 0), (1, 1, 1, 0),
                             (bm, bn + 4, 256, 4), (5, bn, 288, 0), (bm + 16, 12, 300, 0), (7, 9, 95, 1), (bm + 1, 3, 161, 3),
                             (20, 24, 500, 0)):
            for acc in (0, 1):
                p = Problem(ta, tb, m, n, k, pad, seed)
                seed += 1
                want = oracle_sgemm(oracle, p, acc)
                assert_same(gpu_sgemm(p, acc, config=cfg), want, (name, ta, tb, m, n, k, pad, acc))


@pytest.mark.parametrize("M,K,n", [(200, 904, 900), (133, 901, 899)])
def test_ring_row_sums(gpu, oracle, M, K, n):
    """A 2-D weight gradient that takes the ring: dW = G^T X with db folded in, fresh and added."""
    import torch

    import nnh
    x, w, g = synth.normal(1, (M, K)), synth.normal(2, (n, K)), synth.normal(3, (M, n))
    dw0, db0 = synth.normal(4, (n, K)), synth.normal(5, (n,))
    for first in (True, False):
        want = oracle.linear_backward(g, x, w, dw=dw0, dw_first=first, db=db0, db_first=first)
        dw, db = torch.from_numpy(dw0).cuda(), torch.from_numpy(db0).cuda()
        nnh.linear_backward(*(torch.from_numpy(a).cuda() for a in (g, x, w)), dw=dw, dw_first=first, db=db, db_first=first)
        assert_same(host(dw), want[1], ("dw", M, K, n, first))
        assert_same(host(db), want[2], ("db", M, K, n, first))


@pytest.mark.parametrize("M,K,n", [(1000, 128, 900), (777, 99, 1021)])
def test_ring_gelu(gpu, oracle, M, K, n):
    import torch

    import nnh
    L, P = nnh.lib(), nnh._ptr
    x, w, b = synth.normal(11, (M, K)), synth.normal(12, (n, K)), synth.normal(13, (n,))
    h0 = oracle.linear_forward(x, w, b)
    y0, t0 = oracle.gelu_forward(h0)
    xd, wd, bd = (torch.from_numpy(a).cuda() for a in (x, w, b))
    h, y, t = (torch.full((M, n), float(SENTINEL), device="cuda") for _ in range(3))
    nnh.check(L.nnh_linear_gelu_forward(P(xd), M, K, P(wd), n, P(bd), P(h), P(y), P(t), nnh._stream(None)))
    for got, want, what in ((h, h0, "h"), (y, y0, "y"), (t, t0, "tanh")):
        assert_same(host(got), want, (what, M, K, n))


@pytest.mark.parametrize("shape", [(3, 500, 100, 450), (5, 449, 130, 451)])
def test_ring_batches(gpu, oracle, shape):
    """A batch of products, the right operand broadcast; the tiles of different matrices share one launch."""
    import torch

    import nnh
    nb, m, k, n = shape
    a, b = synth.normal(21, (nb, m, k)), synth.normal(22, (nb, k, n))
    got = host(nnh.matmul(torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()))
    for i in range(nb):
        want = oracle.sgemm(0, 0, m, n, k, a[i], k, b[i], n, np.zeros((m, n), np.float32), n, 0)
        assert_same(got[i], want, (shape, i))


@pytest.mark.parametrize("M,K,n", [(256, 256, 256), (255, 260, 253), (128, 517, 130), (300, 900, 131), (640, 324, 256),
                                   (250, 33, 7), (129, 96, 10)])
@pytest.mark.parametrize("first", [True, False])
def test_ring_pairs(gpu, oracle, M, K, n, first):
    """Both gradients of a layer in one grid (the smallest sizes: dW with its row sums on a few tiles), 16-byte and 4-byte
    loads, fresh and added, with and without the bias."""
    import torch

    import nnh
    x, w, g = synth.normal(31, (M, K)), synth.normal(32, (n, K)), synth.normal(33, (M, n))
    dx0, dw0, db0 = synth.normal(34, (M, K)), synth.normal(35, (n, K)), synth.normal(36, (n,))
    xd, wd, gd = (torch.from_numpy(a).cuda() for a in (x, w, g))
    want = oracle.linear_backward(g, x, w, dx=dx0, dx_first=first, dw=dw0, dw_first=first, db=db0, db_first=first)
    for bias in (True, False):
        dx, dw, db = (torch.from_numpy(a).cuda() for a in (dx0, dw0, db0))
        nnh.linear_backward(gd, xd, wd, dx=dx, dx_first=first, dw=dw, dw_first=first, db=db if bias else None, db_first=first)
        for got, ref, what in ((dx, want[0], "dx"), (dw, want[1], "dw"), (db, want[2] if bias else db0, "db")):
            assert_same(host(got), ref, (what, M, K, n, first, bias))
    b = np.ascontiguousarray(w.T)  # the same product as a matmul: dA = G B^T, dB = A^T G
    da, dbm = (torch.from_numpy(a).cuda() for a in (dx0, np.ascontiguousarray(dw0.T)))
    nnh.matmul_backward(gd, xd, torch.from_numpy(b).cuda(), da=da, da_first=first, db=dbm, db_first=first)
    want = oracle.linear_backward(g, x, w, dx=dx0, dx_first=first, dw=dw0, dw_first=first)
    assert_same(host(da), want[0], ("da", M, K, n, first))
    assert_same(host(dbm), want[1].T, ("db matmul", M, K, n, first))


# (ta, tb, batch, m, n, k): both sides of the lines between the ring and the VALU, chain and tile kernels
ROUTES = [(0, 1, 1, 256, 512, 784), (0, 1, 1, 512, 200, 511), (0, 1, 1, 20, 5352, 320), (0, 1, 70, 5, 5, 300), (0, 1, 1, 33, 1934, 901),
          (0, 0, 1, 256, 512, 272), (0, 0, 1, 255, 512, 276), (0, 0, 1, 6, 2976, 256), (0, 0, 549, 4, 2, 260), (0, 0, 1, 64, 1500, 128),
          (0, 0, 4, 2, 4032, 112), (0, 0, 11, 5, 5553, 112), (0, 1, 200, 1, 128, 128), (0, 1, 111, 64, 126, 103), (0, 1, 9, 17, 700, 113),
          (1, 0, 1, 354, 1744, 208), (1, 0, 1, 512, 784, 256), (1, 0, 1, 516, 2048, 176), (1, 0, 3, 64, 128, 101), (1, 1, 2, 40, 900, 127),
          (0, 1, 520, 9, 33, 200), (0, 0, 600, 3, 40, 176), (0, 0, 600, 3, 40, 175), (0, 0, 521, 16, 16, 129), (0, 1, 9, 3888, 3, 96)]


@pytest.mark.parametrize("ta,tb,batch,m,n,k", ROUTES)
def test_routes_of_padded_and_small_products(gpu, oracle, ta, tb, batch, m, n, k):
    import torch

    import nnh
    a, b = synth.normal(61, (batch,) + ((k, m) if ta else (m, k))), synth.normal(62, (batch,) + ((n, k) if tb else (k, n)))
    c0 = synth.normal(63, (batch, m, n))
    ad, bd = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    strides = nnh.make_batch((batch,), (m * k,), (k * n,), (m * n,)) if batch > 1 else None
    for acc in (0, 1):
        c = torch.from_numpy(c0).cuda()
        nnh.sgemm_batched(ta, tb, m, n, k, ad, m if ta else k, bd, k if tb else n, c, n, accumulate=bool(acc), batch=strides)
        got = host(c)
        for i in sorted({0, batch // 2, batch - 1}):
            want = oracle.sgemm(ta, tb, m, n, k, a[i], m if ta else k, b[i], k if tb else n, c0[i].copy(), n, acc)
            assert_same(got[i], want, (ta, tb, batch, m, n, k, i, acc))


def test_more_tiles_than_one_launch_takes(gpu, oracle):
    """2^23 products of one 64 x 96 matrix with columns: on 32 x 32 tiles 2^24 workgroups, more than the 2^32 - 1 work-items of
    a launch."""
    import torch

    import nnh
    batch, m, n, k = 1 << 23, 64, 1, 96
    a = synth.normal(71, (m, k))
    b = torch.empty(batch, k, device="cuda").uniform_(-1, 1, generator=torch.Generator(device="cuda").manual_seed(8))
    c = torch.full((batch, m), float(SENTINEL), device="cuda")
    nnh.sgemm_batched(0, 0, m, n, k, torch.from_numpy(a).cuda(), k, b, n, c, n,
                      batch=nnh.make_batch((batch,), (0,), (k * n,), (m * n,)))
    for i in (0, 1, batch // 2, batch - 2, batch - 1):
        want = oracle.sgemm(0, 0, m, n, k, a, k, b[i].cpu().numpy(), n, np.zeros((m, n), np.float32), n, 0)
        assert_same(host(c[i]).reshape(m, n), want, i)


@pytest.mark.parametrize("M,K,n", [(128, 512, 512), (129, 300, 301), (191, 512, 128), (192, 256, 260), (320, 256, 256), (321, 255, 257),
                                   (700, 1000, 900), (701, 1001, 899), (4100, 272, 260)])
def test_row_sums_among_the_products(gpu, oracle, M, K, n):
    """db beside dW at depths of two and more stages of each tile, whole and with a remainder: the sums' operands are read a
    group of 16 depths ahead, across stages."""
    test_ring_row_sums(gpu, oracle, M, K, n)


@pytest.mark.parametrize("M,K,n", [(33056, 127, 520), (41952, 100, 1000)])
def test_narrow_layer_backward(gpu, oracle, M, K, n):
    """dX of 2^22 outputs and fewer than 128 columns beside a dW of some 32 x 32 tiles: a pair, and on its own."""
    import torch

    import nnh
    x, w, g = synth.normal(81, (M, K)), synth.normal(82, (n, K)), synth.normal(83, (M, n))
    want = oracle.linear_backward(g, x, w, dx=np.zeros_like(x), dw=np.zeros_like(w), db=np.zeros(n, np.float32))
    xd, wd, gd = (torch.from_numpy(a).cuda() for a in (x, w, g))
    dx, dw, db = torch.empty_like(xd), torch.empty_like(wd), torch.empty(n, device="cuda")
    nnh.linear_backward(gd, xd, wd, dx=dx, dw=dw, db=db)
    for got, ref, what in ((dx, want[0], "dx"), (dw, want[1], "dw"), (db, want[2], "db")):
        assert_same(host(got), ref, what)


@pytest.mark.parametrize("bias", ["none", "col", "row"])
@pytest.mark.parametrize("relu", [False, True])
def test_ring_epilogue(gpu, oracle, bias, relu):
    """Every tile's store with a bias down the columns or along the rows, ReLU with its flags, fresh and accumulated below and
    past 256 deep: 16-byte aligned rows, ragged ones, and a batch whose C and flags have a stride between matrices."""
    import torch

    import nnh
    mode = {"none": nnh.BIAS_NONE, "col": nnh.BIAS_COL, "row": nnh.BIAS_ROW}[bias]
    seed = 93000
    for name, cfg in ring_configs().items():
        bm, bn = (int(v) for v in name.split()[1].split("_")[0].split("x"))
        for batch, m, n, k, pad in ((1, bm, bn + 4, 40, 0), (1, bm - 1, bn + 3, 300, 1), (3, bm + 5, bn - 2, 33, 3), (2, bm, bn, 288, 0)):
            lda, ldb, ldc = k + pad, n + pad, n + pad
            a, b = synth.normal(seed, (batch, m, lda)), synth.normal(seed + 1, (batch, k, ldb))
            gap = 8  # floats of C between two matrices that belong to neither
            c0 = synth.normal(seed + 2, (batch, m * ldc + gap))
            bv = synth.normal(seed + 3, (n if bias == "col" else m,))
            seed += 4
            for acc in (0, 1):
                c, flags = torch.from_numpy(c0).cuda(), torch.full(c0.shape, 7, dtype=torch.uint8, device="cuda")
                bd = torch.from_numpy(bv).cuda()
                ep = nnh.make_epilogue(mode, bd if bias != "none" else None, relu, flags if relu else None)
                nnh.sgemm_batched(0, 0, m, n, k, torch.from_numpy(a).cuda(), lda, torch.from_numpy(b).cuda(), ldb, c, ldc, acc,
                                  nnh.make_batch((batch,), (m * lda,), (k * ldb,), (m * ldc + gap,)), ep, cfg)
                want, alive = c0.copy(), np.full(c0.shape, 7, np.uint8)
                for i in range(batch):
                    full = oracle.sgemm(0, 0, m, n, k, a[i], lda, b[i], ldb, c0[i, :m * ldc].reshape(m, ldc).copy(), ldc, acc)
                    v = full[:, :n]
                    v = v + bv[None, :] if bias == "col" else v + bv[:, None] if bias == "row" else v
                    if relu:
                        alive[i, :m * ldc].reshape(m, ldc)[:, :n] = v > 0
                        v = np.where(v > 0, v, np.float32(0))
                    want[i, :m * ldc].reshape(m, ldc)[:, :n] = v
                what = (name, bias, relu, batch, m, n, k, pad, acc)
                assert_same(host(c), want, what)
                if relu:
                    assert np.array_equal(host(flags), alive), what


@pytest.mark.parametrize("M,K,n", [(1024, 512, 768), (777, 130, 1021)])
def test_ring_residual(gpu, oracle, M, K, n):
    """A layer with its residual through the ring, fresh and in the residual's place, with -0, infinities and NaN in it."""
    import torch

    import nnh
    x, w, b, r = synth.normal(41, (M, K)), synth.normal(42, (n, K)), synth.normal(43, (n,)), synth.normal(44, (M, n))
    r[0, :4] = [-0.0, np.inf, -np.inf, np.nan]
    want = r + oracle.linear_forward(x, w, b)
    xd, wd, bd, rd = (torch.from_numpy(a).cuda() for a in (x, w, b, r))
    assert_same(host(nnh.linear_forward_add(xd, wd, bd, rd)), want, ("residual", M, K, n), nan_equal=True)
    nnh.linear_forward_add(xd, wd, bd, rd, out=rd)
    assert_same(host(rd), want, ("in place", M, K, n), nan_equal=True)


@pytest.mark.parametrize("M,K,n", [(1000, 256, 900), (300, 160, 900), (1700, 100, 1000), (1000, 252, 900), (61, 128, 900)])
def test_gelu_routes(gpu, oracle, M, K, n):
    """Aligned layers with GELU on both sides of the line between the ring and the chain kernel."""
    test_ring_gelu(gpu, oracle, M, K, n)
