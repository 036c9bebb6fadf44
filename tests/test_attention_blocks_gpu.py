"""The fused attention kernels (head width 64) at the edges of their blocks: query counts around 32 rows, key counts around
the 16-key tiles, the 64 keys of a wave and the largest the kernels take, whole and partial groups of four steps, with the
causal limit and the padding mask. Every element is one chain in a fixed order, so the tolerance is zero."""
import numpy as np
import pytest

from helpers import assert_same
from nnh import synth

pytestmark = pytest.mark.gpu

SIZES = [(1, 4), (16, 12), (31, 16), (32, 20), (33, 60), (48, 64), (65, 68), (7, 124), (40, 132), (64, 252), (96, 256)]


@pytest.mark.parametrize("tq,tk,causal", [(tq, tk, False) for tq, tk in SIZES] +
                         [(t, t, True) for t in (4, 16, 32, 36, 60, 64, 68, 100, 196, 252, 256)])
@pytest.mark.parametrize("masked", [False, True])
def test_fused_attention_block_edges(gpu, oracle, tq, tk, causal, masked):
    import torch

    import nnh
    n, heads = 3, 2
    d = 64 * heads
    q, k, v, g = (synth.normal(50 + i, (n, t, d)) for i, t in enumerate((tq, tk, tk, tq)))
    mask = None
    if masked:  # one row of keys whole, one with a few, one with none
        mask = np.ones((n, tk), np.float32)
        mask[1, (tk + 2) // 3:] = 0
        mask[2] = 0

    def dev(a):
        return None if a is None else torch.from_numpy(a).cuda()

    dq, dk, dv, dg, dm = (dev(a) for a in (q, k, v, g, mask))
    out, probs = nnh.attention_forward(dq, dk, dv, heads, mask=dm, causal=causal)
    grads = [torch.zeros_like(t) for t in (dq, dk, dv)]  # the oracle adds to zeros
    nnh.attention_backward(dg, dq, dk, dv, probs, heads, dm, causal, grads[0], False, grads[1], False, grads[2], False)
    want_out, want_probs = oracle.attention_forward(q, k, v, heads, mask, causal)
    want = oracle.attention_backward(g, q, k, v, want_probs, heads, mask, causal)
    assert_same(out.cpu().numpy(), want_out, (tq, tk, "out"))
    assert_same(probs.cpu().numpy(), want_probs, (tq, tk, "probs"))
    for name, got, w in zip(("dq", "dk", "dv"), grads, want):
        assert_same(got.cpu().numpy(), w, (tq, tk, name))


def test_more_blocks_than_one_launch_takes(gpu, oracle):
    """2^23 (sample, head) pairs of 33 queries: 2^24 blocks of 32 rows, more than the 2^32 - 1 work-items of a launch. The first
    sample, the last and those on either side of the second launch against the oracle, one between them against equal scores."""
    import torch

    import nnh
    n, heads, tq, tk, d = 1 << 19, 16, 33, 4, 1024
    if torch.cuda.mem_get_info()[0] < 190e9:
        pytest.skip("needs 180 GB of device memory")
    q, k, v = torch.zeros(n, tq, d, device="cuda"), torch.zeros(n, tk, d, device="cuda"), torch.zeros(n, tk, d, device="cuda")
    samples = (0, 1, n - 2, n - 1)
    host = {i: [synth.normal(90 + i % 7, (1, t, d)) for t in (tq, tk, tk)] for i in samples}
    for i, parts in host.items():
        for t, a in zip((q, k, v), parts):
            t[i] = torch.from_numpy(a[0])
    out, probs = nnh.attention_forward(q, k, v, heads)
    for i, (hq, hk, hv) in host.items():
        want_out, want_probs = oracle.attention_forward(hq, hk, hv, heads, None, False)
        assert_same(out[i].cpu().numpy(), want_out[0], (i, "out"))
        assert_same(probs[i].cpu().numpy(), want_probs[0], (i, "probs"))
    assert torch.all(probs[n // 2] == 0.25) and torch.all(probs[n - 3] == 0.25)
    # the scores' gradient takes the same blocks; the keys' gradient alone, since dq would be another 71 GB
    g = out
    want = {i: oracle.attention_backward(out[i:i + 1].cpu().numpy(), *host[i], probs[i:i + 1].cpu().numpy(), heads, None, False)
            for i in samples}
    dk = torch.empty_like(k)
    nnh.attention_backward(g, q, k, v, probs, heads, dk=dk)
    for i in samples:
        assert_same(dk[i].cpu().numpy(), want[i][1][0] + np.float32(0), (i, "dk"))
    del q, k, v, g, out, probs, dk
    torch.cuda.empty_cache()
