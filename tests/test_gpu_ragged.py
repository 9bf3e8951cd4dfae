"""Causal lengths whose query blocks do not fill: the blocks are moved down by whole 64-query groups
and the partial one is the head's first (query_block_base), with enough heads for the narrow forward."""
import numpy as np
import pytest
import torch

from oracle import fa2_oracle as orc

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize("p", [0.0, 0.1])
@pytest.mark.parametrize("B,H,S", [(64, 8, 130),     # forward and narrow dQ blocks moved by 64
                                   (44, 8, 260),     # forward by 64, two-block dQ by 192
                                   (16, 8, 1030)])   # forward by 64, two-block dQ by 192, longer heads
def test_partial_first_query_block(fa, B, H, S, p):
    """Every row of every head is written (finite, on outputs taken from NaN-filled memory), the first
    and last heads match the fp64 oracle (O 2e-3 over 1/(1-p), gradients 1e-2 relative: the bars of the
    other parity tests), and with dropout the keep words give the hash path's bits."""
    print(f"case partial first block B={B} H={H} S={S} p={p}", flush=True)
    ext = fa.extension()
    g = torch.Generator().manual_seed(S)
    q, k, v, do = (torch.randn(B, H, S, 64, generator=g).half().to(DEV) for _ in range(4))
    for _ in range(6):   # the outputs' memory: blocks of their size, NaN, returned to the allocator
        torch.full_like(q, float("nan"))
    o, lse = ext.fa_fwd(q, k, v, p, True, 0.125, 77)
    dq, dk, dv = ext.fa_bwd(q, k, v, o, lse, do, p, True, 0.125, 77, 7)
    outs = (o, lse, dq, dk, dv)
    for t in outs:
        assert torch.isfinite(t).all()
    if p > 0:
        o2, lse2, mask = ext.fa_fwd_mask(q, k, v, p, True, 0.125, 77)
        grads = ext.fa_bwd(q, k, v, o2, lse2, do, p, True, 0.125, 77, 7, mask=mask)
        for a, b in zip((o, lse, dq, dk, dv), (o2, lse2, *grads)):
            assert torch.equal(a, b)
    for b, h in ((0, 0), (B - 1, H - 1)):
        qn, kn, vn, don = (t[b, h][None, None].float().cpu().numpy() for t in (q, k, v, do))
        keep = None
        if p > 0:
            keep = orc.dropout_keep(77, np.arange(S)[:, None], np.arange(S)[None, :], b * H + h, p)[None, None]
        ro, rl = orc.attention_dense_fwd(qn, kn, vn, causal=True, scale=0.125, keep=keep, p=p)
        rg = orc.attention_bwd(qn, kn, vn, ro, rl, don, causal=True, scale=0.125, keep=keep, p=p)[:3]
        got = [t[b, h][None, None].float().cpu().numpy() for t in outs]
        assert orc.max_abs(got[0], ro) <= 2e-3 / (1.0 - p) and orc.max_abs(got[1], rl) <= 1e-3
        for name, a, r in zip(("dQ", "dK", "dV"), got[2:], rg):
            assert orc.rel_l2(a, r) <= 1e-2, (name, b, h)


@pytest.mark.parametrize("B,H,S,causal", [(43, 3, 140, True),    # 129 heads, numbered as 136: grouped orders
                                          (33, 4, 1100, True),   # 132 heads: plain forward, two-block dQ
                                          (43, 3, 150, False)])
def test_padded_head_numbers(fa, B, H, S, causal):
    """B*H no multiple of 8 from 128 heads on: every head of every output is written and gives the bits
    it gives alone in a small batch (up to 127 heads the grid numbers the heads as they are); the forward
    loops and both dQ kernels agree bit for bit."""
    print(f"case padded heads B={B} H={H} S={S} causal={causal}", flush=True)
    ext = fa.extension()
    g = torch.Generator().manual_seed(B * S)
    q, k, v, do = (torch.randn(B, H, S, 64, generator=g).half().to(DEV) for _ in range(4))
    for p in (0.0, 0.1):
        for _ in range(6):
            torch.full_like(q, float("nan"))
        o, lse = ext.fa_fwd(q, k, v, p, causal, 0.125, 5)
        outs = (o, lse, *ext.fa_bwd(q, k, v, o, lse, do, p, causal, 0.125, 5, 7))
        for t in outs:
            assert torch.isfinite(t).all()
        n = 5   # the first batches alone (the dropout hash numbers heads from 0 in both calls)
        a = [t[:n].contiguous() for t in (q, k, v, do)]
        o1, l1 = ext.fa_fwd(*a[:3], p, causal, 0.125, 5)
        alone = (o1, l1, *ext.fa_bwd(*a[:3], o1, l1, a[3], p, causal, 0.125, 5, 7))
        for x, y in zip(outs, alone):
            assert torch.equal(x[:n], y)
        if p == 0:   # and the last batches, whose workgroups sit beside the ones with no head
            a = [t[-n:].contiguous() for t in (q, k, v, do)]
            o1, l1 = ext.fa_fwd(*a[:3], p, causal, 0.125, 5)
            alone = (o1, l1, *ext.fa_bwd(*a[:3], o1, l1, a[3], p, causal, 0.125, 5, 7))
            for x, y in zip(outs, alone):
                assert torch.equal(x[-n:], y)


@pytest.mark.parametrize("S,causal", [(1025, True), (1300, False), (2100, True)])
def test_narrow_dq_on_small_long_grids(fa, S, causal):
    """Longer sequences whose two-block dQ grid leaves slots empty take the narrow kernel: a few heads
    give the bits that the same heads give in a batch large enough for the two-block kernel."""
    print(f"case small long dQ grid S={S} causal={causal}", flush=True)
    ext = fa.extension()
    g = torch.Generator().manual_seed(S)
    B = 520 // ((S + 255) // 256 * 4) + 1   # more than 15/16 of 512 two-block workgroups at H = 4
    q, k, v, do = (torch.randn(B, 4, S, 64, generator=g).half().to(DEV) for _ in range(4))
    for p in (0.0, 0.1):
        o, lse = ext.fa_fwd(q, k, v, p, causal, 0.125, 9)
        big = ext.fa_bwd(q, k, v, o, lse, do, p, causal, 0.125, 9, 7)
        small = ext.fa_bwd(q[:2], k[:2], v[:2], o[:2], lse[:2], do[:2], p, causal, 0.125, 9, 7)
        for x, y in zip(big, small):
            assert torch.equal(x[:2], y)
