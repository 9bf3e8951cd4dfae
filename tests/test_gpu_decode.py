"""Decode (one query, no dropout): cache lengths around the kernel's 64-key blocks, its eight waves'
512-key strides and the binding's slice rule, with plain and with streaming loads, and the merge of
more than 64 slices."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
# O is rounded to fp16 (2^-11 of values up to ~4 on N(0,1) inputs with few keys) and the scores are fp32.
O_TOL = 2e-3


def reference(q, k, v, keys):
    s = torch.matmul(q.float(), k[:, :, :keys].float().transpose(-1, -2).contiguous()) * 0.125
    return torch.matmul(torch.softmax(s, dim=-1), v[:, :, :keys].float()), torch.logsumexp(s, dim=-1)


@pytest.mark.parametrize("B,H,Sk", [(1, 3, 1), (1, 3, 63), (2, 3, 65), (1, 12, 512), (1, 12, 513), (1, 12, 1535),
                                    (1, 12, 1537), (2, 65, 1600), (8, 12, 3413), (8, 12, 3414), (3, 100, 1001)])
@pytest.mark.parametrize("hidden", [0, 1])
def test_decode_lengths(fa, B, H, Sk, hidden):
    """(8, 12, 3413) is the longest cache of at most 80 MiB and takes plain loads, (8, 12, 3414) streams.
    hidden: keys past the query's causal limit, in a cache that is a view of a longer one."""
    print(f"case decode B={B} H={H} Sk={Sk} hidden={hidden}", flush=True)
    g = torch.Generator().manual_seed(Sk + H)
    q = torch.randn(B, H, 1, 64, generator=g).half().to(DEV)
    k, v = (torch.randn(B, H, Sk + 7, 64, generator=g).half().to(DEV)[:, :, :Sk] for _ in range(2))
    keys = max(1, Sk - hidden)
    o, lse = fa.extension().fa_fwd_kv(q, k, v, True, 0.125, keys - 1, 0)
    ro, rl = reference(q, k, v, keys)
    assert (o.float() - ro).abs().max().item() <= O_TOL
    assert (lse - rl).abs().max().item() <= 1e-3


@pytest.mark.parametrize("nsplit", [5, 64, 65, 200])
def test_decode_many_slices(fa, nsplit):
    """The merge reads slices 64 at a time; slices past the cache's 157 blocks are empty."""
    print(f"case decode slices {nsplit}", flush=True)
    g = torch.Generator().manual_seed(nsplit)
    q = torch.randn(1, 2, 1, 64, generator=g).half().to(DEV)
    k, v = (torch.randn(1, 2, 10001, 64, generator=g).half().to(DEV) for _ in range(2))
    o, lse = fa.extension().fa_fwd_kv(q, k, v, True, 0.125, 10000, nsplit)
    ro, rl = reference(q, k, v, 10001)
    assert (o.float() - ro).abs().max().item() <= O_TOL
    assert (lse - rl).abs().max().item() <= 1e-3


def split_inputs(H, Sq, Sk):
    """q, k and V with a mean of 1: O is about 1 and a slice left out of n shows as 1/n of it."""
    g = torch.Generator().manual_seed(Sk)
    q = torch.randn(1, H, Sq, 64, generator=g).half().to(DEV)
    k, v = (torch.randn(1, H, Sk, 64, generator=g).add(m).half().to(DEV) for m in (0.0, 1.0))
    return q, k, v


@pytest.mark.parametrize("Sk", [1, 64, 65, 255, 256, 257, 320])
def test_decode_wave_counts(fa, Sk):
    """Slices of at most 256 keys take four waves, longer ones eight: the same bits as from a longer
    cache whose further keys are hidden (eight waves)."""
    print(f"case decode waves Sk={Sk}", flush=True)
    ext = fa.extension()
    q, k, v = split_inputs(3, 1, 600)
    o, lse = ext.fa_fwd_kv(q, k[:, :, :Sk], v[:, :, :Sk], True, 0.125, Sk - 1, 1)
    o8, lse8 = ext.fa_fwd_kv(q, k, v, True, 0.125, Sk - 1, 1)
    assert torch.equal(o, o8) and torch.equal(lse, lse8)
    ro, rl = reference(q, k, v, Sk)
    assert (o.float() - ro).abs().max().item() <= O_TOL * max(1.0, ro.abs().max().item() / 2)
    assert (lse - rl).abs().max().item() <= 1e-3


@pytest.mark.parametrize("Sq", [1, 5])
@pytest.mark.parametrize("lo", [1, 65, 129])
def test_merge_every_slice_count(fa, Sq, lo):
    """64 slice counts from lo on, every slice one 64-key tile that all queries see: the groups of 16
    lanes that share a query's slices end up with every possible remainder.  O against the reference
    (the smallest share is about 1/192, more than twice O_TOL)."""
    print(f"case slice counts {lo}..{lo + 63} Sq={Sq}", flush=True)
    ext = fa.extension()
    q, k, v = split_inputs(2, Sq, 64 * (lo + 63))
    for n in range(lo, lo + 64):
        kk, vv = k[:, :, :64 * n], v[:, :, :64 * n]
        o, lse = ext.fa_fwd_kv(q, kk, vv, False, 0.125, 0, n)
        ro, rl = reference(q, kk, vv, 64 * n)
        assert (o.float() - ro).abs().max().item() <= O_TOL, n
        assert (lse - rl).abs().max().item() <= 1e-3, n


@pytest.mark.parametrize("H,Sq,Sk,slices", [(8, 1, 4352, 17), (4, 1, 5376, 21), (8, 1, 5376, 21), (4, 1, 8448, 33),
                                            (4, 1, 8704, 34), (1, 1, 16128, 63), (4, 128, 8704, 17),
                                            (12, 128, 8704, 17), (6, 300, 10752, 21)])
def test_merge_of_automatic_slices(fa, H, Sq, Sk, slices):
    """Calls through the public entry point whose automatic slice count is no multiple of four."""
    print(f"case automatic slices H={H} Sq={Sq} Sk={Sk}", flush=True)
    q, k, v = split_inputs(H, Sq, Sk)
    o = fa.flash_attn_kvcache(q, k, v, causal=True)
    ext = fa.extension()
    for nsplit, tol in ((slices, 0.0), (1, O_TOL)):   # the count the rule takes, and the unsplit pass
        assert (o - ext.fa_fwd_kv(q, k, v, True, 0.125, Sk - Sq, nsplit)[0]).abs().max().item() <= tol, nsplit
    rows = torch.arange(Sq, device=DEV)[:, None] + (Sk - Sq)
    s = torch.matmul(q.float(), k.float().transpose(-1, -2).contiguous()) * 0.125
    s.masked_fill_(torch.arange(Sk, device=DEV)[None, :] > rows, float("-inf"))
    ro = torch.matmul(torch.softmax(s, dim=-1), v.float())
    assert (o.float() - ro).abs().max().item() <= O_TOL


@pytest.mark.parametrize("H,Sk,slices", [(12, 1535, 1), (12, 1536, 6), (79, 1536, 3), (80, 2047, 1), (80, 2048, 3),
                                         (96, 2047, 1), (128, 1536, 1), (128, 2048, 2), (129, 4096, 1)])
def test_decode_automatic_slices(fa, H, Sk, slices):
    """Both sides of the slice rule's lines: the same bits as with the count given."""
    print(f"case decode slice rule H={H} Sk={Sk}", flush=True)
    ext = fa.extension()
    q, k, v = split_inputs(H, 1, Sk)
    for a, b in zip(ext.fa_fwd_kv(q, k, v, True, 0.125, Sk - 1, 0), ext.fa_fwd_kv(q, k, v, True, 0.125, Sk - 1, slices)):
        assert torch.equal(a, b)


def test_decode_merge_edges(fa):
    """The merge of slices gives NaN where a slice's softmax met an infinite score (inf - inf), and a
    query that sees no key gives O = 0 and LSE = -inf with one slice and with several."""
    print("case decode merge edges", flush=True)
    ext = fa.extension()
    q = torch.ones(1, 1, 1, 64, device=DEV).half()
    k = torch.zeros(1, 1, 2000, 64, device=DEV).half()
    v = torch.ones_like(k)
    k[0, 0, 700, 3] = float("inf")
    o, _ = ext.fa_fwd_kv(q, k, v, True, 0.125, 1999, 4)
    assert torch.isnan(o).all()
    for nsplit in (1, 4):
        o, lse = ext.fa_fwd_kv(q, k, v, True, 0.125, -1, nsplit)
        assert (o == 0).all() and (lse == float("-inf")).all(), nsplit


@pytest.mark.parametrize("op,BH", [("decode", (1 << 23) + 3), ("forward", (1 << 24) - 1)])
def test_many_heads_of_one_key(fa, op, BH):
    """More heads than one launch of eight-wave decode workgroups can number, and the most the forward's
    grid can: with one key, O is V and LSE the score."""
    print(f"case one key op={op} BH={BH}", flush=True)
    g = torch.Generator(DEV).manual_seed(1)
    q, k, v = (torch.randn(1, BH, 1, 64, generator=g, device=DEV, dtype=torch.float16) for _ in range(3))
    ext = fa.extension()
    o, lse = ext.fa_fwd_kv(q, k, v, True, 0.125, 0, 0) if op == "decode" else ext.fa_fwd(q, k, v, 0.0, True, 0.125, 0)
    assert torch.equal(o, v)
    for part in (slice(0, 1000), slice((1 << 22) - 500, (1 << 22) + 500), slice(BH - 1000, BH)):
        s = (q[0, part, 0].float() * k[0, part, 0].float()).sum(-1) * 0.125
        assert (lse[0, part, 0] - s).abs().max().item() <= 1e-3
