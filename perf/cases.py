"""The workloads the attention path is timed on: what its users have it do.

Four kinds of call, each through the module's public entry points:

  train   causal attention of one layer, forward and backward, from the views
          the trainer makes: q and k [B,S,H,D] tensors seen as [B,H,S,D], v a
          view of the fused qkv projection, the output gradient in the same
          order.  Without dropout through ``flash_attn_v100`` and autograd; with
          dropout through the extension's ops that the autograd wrapper calls
          (forward with keep words, backward reading them), where the seed is an
          argument and so the mask is the same on every pass.
  rope    rotary embedding of q and k (views of the fused qkv projection),
          forward and backward.
  chunk   inference: S_q new queries against S_k cached keys (a prompt, or a
          prefill chunk), causal aligned bottom-right, or non-causal through the
          ``sdpa`` shim.
  decode  inference: one query against S_k cached keys.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "universal-lm-trainer_amd"))
import flash_attn_v100_cuda as fa  # noqa: E402

D = 64
SCALE = D ** -0.5
DEV = "cuda"


def _train(name, B, H, S, p=0.0, causal=True, outliers=False):
    case = {"kind": "train", "B": B, "H": H, "S": S, "p": p, "causal": causal, "outliers": outliers}
    return dict(case, name=name) if name else case


def _rope(name, B, H, S):
    case = {"kind": "rope", "B": B, "H": H, "S": S}
    return dict(case, name=name) if name else case


def _infer(name, kind, B, H, Sq, Sk, causal=True, spare=0):
    # spare: positions the cache is allocated beyond the S_k in use
    case = {"kind": kind, "B": B, "H": H, "Sq": Sq, "Sk": Sk, "causal": causal, "spare": spare}
    return dict(case, name=name) if name else case


def listed():
    return [
        # A debugging run or a very small model: three short launches, latency and host work.
        _train("train_b2_h4_s256", 2, 4, 256),
        # The trainer's token budget (32k tokens a step) spent on its shortest common bucket.
        _train("train_b64_h12_s512", 64, 12, 512),
        # A token-budget bucket as the sampler makes them: a length that is no multiple of 64, an odd batch.
        _train("train_b31_h12_s1050", 31, 12, 1050),
        # The headline training shape: the full context length.
        _train("train_b8_h12_s4096", 8, 12, 4096),
        # Pretraining runs with dropout 0.1: a middle bucket and a ragged longer one.
        _train("train_drop_b32_h12_s1024", 32, 12, 1024, p=0.1),
        _train("train_drop_b15_h12_s2050", 15, 12, 2050, p=0.1),
        # Rotary embedding of one layer at the headline shape.
        _rope("rope_b8_h12_s4096", 8, 12, 4096),
        # A prompt of one user at the start of a generation.
        _infer("prefill_b1_h12_s200", "chunk", 1, 12, 200, 200),
        # Chunked prefill of a batch against a full context.
        _infer("chunk_b8_h12_q512_k4096", "chunk", 8, 12, 512, 4096),
        # One generated token: one user early in a conversation, a batch at full context, long contexts.
        _infer("decode_b1_h12_k1000", "decode", 1, 12, 1, 1000),
        _infer("decode_b8_h12_k4096", "decode", 8, 12, 1, 4096),
        _infer("decode_b8_h12_k16384", "decode", 8, 12, 1, 16384, spare=128),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "train", "train_drop", "rope", "chunk", "decode", "decode"])
    H = rng.choice([4, 8, 12, 12, 16])
    if kind in ("train", "train_drop"):
        S = _logint(rng, 100, 4096)
        tokens = _logint(rng, 1024, 32768)
        B = max(1, min(tokens // S, 96 * 4096 * 4096 // (H * S * S)))
        return _train(None, B, H, S, p=0.1 if kind == "train_drop" else 0.0, causal=rng.random() < 0.85,
                      outliers=rng.random() < 0.2)
    if kind == "rope":
        S = _logint(rng, 50, 4096)
        return _rope(None, max(1, min(_logint(rng, 256, 32768), 96 * 4096 // H) // S), H, S)
    if kind == "chunk":
        Sk = _logint(rng, 64, 8192)
        Sq = min(Sk, _logint(rng, 16, 2048))
        B = _logint(rng, 1, 16)
        B = max(1, min(B, 96 * 2048 * 4096 // (H * Sq * Sk)))
        return _infer(None, kind, B, H, Sq, Sk, causal=rng.random() < 0.8, spare=rng.choice([0, 0, 64, 333]))
    Sk = _logint(rng, 100, 32768)
    B = max(1, min(_logint(rng, 1, 64), 96 * 16384 // (H * Sk)))
    return _infer(None, kind, B, H, 1, Sk, spare=rng.choice([0, 0, 64, 333]))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _tables(S, d_model=768, base=10000.0):
    """cos / sin [S, 64] as the trainer builds them: frequencies over d_model, first head_dim columns."""
    inv = 1.0 / (base ** (torch.arange(0, d_model, 2, device=DEV).float() / d_model))
    ang = torch.outer(torch.arange(S, device=DEV).float(), inv)
    ang = torch.cat((ang, ang), dim=-1)[:, :D]
    return ang.cos().contiguous(), ang.sin().contiguous()


def prepare(case, seed):
    g = torch.Generator(DEV).manual_seed(int(seed))
    B, H = case["B"], case["H"]
    kind = case["kind"]
    if kind == "train":
        S = case["S"]
        q, k, do = (_randn(g, B, S, H, D).half().transpose(1, 2) for _ in range(3))
        if case["outliers"]:   # one query row in a hundred is eight times larger
            rows = torch.rand(B, H, S, 1, generator=g, device=DEV) < 0.01
            q = torch.where(rows, q * 8, q)
        v = _randn(g, B, S, 3, H, D).half()[:, :, 2].transpose(1, 2)
        # Non-leaf in the trainer; here leaves, so that autograd.grad gives their gradients.
        q, k, v = (t.detach().requires_grad_(case["p"] == 0) for t in (q, k, v))
        return {"case": case, "q": q, "k": k, "v": v, "do": do, "seed": int(seed) & 0xFFFFFFFF}
    if kind == "rope":
        S = case["S"]
        qkv = _randn(g, B, S, 3, H, D).half()
        q, k = (qkv[:, :, i].transpose(1, 2).detach().requires_grad_(True) for i in (0, 1))
        dq, dk = (_randn(g, B, H, S, D).half() for _ in range(2))   # the attention backward's layout
        cos, sin = _tables(S)
        return {"case": case, "q": q, "k": k, "dq": dq, "dk": dk, "cos": cos, "sin": sin}
    Sq, Sk, cap = case["Sq"], case["Sk"], case["Sk"] + case["spare"]
    q = _randn(g, B, Sq, H, D).half().transpose(1, 2)
    k, v = (_randn(g, B, H, cap, D).half()[:, :, :Sk] for _ in range(2))
    return {"case": case, "q": q, "k": k, "v": v}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "train":
        q, k, v, do = state["q"], state["k"], state["v"], state["do"]
        if case["p"] > 0:
            ext = fa.extension()
            o, lse, mask = ext.fa_fwd_mask(q, k, v, case["p"], case["causal"], SCALE, state["seed"])
            dq, dk, dv = ext.fa_bwd(q, k, v, o, lse, do, case["p"], case["causal"], SCALE, state["seed"], 7, mask=mask)
            return o, dq, dk, dv
        o = fa.flash_attn_v100(q, k, v, dropout_p=0.0, causal=case["causal"])
        return (o.detach(), *torch.autograd.grad(o, (q, k, v), do))
    if kind == "rope":
        q, k = state["q"], state["k"]
        qo, ko = fa.rope(q, k, state["cos"], state["sin"])
        gq, gk = torch.autograd.grad((qo, ko), (q, k), (state["dq"], state["dk"]))
        return qo.detach(), ko.detach(), gq, gk
    with torch.no_grad():
        if case["causal"]:
            return fa.flash_attn_kvcache(state["q"], state["k"], state["v"], causal=True)
        return fa.sdpa(state["q"], state["k"], state["v"])


def _visible_pairs(case):
    """Query / key pairs a call has to look at, of one head."""
    if case["kind"] == "train":
        S = case["S"]
        return S * (S + 1) // 2 if case["causal"] else S * S
    Sq, Sk = case["Sq"], case["Sk"]
    return Sq * (Sk - Sq) + Sq * (Sq + 1) // 2 if case["causal"] else Sq * Sk


def work(case):
    BH = case["B"] * case["H"]
    if case["kind"] == "train":
        # read q, k, v, dO; write O, dQ, dK, dV; 2 products forward and 5 backward
        return {"bytes": 8 * BH * case["S"] * D * 2, "flops": 7 * 2 * D * BH * _visible_pairs(case)}
    if case["kind"] == "rope":
        # q, k and their gradients each read and written once; the tables once
        return {"bytes": 8 * BH * case["S"] * D * 2 + 2 * case["S"] * D * 4, "flops": 4 * 3 * BH * case["S"] * D}
    return {"bytes": 2 * BH * (2 * case["Sq"] + 2 * case["Sk"]) * D, "flops": 2 * 2 * D * BH * _visible_pairs(case)}


def tolerance(case):
    # fp16 operands, P and dS rounded to fp16, fp32 sums, fp16 outputs: every output was measured
    # 2e-4 to 4.5e-4 (2-norm, relative) from 64 bits; about four times that.  RoPE: one rounding.
    return {"rel": 1e-3} if case["kind"] == "rope" else {"rel": 2e-3}


def _hash_keep(seed, bh, S, p):
    """Keep mask [S, S] of head bh: lowbias32 of the mixed (seed, row, col, head), its upper 24 bits
    as a fraction compared with p."""
    m = 0xFFFFFFFF
    i = torch.arange(1, S + 1, device=DEV, dtype=torch.int64)
    x = (((seed * 0x9E3779B1) ^ ((bh + 1) * 0x27D4EB2F)) & m) ^ ((i * 0x85EBCA6B) & m)[:, None]
    x = x ^ ((i * 0xC2B2AE35) & m)[None, :]
    x = x ^ (x >> 16)
    x = (x * 0x7FEB352D) & m
    x = x ^ (x >> 15)
    x = ((x & 0xFFFF) * 0x846CA68B + ((((x >> 16) * 0x846CA68B) & 0xFFFF) << 16)) & m   # no 64-bit overflow
    x = x ^ (x >> 16)
    return (x >> 8).double() * 2.0 ** -24 >= float(torch.tensor(p, dtype=torch.float32))


def _rotate(x, cos, sin):
    x1, x2 = x.chunk(2, dim=-1)
    return x * cos + torch.cat((-x2, x1), dim=-1) * sin


def _exact_train(case, st):
    B, H, S, p = case["B"], case["H"], case["S"], case["p"]
    outs = [torch.empty(B, H, S, D, dtype=torch.float64, device=DEV) for _ in range(4)]
    hidden = torch.ones(S, S, dtype=torch.bool, device=DEV).triu(1) if case["causal"] else None
    for b in range(B):
        for h in range(H):
            q, k, v, do = (st[n][b, h].detach().double() for n in ("q", "k", "v", "do"))
            s = (q @ k.T).mul_(SCALE)
            if hidden is not None:
                s.masked_fill_(hidden, -math.inf)
            P = torch.softmax(s, dim=-1)
            if p > 0:
                keep = _hash_keep(st["seed"], b * H + h, S, p).double().div_(1.0 - p)
                Pd, dP = P * keep, (do @ v.T).mul_(keep)
            else:
                Pd, dP = P, do @ v.T
            o = Pd @ v
            dS = P * (dP - (o * do).sum(-1, keepdim=True))
            for out, x in zip(outs, (o, (dS @ k) * SCALE, (dS.T @ q) * SCALE, Pd.T @ do)):
                out[b, h] = x
    return tuple(outs)


def exact(case, seed):
    st = prepare(case, seed)
    if case["kind"] == "train":
        return _exact_train(case, st)
    if case["kind"] == "rope":
        cos, sin = st["cos"].double(), st["sin"].double()
        q, k = (st[n].detach().double() for n in ("q", "k"))

        def back(g):   # the adjoint of _rotate
            gs = g * sin
            g1, g2 = gs.chunk(2, dim=-1)
            return g * cos + torch.cat((g2, -g1), dim=-1)

        return _rotate(q, cos, sin), _rotate(k, cos, sin), back(st["dq"].double()), back(st["dk"].double())
    B, H, Sq, Sk = case["B"], case["H"], case["Sq"], case["Sk"]
    out = torch.empty(B, H, Sq, D, dtype=torch.float64, device=DEV)
    hidden = torch.ones(Sq, Sk, dtype=torch.bool, device=DEV).triu(Sk - Sq + 1) if case["causal"] else None
    for b in range(B):
        for h in range(H):
            s = (st["q"][b, h].double() @ st["k"][b, h].double().T).mul_(SCALE)
            if hidden is not None:
                s.masked_fill_(hidden, -math.inf)
            out[b, h] = torch.softmax(s, dim=-1) @ st["v"][b, h].double()
    return out
