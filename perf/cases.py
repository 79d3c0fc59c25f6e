"""The calls whose speed and results this framework is judged by, one dict per case.

`listed()` holds the named cases, `draw(rng)` one more of the same ranges.  `prepare(case, seed)` makes what a
caller has in hand before the call (inputs on the GPU, drop-in modules with their weights and caches), `run(state)`
is one pass through the public entry points, `work(case)` the bytes and operations that the pass cannot do without,
`tolerance(case)` how far two correct implementations may differ, and `exact(case, seed)` the outputs in 64 bits.

Kinds:
  sinkhorn      drop-in Sinkhorn module on n 4x4 matrices
  mhc           a hyper-connection block (logits, layer input, residual update) on n tokens, the layer itself left out
  indexer       fused indexer operator, fp32 head weights, q and k rotated, causal at the end of the sequence
  layer         drop-in indexer module with its projections: prefill (start_pos 0) or decode (one token), bf16 weights
  fp8           queries quantised, then the indexer over a quantised key cache
  attn          top-k sparse attention, head dim 128, causal index lists
  dropin_attn   drop-in sparse-attention module on a small kv set
  mla           top-k sparse attention on a 512 + 64 latent cache
"""
from __future__ import annotations

import math

import torch

from kernelswift_amd import ops
from kernelswift_amd.mhc import HyperConnection
from kernelswift_amd.optimized import indexer as dropin_indexer
from kernelswift_amd.optimized import sinkhorn as dropin_sinkhorn
from kernelswift_amd.optimized import sparse_attention as dropin_attention
from kernelswift_amd.workloads import freqs_table

DEV = "cuda"


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one layer's residual-mixing matrices of a 1024-token call: the smallest call, all launch and latency
        dict(name="sinkhorn_call", kind="sinkhorn", n=1024, repeat=10),
        # the same for a whole batch of training-sized sequences, an odd count
        dict(name="sinkhorn_batch", kind="sinkhorn", n=1000003, repeat=10),
        # one hyper-connection block around a layer of width 4096 over a 4096-token prefill
        dict(name="mhc_block", kind="mhc", n=4096, dim=4096),
        # a prefill chunk's indexer over a short context
        dict(name="indexer_short", kind="indexer", b=1, s=128, t=4096, heads=64, dim=128, k=512),
        # the same deep in a long context
        dict(name="indexer_long", kind="indexer", b=1, s=64, t=32768, heads=64, dim=128, k=2048),
        # the drop-in indexer layer at its default arguments, whole prompts (compressed keys, ragged length)
        dict(name="layer_prefill", kind="layer", b=2, s=3001, start=0, heads=64, dim=128, rope=64, width=4096,
             lora=1024, k=512),
        # the same layer generating: one token for each of 16 sequences over long compressed caches
        dict(name="layer_decode", kind="layer", b=16, s=1, start=65530, heads=64, dim=128, rope=64, width=4096,
             lora=1024, k=512),
        # a prefill chunk of two sequences whose key cache is kept in FP8
        dict(name="fp8_chunk", kind="fp8", b=2, s=64, t=12000, heads=64, dim=128, k=2048),
        # sparse attention of a prefill chunk, one kv head shared by 16 query heads
        dict(name="attn_chunk", kind="attn", b=1, m=128, heads=16, n=8192, k=2048, start=8064),
        # the drop-in sparse-attention module at its example shape: long batches over tiny kv sets
        dict(name="attn_dropin", kind="dropin_attn", b=8, m=2600, heads=64, n=32, k=16),
        # latent-cache attention, decode: one token for each of 32 long sequences
        dict(name="mla_decode", kind="mla", b=32, m=1, heads=128, n=65536, k=2048, start=65535),
        # latent-cache attention, a prefill chunk in the middle of a sequence
        dict(name="mla_prefill", kind="mla", b=1, m=512, heads=128, n=8192, k=2048, start=7680),
    ]


def _log(rng, lo, hi):
    """An integer spread evenly over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["sinkhorn", "mhc", "indexer", "indexer", "layer", "layer", "fp8", "attn", "dropin_attn", "mla",
                       "mla"])
    if kind == "sinkhorn":
        return dict(kind=kind, n=_log(rng, 1, 4000000), repeat=rng.choice([10, 20]))
    if kind == "mhc":
        return dict(kind=kind, n=_log(rng, 1, 4096), dim=8 * rng.randint(64, 512))
    if kind == "indexer":
        t = _log(rng, 300, 65536)
        s = _log(rng, 1, max(1, min(t, 2 ** 22 // t)))
        heads, dim = rng.choice([(64, 128), (64, 128), (64, 128), (32, 128), (16, 64)])
        return dict(kind=kind, b=rng.choice([1, 1, 2]), s=s, t=t, heads=heads, dim=dim,
                    k=rng.choice([512, 2048, rng.randint(64, 2048)]))
    if kind == "layer":
        heads, dim, rope, width, lora, k = rng.choice([(64, 128, 64, 4096, 1024, 512), (64, 128, 64, 4096, 1024, 2048),
                                                       (16, 64, 32, 1024, 256, 128)])
        if rng.random() < 0.5:
            return dict(kind=kind, b=rng.randint(1, 2), s=_log(rng, 64, 3001), start=0, heads=heads, dim=dim, rope=rope,
                        width=width, lora=lora, k=k)
        return dict(kind=kind, b=rng.randint(1, 16), s=1, start=_log(rng, 1000, 65535), heads=heads, dim=dim,
                    rope=rope, width=width, lora=lora, k=k)
    if kind == "fp8":
        t = _log(rng, 512, 24000)
        return dict(kind=kind, b=rng.randint(1, 2), s=_log(rng, 1, min(128, 1500000 // t)), t=t, heads=64, dim=128,
                    k=rng.choice([512, 2048]))
    if kind == "attn":
        heads = rng.choice([16, 32, 64, 128])
        n = _log(rng, 100, 65536)
        m = _log(rng, 1, min(n, 4096 // heads * 2))
        return dict(kind=kind, b=rng.randint(1, 4), m=m, heads=heads, n=n, k=_log(rng, 64, 2048),
                    start=rng.randint(0, n - m))
    if kind == "dropin_attn":
        n = rng.randint(8, 64)
        return dict(kind=kind, b=rng.randint(1, 8), m=_log(rng, 1, 2600), heads=rng.choice([16, 32, 64]), n=n,
                    k=rng.randint(4, 32))
    heads = rng.choice([32, 64, 128, 128])
    if rng.random() < 0.5:  # decode: one or two tokens a sequence
        n = _log(rng, 500, 65536)
        m = rng.randint(1, 2)
        return dict(kind=kind, b=rng.randint(1, 32), m=m, heads=heads, n=n, k=rng.choice([512, 2048]), start=n - m)
    n = _log(rng, 600, 32768)
    m = _log(rng, 8, 512)
    return dict(kind=kind, b=1, m=m, heads=heads, n=n, k=rng.choice([512, 2048]), start=rng.randint(0, n - m))


# ---------------------------------------------------------------- inputs
def _gen(seed, device=DEV):
    return torch.Generator(device=device).manual_seed(seed)


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)


def _index_lists(g, b, m, n, k, start):
    """Per query, k distinct positions of its causal prefix in random order; -1 past a prefix shorter than k."""
    out = torch.full((b, m, k), -1, dtype=torch.int32, device=DEV)
    kk = min(k, n)
    pos = start + torch.arange(m, device=DEV)
    for i in range(b):
        for j in range(0, m, 64):  # bounds the random matrix at 64 rows of n
            p = pos[j:j + 64, None]
            r = torch.rand(p.shape[0], n, generator=g, device=DEV)
            r = torch.where(torch.arange(n, device=DEV)[None] <= p, r, -1.0)
            top = r.topk(kk, dim=1)
            out[i, j:j + 64, :kk] = torch.where(top.values >= 0, top.indices, -1).to(torch.int32)
    return out


def _inputs(case, seed):
    """The tensors of a case, made from the seed alone."""
    g = _gen(seed)
    c, kind, bf = case, case["kind"], torch.bfloat16
    if kind == "sinkhorn":
        return dict(x=_randn(g, 1, c["n"], 4, 4))
    if kind == "mhc":
        n, d = c["n"], c["dim"]
        return dict(x=_randn(g, n, 4, d, dtype=bf), phi=_randn(g, 4 * d, 24) * (4 * d) ** -0.5,
                    alpha=0.5 + torch.rand(3, generator=g, device=DEV), base=_randn(g, 24) * 0.5)
    if kind in ("indexer", "fp8"):
        return dict(q=_randn(g, c["b"], c["s"], c["heads"], c["dim"], dtype=bf),
                    k=_randn(g, c["b"], c["t"], c["dim"], dtype=bf), w=_randn(g, c["b"], c["s"], c["heads"]) / 8)
    if kind == "layer":
        t = (c["start"] + c["s"]) // 4
        return dict(x=_randn(g, c["b"], c["s"], c["width"], dtype=bf), qr=_randn(g, c["b"], c["s"], c["lora"], dtype=bf),
                    kv=_randn(g, c["b"], t + 64, c["dim"], dtype=bf),
                    wq=_randn(g, c["heads"] * c["dim"], c["lora"], dtype=bf) * c["lora"] ** -0.5,
                    ww=_randn(g, c["heads"], c["width"], dtype=bf) * c["width"] ** -0.5)
    dqk = 576 if kind == "mla" else 128
    q = _randn(g, c["b"], c["m"], c["heads"], dqk, dtype=bf)
    kv = torch.empty(c["b"], c["n"], dqk, dtype=bf, device=DEV)
    for i in range(c["b"]):  # a sequence at a time: the fp32 draw stays small beside a large cache
        kv[i] = torch.randn(c["n"], dqk, generator=g, device=DEV).to(bf)
    sink = _randn(g, c["heads"])
    if kind == "dropin_attn":
        idx = torch.randint(0, c["n"], (c["b"], c["m"], c["k"]), generator=g, device=DEV, dtype=torch.int32)
    else:
        idx = _index_lists(g, c["b"], c["m"], c["n"], c["k"], c["start"])
    return dict(q=q, kv=kv, sink=sink, idx=idx)


def prepare(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    state = dict(case=case, **t)
    if kind == "sinkhorn":
        state["mod"] = dropin_sinkhorn.ModelNew(case["repeat"], 1e-6)
    elif kind == "mhc":
        mod = HyperConnection(case["dim"]).to(DEV).requires_grad_(False)
        mod.phi.copy_(t["phi"])
        mod.alpha.copy_(t["alpha"])
        mod.base.copy_(t["base"])
        state["mod"] = mod
    elif kind == "indexer":
        state["freqs"] = freqs_table(64 if case["dim"] == 128 else 32, case["t"]).to(DEV)
    elif kind == "fp8":
        state["kc"], state["ks"] = ops.fp8_quant(t["k"], block=case["dim"])
        state["ks"] = state["ks"].squeeze(-1)
    elif kind == "layer":
        args = dropin_indexer.ModelArgs(max_batch_size=case["b"], max_seq_len=case["start"] + case["s"],
                                        dim=case["width"], index_n_heads=case["heads"], index_head_dim=case["dim"],
                                        index_topk=case["k"], q_lora_rank=case["lora"], rope_head_dim=case["rope"])
        cis = torch.view_as_complex(freqs_table(case["rope"], case["start"] + case["s"])).to(DEV)
        mod = dropin_indexer.ModelNew(args, cis, t["kv"], 4).to(DEV).requires_grad_(False)
        mod.wq_b.weight.copy_(t["wq"])
        mod.weights_proj.weight.copy_(t["ww"])
        state["mod"] = mod
    elif kind == "dropin_attn":
        mod = dropin_attention.ModelNew(case["heads"], 128).to(DEV).requires_grad_(False)
        mod.attn_sink.copy_(t["sink"])
        state["mod"] = mod
    return state


def run(state):
    c = state["case"]
    kind = c["kind"]
    with torch.no_grad():
        if kind == "sinkhorn":
            return state["mod"](state["x"])
        if kind == "mhc":
            return state["mod"](state["x"], lambda h: h)
        if kind == "indexer":
            return ops.indexer(state["q"], state["k"], state["w"], state["freqs"], c["k"], True, c["t"] - c["s"],
                               rope_dim=2 * state["freqs"].shape[1])
        if kind == "layer":
            return state["mod"](state["x"], state["qr"], c["start"], 0)
        if kind == "fp8":
            qc, qs = ops.fp8_quant(state["q"], block=c["dim"])
            idx = ops.indexer_fp8(qc, qs.squeeze(-1), state["kc"], state["ks"], state["w"], c["k"], True,
                                  c["t"] - c["s"])
            return qc.view(torch.uint8), qs, idx
        if kind == "dropin_attn":
            return state["mod"](state["q"], state["kv"], state["idx"])
        if kind == "attn":
            return ops.sparse_attn(state["q"], state["kv"], state["sink"], state["idx"], 128 ** -0.5)
        return ops.sparse_attn(state["q"], state["kv"], state["sink"], state["idx"], 576 ** -0.5, dv=512)


# ---------------------------------------------------------------- work
def _live_keys(case):
    """Keys scored by causal queries at positions start .. start + s - 1 over t keys (position // ratio)."""
    c = case
    if c["kind"] == "layer":
        t = (c["start"] + c["s"]) // 4
        return t if c["start"] else sum((i + 1) // 4 for i in range(c["s"]))
    return sum(c["t"] - c["s"] + i + 1 for i in range(c["s"]))


def work(case):
    c, kind = case, case["kind"]
    if kind == "sinkhorn":
        return {"bytes": 128 * c["n"], "flops": c["n"] * c["repeat"] * 64}
    if kind == "mhc":
        n, d = c["n"], c["dim"]
        # streams in and out, the layer input out (it is the layer's argument) and the layer output in, phi once
        return {"bytes": n * d * (8 + 8 + 2 + 2) + 4 * d * 24 * 4, "flops": n * d * (4 * 24 * 2 + 8 + 40)}
    if kind in ("indexer", "layer", "fp8"):
        h, d = c["heads"], c["dim"]
        t = (c["start"] + c["s"]) // 4 if kind == "layer" else c["t"]
        rows = c["b"] * c["s"]
        kk = min(c["k"], t)
        live = c["b"] * _live_keys(c)
        flops = 2 * live * h * d
        if kind == "layer":
            by = 2 * (rows * (c["width"] + c["lora"]) + h * d * c["lora"] + h * c["width"] + c["b"] * t * d) + 8 * rows * kk
            return {"bytes": by, "flops": flops + 2 * rows * h * (d * c["lora"] + c["width"])}
        if kind == "fp8":
            return {"bytes": rows * h * (3 * d + 8) + c["b"] * t * (d + 4) + 4 * rows * kk, "flops": flops}
        return {"bytes": rows * h * (2 * d + 4) + c["b"] * t * (2 * d + 4 * (64 if d == 128 else 32)) + 4 * rows * kk,
                "flops": flops}
    dqk, dv = (576, 512) if kind == "mla" else (128, 128)
    rows = c["b"] * c["m"]
    if kind == "dropin_attn":
        picks, kv_rows = rows * c["k"], c["b"] * c["n"]
    else:
        per = [min(c["k"], c["start"] + i + 1) for i in range(c["m"])]
        picks = c["b"] * sum(per)
        kv_rows = c["b"] * min(c["n"], sum(per))
    return {"bytes": 2 * rows * c["heads"] * (dqk + dv) + 2 * kv_rows * dqk + 4 * rows * c["k"],
            "flops": 2 * picks * c["heads"] * (dqk + dv)}


# ---------------------------------------------------------------- correctness
def tolerance(case):
    kind = case["kind"]
    if kind in ("indexer", "layer", "fp8"):
        return "exact"  # indices, and e4m3 codes with their scales: defined to the last bit
    if kind == "sinkhorn":
        return {"rel": 3e-6}  # 32-bit sums: 1e-7 measured
    return {"rel": 8e-3}  # bf16 results: 2.0e-3 to 2.3e-3 measured against 64 bits


def _sinkhorn64(x, repeat, eps):
    x = torch.softmax(x.double(), -1) + eps
    x = x / (x.sum(-2, keepdim=True) + eps)
    for _ in range(repeat - 1):
        x = x / (x.sum(-1, keepdim=True) + eps)
        x = x / (x.sum(-2, keepdim=True) + eps)
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind in ("indexer", "layer", "fp8"):
        return None  # whole numbers
    t = _inputs(case, seed)
    if kind == "sinkhorn":
        return torch.cat([_sinkhorn64(x, case["repeat"], 1e-6) for x in t["x"].split(1 << 18, 1)], 1)
    if kind == "mhc":
        out = []
        phi, al, base = t["phi"].double(), t["alpha"].double(), t["base"].double()
        for x in t["x"].split(512):
            x = x.double()
            xn = x.flatten(1)
            z = (xn * torch.rsqrt(xn.pow(2).mean(-1, keepdim=True) + 1e-6)) @ phi
            pre, post = al[0] * z[:, :4] + base[:4], al[1] * z[:, 4:8] + base[4:8]
            res = (al[2] * z[:, 8:] + base[8:]).view(-1, 4, 4)
            h = (torch.sigmoid(pre)[:, :, None] * x).sum(1)
            out.append(_sinkhorn64(res, 20, 1e-6) @ x + 2 * torch.sigmoid(post)[:, :, None] * h[:, None])
        return torch.cat(out)
    dqk, dv = (576, 512) if kind == "mla" else (128, 128)
    b, m, h = case["b"], case["m"], case["heads"]
    out = torch.empty(b, m, h, dv, dtype=torch.float64, device=DEV)
    step = max(1, min(m, (1 << 18) // case["k"]))
    for i in range(b):
        for j in range(0, m, step):
            idx = t["idx"][i, j:j + step].long()
            rows = t["kv"][i][idx.clamp(min=0)].double()
            q = t["q"][i, j:j + step].double()
            s = torch.matmul(q, rows.transpose(1, 2).contiguous()) * dqk ** -0.5
            s = s.masked_fill((idx < 0)[:, None], float("-inf"))
            s = torch.cat([s, t["sink"].double()[None, :, None].expand(s.shape[0], -1, 1)], -1)
            p = torch.softmax(s, -1)[..., :-1].contiguous()
            out[i, j:j + step] = torch.matmul(p, rows[..., :dv].contiguous())
    return out
