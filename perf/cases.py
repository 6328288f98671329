"""The framework's work at the sizes its users run it: an engine's decode and prefill steps, layer by
layer, and one whole decode step.

Every case is a dict of plain values with a "kind":

  decode    paged decode attention, one new token a sequence; "entry" names the call: "layer"
            (Attention.forward: store + attention), "fused" (qkv_decode_attention: q/k norm, RoPE,
            store and attention) or "paged" (varlen_attention over keys that are already stored)
  shared    paged decode of sequences whose leading blocks are the same (prefix caching)
  dense     Attention.forward of a step of fresh prompts (store + attention over the new keys)
  paged     Attention.forward of a chunked-prefill step over cached prefixes, decode rows first
  rows      the row-wise half of a prefill layer: residual RMSNorm, q/k norm + RoPE + store, SiLU * mul
  linears   the four projections of one decode layer with their fused epilogues, as the decode graph
            replays them
  head      the greedy LM head
  model     one decode step of a whole model, embedding to final norm, as the decode graph replays it;
            of four layers, because each layer passes its bf16 roundings on: the full depth of 28 moves
            its output by 3% for another order of a GEMM's sums, four by 0.6%

Lengths come from the case ("lens" seeds them), tensor values and block placement from the seed.
The geometry is the 0.6B model's (16 query and 8 kv heads of 128, hidden 1024, FFN 3072, vocabulary
151936, blocks of 256) or one tensor-parallel rank's share of its heads.
"""
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "nano-vllm-diy_amd"))

import pagedkv  # noqa: E402
from pagedkv import ops  # noqa: E402
from pagedkv.qwen3 import Qwen3Config, Qwen3Model, Qwen3Weights  # noqa: E402

D, BS, HIDDEN, INTER, VOCAB, EPS = 128, 256, 1024, 3072, 151936, 1e-6
HQ, HKV = 16, 8
SCALE = D ** -0.5
DEV = "cuda"


def listed():
    return [
        # the interactive end: a handful of chats, each step bound by latency and launches
        dict(name="decode_layer_8", kind="decode", entry="layer", seqs=8, lo=256, hi=2048, tp=1, lens=1),
        # the serving run's decode step: the scheduler's cap of live sequences, prompts + outputs to 2048
        dict(name="decode_fused_128", kind="decode", entry="fused", seqs=128, lo=100, hi=2048, tp=1, lens=9),
        # decode at serving scale: long contexts, the K/V stream is everything
        dict(name="decode_long_256", kind="decode", entry="paged", seqs=256, lo=1024, hi=8192, tp=1, lens=2),
        # many requests on one system prompt: 2048 shared keys, private suffixes
        dict(name="decode_shared_64", kind="shared", seqs=64, prefix=2048, lo=256, hi=1024, lens=4),
        # the serving run's first step: as many fresh prompts as the 16384-token budget takes
        dict(name="prefill_dense_16k", kind="dense", prompts=31, lo=100, hi=1024, tp=1, lens=5),
        # a mixed step: every live sequence decodes while a few prompts go through in chunks of 512
        dict(name="prefill_mixed", kind="paged", decodes=128, dlo=512, dhi=4096, chunks=8, qlo=512, qhi=512,
             plo=0, phi=4096, tp=1, lens=3),
        # long documents: large chunks over long cached prefixes, enough work for every CU
        dict(name="prefill_long", kind="paged", decodes=0, dlo=0, dhi=0, chunks=16, qlo=1024, qhi=1024,
             plo=4096, phi=4096, tp=1, lens=6),
        # what a prefill layer does between its GEMMs, a ragged step
        dict(name="prefill_rows_13001", kind="rows", tokens=13001),
        # one sequence decoding, and the full decode batch: weights read for few rows
        dict(name="layer_linears_1", kind="linears", rows=1),
        dict(name="layer_linears_128", kind="linears", rows=128),
        # the head of a nearly full decode batch
        dict(name="head_97", kind="head", rows=97),
        # a decode step of the serving run through a whole (shallow) model
        dict(name="model_decode_128", kind="model", layers=4, seqs=128, lo=100, hi=2048, lens=10),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["decode", "decode", "shared", "dense", "paged", "paged", "rows", "linears", "head", "model"])
    lens = rng.randrange(1 << 20)
    if kind == "decode":
        # from one sequence to 256, contexts from one key to 8192, any tensor-parallel share
        lo, hi = sorted((_log_int(rng, 1, 8192), _log_int(rng, 64, 8192)))
        return dict(kind=kind, entry=rng.choice(["layer", "fused", "paged"]), seqs=_log_int(rng, 1, 256), lo=lo, hi=hi,
                    tp=rng.choice([1, 1, 2, 4, 8]), lens=lens)
    if kind == "shared":
        lo, hi = sorted((rng.randint(1, 1024), rng.randint(1, 1024)))
        return dict(kind=kind, seqs=_log_int(rng, 2, 128), prefix=BS * rng.randint(1, 8), lo=lo, hi=hi, lens=lens)
    if kind == "dense":
        # a step's prompts stay within the token budget
        hi = _log_int(rng, 16, 4096)
        return dict(kind=kind, prompts=_log_int(rng, 1, max(1, min(64, 16384 // hi))), lo=rng.randint(1, hi), hi=hi,
                    tp=rng.choice([1, 1, 2, 4, 8]), lens=lens)
    if kind == "paged":
        qlo, qhi = sorted((rng.randint(2, 1024), rng.randint(2, 1024)))
        plo, phi = sorted((rng.randint(0, 4096), rng.randint(0, 4096)))
        dlo, dhi = sorted((rng.randint(1, 4096), rng.randint(1, 4096)))
        return dict(kind=kind, decodes=rng.choice([0, 0, rng.randint(1, 128)]), dlo=dlo, dhi=dhi,
                    chunks=_log_int(rng, 1, 15), qlo=qlo, qhi=qhi, plo=plo, phi=phi, tp=rng.choice([1, 1, 2, 4, 8]),
                    lens=lens)
    if kind == "rows":
        return dict(kind=kind, tokens=_log_int(rng, 129, 16384))
    if kind in ("linears", "head"):
        return dict(kind=kind, rows=rng.randint(2, 127), lens=lens)
    lo, hi = sorted((rng.randint(1, 2048), rng.randint(1, 2048)))
    return dict(kind=kind, layers=4, seqs=_log_int(rng, 1, 128), lo=lo, hi=hi, lens=lens)


# ---------------------------------------------------------------- shapes of a case ---
def _seqs(case):
    """(query rows, keys) of every sequence, in batch order."""
    r = random.Random(case["lens"])
    if case["kind"] in ("decode", "model"):
        return [(1, r.randint(case["lo"], case["hi"])) for _ in range(case["seqs"])]
    if case["kind"] == "shared":
        return [(1, case["prefix"] + r.randint(case["lo"], case["hi"])) for _ in range(case["seqs"])]
    if case["kind"] == "dense":
        n = [r.randint(case["lo"], case["hi"]) for _ in range(case["prompts"])]
        return [(x, x) for x in n]
    out = [(1, r.randint(case["dlo"], case["dhi"])) for _ in range(case["decodes"])]
    for _ in range(case["chunks"]):
        q = r.randint(case["qlo"], case["qhi"])
        out.append((q, q + r.randint(case["plo"], case["phi"])))
    return out


def _heads(case):
    tp = case.get("tp", 1)
    return HQ // tp, HKV // tp


def work(case):
    """Bytes: inputs read once, outputs written once. Flops: multiplies and adds, causal pairs only."""
    kind = case["kind"]
    if kind == "rows":
        n = case["tokens"]
        qkv = (HQ + 2 * HKV) * D
        return {"bytes": 2 * n * (4 * HIDDEN + 2 * qkv + 3 * INTER), "flops": 10 * n * (HIDDEN + qkv + INTER)}
    layer = (HQ + 2 * HKV) * D * HIDDEN + HQ * D * HIDDEN + 3 * INTER * HIDDEN
    if kind == "linears":
        m = case["rows"]
        return {"bytes": 2 * layer + 2 * m * (HIDDEN + 2 * HQ * D + 2 * HKV * D + 5 * HIDDEN + INTER + HQ * D),
                "flops": 2 * m * layer}
    if kind == "head":
        return {"bytes": 2 * VOCAB * HIDDEN + case["rows"] * (2 * HIDDEN + 4), "flops": 2 * case["rows"] * VOCAB * HIDDEN}
    seqs = _seqs(case)
    hq, hkv = _heads(case)
    new, keys = sum(q for q, _ in seqs), sum(k for _, k in seqs)
    if kind == "shared":
        keys = case["prefix"] + sum(k - case["prefix"] for _, k in seqs)
    pairs = sum(q * (k - q) + q * (q + 1) // 2 for q, k in seqs)
    row = 2 * hkv * D * 2
    flops = 4 * hq * D * pairs
    stored = new if kind in ("dense", "paged") or case.get("entry") in ("layer", "fused") else 0
    nbytes = keys * row + stored * row + 2 * new * hq * D * 2
    if kind == "model":
        return {"bytes": case["layers"] * (nbytes + new * row + 2 * layer) + 4 * new * HIDDEN,
                "flops": case["layers"] * (flops + 2 * new * layer)}
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """The largest differences that another order of the same bf16 paths' sums makes, times about four.
    Measured: attention with other key splits 0.0035 (max 0.017), the four layers with other GEMMs 0.0058
    (max 0.041)."""
    kind = case["kind"]
    if kind == "head":
        return {"differ": 0.01}        # ties of bf16 logits
    if kind == "rows":
        return {"rel": 2e-3, "max": 0.02}   # single ulps of bf16
    if kind == "model":
        return {"rel": 0.024, "max": 0.17}
    return {"rel": 0.014, "max": 0.07}


# ------------------------------------------------------------------------- inputs ---
def _randn(g, *shape, std=1.0):
    t = torch.randn(*shape, generator=g, device=DEV, dtype=torch.bfloat16)
    return t if std == 1.0 else t.mul_(std)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


def _tables(case, seqs, seed):
    """Block ids per sequence from a shuffled pool (the shared prefix's first), and the pool's size."""
    shared = case["prefix"] // BS if case["kind"] == "shared" else 0
    need = [-(-k // BS) - shared for _, k in seqs]
    total = shared + sum(need)
    pool = list(range(total))
    random.Random(seed).shuffle(pool)
    out, at = [], shared
    for n in need:
        out.append(pool[:shared] + pool[at:at + n])
        at += n
    return out, total


def _paged_inputs(case, seed):
    seqs = _seqs(case)
    tables, total = _tables(case, seqs, seed)
    w = max(len(t) for t in tables)
    cu_q, cu_k, slots, pos = [0], [0], [], []
    for (q, k), t in zip(seqs, tables):
        cu_q.append(cu_q[-1] + q)
        cu_k.append(cu_k[-1] + k)
        slots += [t[p // BS] * BS + p % BS for p in range(k - q, k)]
        pos += range(k - q, k)
    return dict(seqs=seqs, tables=tables, total=total, cu_q=_i32(cu_q), cu_k=_i32(cu_k), slots=_i32(slots),
                pos=torch.tensor(pos, dtype=torch.int64, device=DEV),
                bt=_i32([t + [-1] * (w - len(t)) for t in tables]),
                max_q=max(q for q, _ in seqs), max_k=max(k for _, k in seqs))


def _attention_inputs(case, seed):
    p = _paged_inputs(case, seed)
    hq, hkv = _heads(case)
    g, n = _gen(seed), len(p["pos"])
    p["kc"], p["vc"] = (_randn(g, p["total"], BS, hkv, D) for _ in range(2))
    p["qkv"] = _randn(g, n, (hq + 2 * hkv) * D)
    # q and k leave the producer contiguous, v stays a view of the fused projection's rows
    p["q"] = p["qkv"][:, :hq * D].reshape(n, hq, D).clone()
    p["k"] = p["qkv"][:, hq * D:(hq + hkv) * D].reshape(n, hkv, D).clone()
    p["v"] = p["qkv"][:, (hq + hkv) * D:].view(n, hkv, D)
    p["wq"], p["wk"] = (1 + 0.1 * torch.randn(2, D, generator=g, device=DEV)).to(torch.bfloat16)
    return p


def _rows_inputs(case, seed):
    n, g = case["tokens"], _gen(seed)
    perm = torch.randperm(-(-n // BS), generator=torch.Generator().manual_seed(seed))
    i = torch.arange(n)
    slots = (perm[i // BS] * BS + i % BS).to(torch.int32).to(DEV)
    return dict(h=_randn(g, n, HIDDEN), res=_randn(g, n, HIDDEN), qkv=_randn(g, n, (HQ + 2 * HKV) * D),
                gu=_randn(g, n, 2 * INTER), slots=slots, pos=(i % 1024).to(DEV), nb=len(perm),
                wn=(1 + 0.1 * torch.randn(HIDDEN, generator=g, device=DEV)).to(torch.bfloat16),
                wq=(1 + 0.1 * torch.randn(D, generator=g, device=DEV)).to(torch.bfloat16),
                wk=(1 + 0.1 * torch.randn(D, generator=g, device=DEV)).to(torch.bfloat16))


def _linears_inputs(case, seed):
    m, g = case["rows"], _gen(seed)
    return dict(x=_randn(g, m, HIDDEN), attn=_randn(g, m, HQ * D, std=0.3), res=_randn(g, m, HIDDEN),
                wqkv=_randn(g, (HQ + 2 * HKV) * D, HIDDEN, std=0.02), wo=_randn(g, HIDDEN, HQ * D, std=0.02),
                wgu=_randn(g, 2 * INTER, HIDDEN, std=0.02), wd=_randn(g, HIDDEN, INTER, std=0.02),
                n1=(1 + 0.1 * torch.randn(HIDDEN, generator=g, device=DEV)).to(torch.bfloat16),
                n2=(1 + 0.1 * torch.randn(HIDDEN, generator=g, device=DEV)).to(torch.bfloat16))


def _head_inputs(case, seed):
    g = _gen(seed)
    return dict(x=_randn(g, case["rows"], HIDDEN), w=_randn(g, VOCAB, HIDDEN, std=0.02))


def _model_inputs(case, seed):
    p = _paged_inputs(case, seed)
    g = _gen(seed)
    p["kc"], p["vc"] = (_randn(g, case["layers"], p["total"], BS, HKV, D) for _ in range(2))
    p["ids"] = torch.randint(0, VOCAB, (case["seqs"],), generator=g, device=DEV)
    p["cfg"] = Qwen3Config(num_hidden_layers=case["layers"])
    p["w"] = Qwen3Weights(p["cfg"], torch.device(DEV), seed)
    return p


# ---------------------------------------------------------------- prepare and run ---
def _graph(fn):
    """fn once eagerly, then captured, as the runner makes its decode graphs; returns (replay, outputs)."""
    fn()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = fn()
    return g, out


def _context(case, p, tables=True):
    kind = case["kind"]
    return pagedkv.Context(is_prefill=p["max_q"] > 1, cu_seqlens_q=p["cu_q"], cu_seqlens_k=p["cu_k"],
                           max_seqlen_q=p["max_q"], max_seqlen_k=p["max_k"], slot_mapping=p["slots"],
                           block_tables=p["bt"] if tables else None,
                           cached_prefix_keys=case["prefix"] if kind == "shared" else 0)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "rows":
        p = _rows_inputs(case, seed)
        p["kc"], p["vc"] = (torch.zeros(p["nb"], BS, HKV, D, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        p["table"] = ops.rope_cos_sin(1024, D, device=DEV)
    elif kind == "linears":
        p = _linears_inputs(case, seed)

        def layer():
            qkv = pagedkv.linear(p["x"], p["wqkv"])
            x, r = pagedkv.linear_add_rmsnorm(p["attn"], p["wo"], p["res"], p["n1"], EPS)
            act = pagedkv.linear_silu_mul(x, p["wgu"])
            y, r2 = pagedkv.linear_add_rmsnorm(act, p["wd"], r, p["n2"], EPS)
            return dict(qkv=qkv, x=x, r=r, act=act, y=y, r2=r2)

        p["graph"], p["out"] = _graph(layer)
    elif kind == "head":
        p = _head_inputs(case, seed)
    elif kind == "model":
        p = _model_inputs(case, seed)
        model = Qwen3Model(p["cfg"], p["w"], p["kc"], p["vc"], 4096)
        ctx = _context(case, p)
        p["model"] = model
        p["graph"], p["out"] = _graph(lambda: model.forward(p["ids"], p["pos"], ctx))
    else:
        p = _attention_inputs(case, seed)
        hq, hkv = _heads(case)
        if case.get("entry") == "fused":
            p["table"] = ops.rope_cos_sin(8192, D, device=DEV)
        elif case.get("entry") != "paged":
            p["layer"] = pagedkv.Attention(D, hq, hkv, SCALE)
            p["layer"].k_cache, p["layer"].v_cache = p["kc"], p["vc"]
            p["ctx"] = _context(case, p, tables=kind != "dense")
    p["case"] = case
    return p


def run(p):
    case = p["case"]
    kind = case["kind"]
    if kind in ("linears", "model"):
        p["graph"].replay()
        return p["out"]
    if kind == "head":
        return pagedkv.lm_head_greedy(p["x"], p["w"])
    if kind == "rows":
        x, res = pagedkv.add_rmsnorm(p["h"], p["wn"], EPS, residual=p["res"])
        q, _ = pagedkv.qk_norm_rope_store(p["qkv"], p["pos"], p["table"], HQ, HKV, D, p["wq"], p["wk"], EPS,
                                          p["kc"], p["vc"], p["slots"])
        return dict(x=x, res=res, q=q, kc=p["kc"], vc=p["vc"], act=pagedkv.silu_and_mul(p["gu"]))
    if kind == "decode" and case["entry"] == "paged":
        return pagedkv.varlen_attention(p["q"], p["kc"], p["vc"], p["cu_q"], p["cu_k"], p["max_q"], p["max_k"], SCALE,
                                        True, p["bt"], cached_prefix_keys=0)
    if kind == "decode" and case["entry"] == "fused":
        hq, hkv = _heads(case)
        out = pagedkv.qkv_decode_attention(p["qkv"], p["pos"], p["table"], hq, hkv, D, p["wq"], p["wk"], EPS, p["kc"],
                                           p["vc"], p["slots"], p["cu_q"], p["cu_k"], p["max_k"], SCALE, p["bt"],
                                           cached_prefix_keys=0)
    else:
        out = p["layer"](p["q"], p["k"], p["v"], p["ctx"])
    return dict(out=out, kc=p["kc"], vc=p["vc"])


# ------------------------------------------------------------------ in 64 bits ------
def _norm64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, pos, most):
    """x (N, H, D) in 64 bits, rotated by the float32 table's rows."""
    inv = 1.0 / (1000000.0 ** (torch.arange(0, D, 2, device=DEV).float() / D))
    ang = torch.outer(torch.arange(most, dtype=torch.float, device=DEV), inv)[pos]
    c, s = ang.cos().double().unsqueeze(1), ang.sin().double().unsqueeze(1)
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _attend64(q, k, v):
    """One sequence: q (Lq, Hq, D), k and v (Lk, Hkv, D) in 64 bits, bottom-right causal."""
    lq, hq, _ = q.shape
    lk, hkv, _ = k.shape
    qs = q.reshape(lq, hkv, hq // hkv, D).permute(1, 2, 0, 3).reshape(hkv, -1, D)
    s = torch.matmul(qs, k.permute(1, 2, 0).contiguous()).view(hkv, hq // hkv, lq, lk) * SCALE
    if lq > 1:
        at = torch.arange(lk, device=DEV) - (lk - lq)
        s.masked_fill_(at[None, :] > torch.arange(lq, device=DEV)[:, None], float("-inf"))
    o = torch.matmul(torch.softmax(s, -1).view(hkv, -1, lk), v.permute(1, 0, 2).contiguous())
    return o.view(hkv, hq // hkv, lq, D).permute(2, 0, 1, 3).reshape(lq, hq, D)


def _batch64(p, q, kc, vc):
    """Every sequence's attention over its cached rows; caches hold the new rows already."""
    out, at = [], 0
    for (lq, lk), t in zip(p["seqs"], p["tables"]):
        ids = torch.tensor(t, device=DEV)
        k, v = (c[ids].reshape(-1, *c.shape[2:])[:lk].double() for c in (kc, vc))
        out.append(_attend64(q[at:at + lq], k, v))
        at += lq
    return torch.cat(out)


def _put(cache, slots, rows):
    cache.view(-1, *cache.shape[2:])[slots.long()] = rows.to(cache.dtype)


def exact(case, seed):
    kind = case["kind"]
    if kind == "rows":
        p = _rows_inputs(case, seed)
        s = p["h"].double() + p["res"].double()
        q, k, v = p["qkv"].double().split([HQ * D, HKV * D, HKV * D], -1)
        q = _rope64(_norm64(q.view(-1, HQ, D), p["wq"]), p["pos"], 1024)
        k = _rope64(_norm64(k.view(-1, HKV, D), p["wk"]), p["pos"], 1024)
        kc, vc = (torch.zeros(p["nb"], BS, HKV, D, dtype=torch.float64, device=DEV) for _ in range(2))
        _put(kc, p["slots"], k)
        _put(vc, p["slots"], v.view(-1, HKV, D))
        a, b = p["gu"].double().chunk(2, -1)
        return dict(x=_norm64(s, p["wn"]), res=s, q=q, kc=kc, vc=vc, act=a * torch.sigmoid(a) * b)
    if kind == "linears":
        p = {k: v.double() for k, v in _linears_inputs(case, seed).items()}
        r = p["res"] + p["attn"] @ p["wo"].t()
        x = _norm64(r, p["n1"])
        a, b = (x @ p["wgu"].t()).chunk(2, -1)
        act = a * torch.sigmoid(a) * b
        r2 = r + act @ p["wd"].t()
        return dict(qkv=p["x"] @ p["wqkv"].t(), x=x, r=r, act=act, y=_norm64(r2, p["n2"]), r2=r2)
    if kind == "head":
        p = _head_inputs(case, seed)
        logits = p["x"].double() @ p["w"].double().t()
        return logits.to(torch.bfloat16).float().cpu().numpy().argmax(-1).astype("int32")   # the first of equals
    if kind == "model":
        p = _model_inputs(case, seed)
        n, w = case["seqs"], p["w"]
        r, h = 0.0, w.embed[p["ids"]].double()
        for li, L in enumerate(w.layers):
            r = r + h
            qkv = _norm64(r, L["input_norm"]) @ L["qkv"].double().t()
            q, k, v = qkv.split([HQ * D, HKV * D, HKV * D], -1)
            q = _rope64(_norm64(q.view(n, HQ, D), L["q_norm"]), p["pos"], 4096)
            k = _rope64(_norm64(k.view(n, HKV, D), L["k_norm"]), p["pos"], 4096)
            _put(p["kc"][li], p["slots"], k)
            _put(p["vc"][li], p["slots"], v.view(n, HKV, D))
            r = r + _batch64(p, q, p["kc"][li], p["vc"][li]).view(n, -1) @ L["o"].double().t()
            a, b = (_norm64(r, L["post_norm"]) @ L["gate_up"].double().t()).chunk(2, -1)
            h = (a * torch.sigmoid(a) * b) @ L["down"].double().t()
        return _norm64(r + h, w.final_norm)
    p = _attention_inputs(case, seed)
    hq, hkv = _heads(case)
    q, k, v = p["q"].double(), p["k"].double(), p["v"].double()
    if case.get("entry") == "fused":
        q, k = (_rope64(_norm64(t, p[w]), p["pos"], 8192) for t, w in ((q, "wq"), (k, "wk")))
    if case.get("entry") == "paged":
        return _batch64(p, q, p["kc"], p["vc"])
    _put(p["kc"], p["slots"], k)
    _put(p["vc"], p["slots"], v)
    if kind == "dense":
        at, out = 0, []
        for lq, _ in p["seqs"]:
            out.append(_attend64(q[at:at + lq], k[at:at + lq], v[at:at + lq]))
            at += lq
        o = torch.cat(out)
    else:
        o = _batch64(p, q, p["kc"], p["vc"])
    # the stored keys of the fused step are computed numbers, the rest of the caches copies
    return dict(out=o, kc=p["kc"], vc=p["vc"])
