"""The work this framework is measured on: speculative-decoding steps of the two
shapes it is built for -- the 0.5B shape (hidden 896, 14 query / 2 KV heads of
64, 24 layers, vocabulary 151,936) and the 8B shape (hidden 4096, 32 / 8 heads
of 128, FP8 linears, vocabulary 128,256) -- from a single request's decode
step to a batch of long contexts and the prefill of its prompts.

A case is one pass through the public entry points (``kernels.*``,
``BatchPrefillWithPagedKVCacheWrapper``, ``CausalLM.forward_packed``).  The
calls of a decode / verify step that the engine replays as a HIP graph are
captured once in :func:`prepare` and replayed here too (``graph``), over
``layers`` layers with weights or K / V of their own, as in a model; prefill,
acceptance and sampling are eager calls.  Sequence lengths follow from the
case alone (``lens``), every value from the seed.
"""

from __future__ import annotations

import math
import random

import torch

from nanosglang_amd import kernels
from nanosglang_amd.kernels import BatchPrefillWithPagedKVCacheWrapper
from nanosglang_amd.model.causal_lm import CausalLM, ModelConfig

DEV = "cuda"
BF16 = torch.bfloat16
SMALL = {"hq": 14, "hkv": 2, "d": 64}     # the 0.5B shape's heads
LARGE = {"hq": 32, "hkv": 8, "d": 128}    # the 8B shape's heads
SMALL_MLP = {"hidden": 896, "inter": 4864}
LARGE_MLP = {"hidden": 4096, "inter": 14336}


def listed():
    return [
        # one request's decode step (the smallest call: launches and latency)
        {"name": "attn_decode_1", "kind": "attn", **SMALL, "batch": 1, "q": 1, "lo": 300, "hi": 400,
         "lens": 1, "page": 16, "layers": 24, "graph": True},
        # the verify step of 32 requests: 4 drafts and the bonus token
        {"name": "attn_verify_32", "kind": "attn", **SMALL, "batch": 32, "q": 5, "lo": 100,
         "hi": 640, "lens": 2, "page": 16, "layers": 24, "graph": True},
        # verify over long contexts, 8B shape (k = 8): the KV stream
        {"name": "attn_verify_long", "kind": "attn", **LARGE, "batch": 64, "q": 9, "lo": 2048,
         "hi": 8192, "lens": 3, "page": 16, "layers": 1, "graph": False},
        # prefill of a batch of prompts, all positions query positions
        {"name": "attn_prefill_32", "kind": "attn", **SMALL, "batch": 32, "q": 0, "lo": 100,
         "hi": 512, "lens": 4, "page": 16, "layers": 1, "graph": False},
        # prefill of long prompts, 8B shape
        {"name": "attn_prefill_long", "kind": "attn", **LARGE, "batch": 2, "q": 0, "lo": 2048,
         "hi": 8192, "lens": 5, "page": 16, "layers": 1, "graph": False},
        # the MLP of a verify forward (32 requests x 5 rows), norms folded in
        {"name": "mlp_verify_160", "kind": "mlp", **SMALL_MLP, "rows": 160, "fp8": False,
         "layers": 24, "graph": True},
        # the MLP of the 8B shape's draft forwards, FP8 weights, 64 requests
        {"name": "mlp_fp8_64", "kind": "mlp", **LARGE_MLP, "rows": 64, "fp8": True, "layers": 4,
         "graph": True},
        # greedy token of every verify row: lm_head with the final norm folded
        {"name": "lm_head_160", "kind": "lm_head", "hidden": 896, "vocab": 151936, "rows": 160,
         "tokens": True},
        # stochastic acceptance of 64 requests, 4 drafts
        {"name": "accept_stochastic", "kind": "accept", "batch": 64, "k": 4, "vocab": 151936,
         "temp": 0.8, "fp32": False},
        # greedy acceptance from logits, 8 drafts
        {"name": "accept_greedy", "kind": "accept", "batch": 64, "k": 8, "vocab": 128256,
         "temp": 0.0, "fp32": False},
        # a filtered draw for 32 requests (a draft token or the bonus)
        {"name": "sample_filtered", "kind": "sample", "rows": 32, "vocab": 151936, "temp": 0.8,
         "top_k": 50, "top_p": 0.9, "fp32": False},
        # a whole verify forward, 32 requests x 5 rows, all logits: 8 layers, so
        # that bf16 roundings of the first do not drown the last one's
        {"name": "model_verify", "kind": "model", "model_layers": 8, "batch": 32, "q": 5,
         "lo": 100, "hi": 640, "lens": 6, "page": 16, "graph": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "mlp", "lm_head", "accept", "sample",
                       "model"])
    if kind == "decode":
        heads = rng.choice([SMALL, LARGE])
        batch, lo = _log_int(rng, 1, 64), _log_int(rng, 16, 2048)
        hi = min(8192, int(lo * rng.uniform(1, 5)))
        # as many layers as the largest listed case's bytes allow
        layers = min(24, 300_000_000 // (batch * hi * heads["hkv"] * heads["d"]))
        return {"kind": "attn", **heads, "batch": batch, "q": rng.choice([1, 2, 3, 5, 9]),
                "lo": lo, "hi": hi, "lens": rng.randrange(1 << 20),
                "page": rng.choice([16, 16, 32]), "layers": max(1, layers), "graph": layers > 3}
    if kind == "prefill":
        heads = rng.choice([SMALL, LARGE])
        hi = _log_int(rng, 32, 8192)
        batch = _log_int(rng, 1, max(1, min(64, 16384 // hi)))
        return {"kind": "attn", **heads, "batch": batch, "q": 0, "lo": max(1, hi // 4), "hi": hi,
                "lens": rng.randrange(1 << 20), "page": rng.choice([16, 16, 32]), "layers": 1,
                "graph": False}
    if kind == "mlp":
        fp8 = rng.random() < 0.5
        return {"kind": "mlp", **(LARGE_MLP if fp8 else SMALL_MLP),
                "rows": _log_int(rng, 1, 160), "fp8": fp8, "layers": 4 if fp8 else 24,
                "graph": True}
    if kind == "lm_head":
        return {"kind": "lm_head", "hidden": 896, "vocab": 151936, "rows": _log_int(rng, 1, 160),
                "tokens": rng.random() < 0.7}
    if kind == "accept":
        return {"kind": "accept", "batch": _log_int(rng, 1, 64), "k": rng.randint(1, 8),
                "vocab": rng.choice([151936, 128256, 32000, rng.randint(1000, 140000)]),
                "temp": rng.choice([0.0, 0.7, 0.8, 1.0]), "fp32": rng.random() < 0.25}
    if kind == "sample":
        top_k, top_p = rng.choice([(0, 0.9), (50, 1.0), (50, 0.9), (0, 1.0),
                                   (rng.randint(1, 200), rng.uniform(0.5, 0.99))])
        return {"kind": "sample", "rows": _log_int(rng, 1, 64),
                "vocab": rng.choice([151936, 128256, 32000, rng.randint(1000, 140000)]),
                "temp": rng.choice([0.7, 0.8, 1.0]), "top_k": top_k, "top_p": top_p,
                "fp32": rng.random() < 0.25}
    lo = _log_int(rng, 32, 256)
    return {"kind": "model", "model_layers": 8, "batch": _log_int(rng, 1, 32),
            "q": rng.choice([1, 3, 5]), "lo": lo, "hi": lo * 3, "lens": rng.randrange(1 << 20),
            "page": 16, "graph": True}


# ---------------------------------------------------------------- sizes

def _lens(case):
    """(query lengths, KV lengths) of a case's requests."""
    r = random.Random(case["lens"])
    kv = [r.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]
    if case["q"] == 0:                       # prefill: every position is a query
        return list(kv), kv
    kv = [max(n, case["q"]) for n in kv]
    return [case["q"]] * case["batch"], kv


def _pairs(ql, kl):
    """Visible (query, key) pairs under the bottom-right causal rule."""
    return sum(q * k - q * (q - 1) // 2 for q, k in zip(ql, kl))


def _attn_work(case):
    ql, kl = _lens(case)
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    return (sum(kl) * hkv * d * 4 + 2 * sum(ql) * hq * d * 2, 4 * _pairs(ql, kl) * hq * d)


def work(case):
    kind = case["kind"]
    if kind == "attn":
        b, f = _attn_work(case)
        return {"bytes": b * case["layers"], "flops": f * case["layers"]}
    if kind == "mlp":
        H, I, M = case["hidden"], case["inter"], case["rows"]
        w = 3 * H * I * (1 if case["fp8"] else 2)
        return {"bytes": (w + 3 * M * H * 2) * case["layers"],
                "flops": 6 * M * H * I * case["layers"]}
    if kind == "lm_head":
        H, V, M = case["hidden"], case["vocab"], case["rows"]
        out = M * 8 if case["tokens"] else M * V * 2
        return {"bytes": V * H * 2 + M * H * 2 + out, "flops": 2 * M * V * H}
    if kind == "accept":
        rows = case["batch"] * (case["k"] + 1 + (case["k"] if case["temp"] else 0))
        n = rows * case["vocab"]
        return {"bytes": n * (4 if case["fp32"] else 2), "flops": 3 * n}
    if kind == "sample":
        n = case["rows"] * case["vocab"]
        return {"bytes": n * (4 if case["fp32"] else 2), "flops": 3 * n}
    c = ModelConfig(num_hidden_layers=case["model_layers"])
    ql, kl = _lens(case)
    M, H, I, D = sum(ql), c.hidden_size, c.intermediate_size, c.head_dim
    nq = (c.num_attention_heads + 2 * c.num_key_value_heads) * D
    w = nq * H + H * H + 3 * H * I
    ab, af = _attn_work({**case, **SMALL})
    return {"bytes": c.num_hidden_layers * (2 * w + ab) + 2 * c.vocab_size * (H + M),
            "flops": c.num_hidden_layers * (2 * M * w + af) + 2 * M * H * c.vocab_size}


def tolerance(case):
    kind = case["kind"]
    if kind == "attn":
        # bf16 output and bf16 probabilities: measured 2e-3 - 3e-3 from 64 bits
        return {"rel": 8e-3, "max": 0.08}
    if kind == "mlp":
        # bf16 hidden and output, fp32 sums: measured 2e-3 (residual added) and
        # 4.7e-3 (the MLP's own output) from 64 bits
        return {"rel": 0.015, "max": 0.1} if case["fp8"] else {"rel": 8e-3, "max": 0.08}
    if kind == "lm_head":
        # logits: one bf16 rounding; tokens: two logits of a row may round to a tie
        return {"rel": 8e-3, "max": 0.05, "differ": 0.01}
    if kind == "accept":
        # greedy: whole numbers from whole comparisons; stochastic: a draw
        # within fp32 rounding of a boundary may fall on its other side
        return {"rel": 0.0, "differ": 0.005} if case["temp"] else "exact"
    if kind == "sample":
        return "exact"                       # integer masses by definition
    # bf16 residual stream through the layers
    return {"rel": 0.03, "max": 0.3}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, *shape, std=1.0, dtype=BF16):
    out = torch.empty(*shape, dtype=dtype, device=DEV)
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 27):      # pieces: fp32 draws need little room
        n = min(1 << 27, flat.numel() - i)
        flat[i:i + n] = torch.randn(n, generator=g, device=DEV) * std
    return out


def _tables(case, seed):
    """CSR page table of the case's requests on scattered pages of a pool."""
    ql, kl = _lens(case)
    P = case["page"]
    need = [-(-n // P) for n in kl]
    total = sum(need)
    pages = total + max(8, total // 8)
    perm = torch.randperm(pages, generator=torch.Generator().manual_seed(seed))[:total]
    qo = [0]
    kv = [0]
    for q, n in zip(ql, need):
        qo.append(qo[-1] + q)
        kv.append(kv[-1] + n)
    i32 = torch.int32
    return {"qo": torch.tensor(qo, dtype=i32), "kvp": torch.tensor(kv, dtype=i32),
            "idx": perm.to(i32), "last": torch.tensor([n - (m - 1) * P for n, m in zip(kl, need)],
                                                      dtype=i32), "pages": pages}


def _planned(case, t, hq, hkv, d):
    w = BatchPrefillWithPagedKVCacheWrapper(
        torch.empty(256 << 20, dtype=torch.uint8, device=DEV), "NHD")
    w.plan(t["qo"], t["kvp"], t["idx"], t["last"], hq, hkv, d, case["page"], causal=True)
    return w


def _attn_inputs(case, seed):
    t = _tables(case, seed)
    g = _gen(seed)
    hq, hkv, d, L = case["hq"], case["hkv"], case["d"], case["layers"]
    q = _normal(g, L, int(t["qo"][-1]), hq, d)
    k = _normal(g, L, t["pages"], case["page"], hkv, d, std=0.5)
    v = _normal(g, L, t["pages"], case["page"], hkv, d, std=0.5)
    return t, q, k, v


def _mlp_inputs(case, seed):
    g = _gen(seed)
    H, I, L = case["hidden"], case["inter"], case["layers"]
    x = _normal(g, case["rows"], H)
    gate_up = [_normal(g, 2 * I, H, std=0.02) for _ in range(L)]
    down = [_normal(g, H, I, std=0.02) for _ in range(L)]
    return x, gate_up, down


def _lm_inputs(case, seed):
    g = _gen(seed)
    return _normal(g, case["rows"], case["hidden"]), _normal(g, case["vocab"], case["hidden"],
                                                             std=0.02)


def _fp8(w, parts):
    from nanosglang_amd.model.quantization import fp8_quantize_rows
    return fp8_quantize_rows(w, parts)


def _capture(state, call):
    """The step graph of a decode / verify call, as the engine captures it."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        call()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        state["out"] = call()
    state["replay"] = graph.replay
    return state


def _attn_call(s):
    for i in range(s["q"].shape[0]):
        s["wrapper"].run(s["q"][i], (s["k"][i], s["v"][i]), out=s["o"][i])
    return s["o"]


def _mlp_call(s):
    """Norm + SwiGLU MLP + residual of each layer on the same rows: the folded
    norm's form with bf16 weights, the norm kernel with FP8 ones."""
    x = s["x"]
    for i, (gu, dn) in enumerate(zip(s["gate_up"], s["down"])):
        if s["fp8"]:
            h = kernels.rmsnorm(x, s["ones"], 1e-6)
            g = kernels.linear(h, gu[0], swiglu=True, w_scale=gu[1])
            kernels.linear(g, dn[0], w_scale=dn[1], out=s["o"][i])
        else:
            g = kernels.linear(x, gu, swiglu=True, sumsq_in=s["ss"], norm_eps=1e-6)
            kernels.linear(g, dn, residual=x, sumsq_out=s["sso"][i], out=s["o"][i])
    return s["o"]


def _model_call(s):
    return s["model"].forward_packed(s["ids"], s["pos"], s["kv"], s["wrapper"], s["slots"])


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": case}
    if kind == "attn":
        t, s["q"], s["k"], s["v"] = _attn_inputs(case, seed)
        s["wrapper"] = _planned(case, t, case["hq"], case["hkv"], case["d"])
        s["o"] = torch.empty_like(s["q"])
        s["call"] = _attn_call
    elif kind == "mlp":
        s["x"], gate_up, down = _mlp_inputs(case, seed)
        H, I, L, M = case["hidden"], case["inter"], case["layers"], case["rows"]
        s["fp8"] = case["fp8"]
        if case["fp8"]:
            gate_up = [_fp8(w, [I, I]) for w in gate_up]
            down = [_fp8(w, [H]) for w in down]
            s["ones"] = torch.ones(H, dtype=BF16, device=DEV)
        else:
            s["ss"] = kernels.row_sumsq(s["x"])
            s["sso"] = torch.empty(L, H // 16, M, dtype=torch.float32, device=DEV)
        s["gate_up"], s["down"] = gate_up, down
        s["o"] = torch.empty(L, M, H, dtype=BF16, device=DEV)
        s["call"] = _mlp_call
    elif kind == "lm_head":
        s["x"], s["w"] = _lm_inputs(case, seed)
        s["ss"] = kernels.row_sumsq(s["x"])
    elif kind == "accept":
        g = _gen(seed)
        B, k, V = case["batch"], case["k"], case["vocab"]
        dt = torch.float32 if case["fp32"] else BF16
        draft = torch.randn(B, k, V, generator=g, device=DEV) * 2.0
        target = torch.empty(B, k + 1, V, dtype=dt, device=DEV)
        target[:, :k] = draft + 0.5 * torch.randn(B, k, V, generator=g, device=DEV)
        target[:, k] = 2.06 * torch.randn(B, V, generator=g, device=DEV)
        s["draft"], s["target"] = draft.to(dt), target
        if case["temp"]:
            p = torch.softmax(s["draft"].float() / case["temp"], -1)
            tok = torch.multinomial(p.view(B * k, V), 1, generator=g).view(B, k)
            s["u"] = torch.rand(B, k + 1, generator=g, device=DEV)
        else:
            # a draft that agrees with the target two times in three
            tok = target[:, :k].argmax(-1)
            other = torch.randint(0, V, (B, k), generator=g, device=DEV)
            tok = torch.where(torch.rand(B, k, generator=g, device=DEV) < 0.67, tok, other)
            s["u"] = None
        s["tok"] = tok.contiguous()
        tab = _tables({"batch": B, "q": k + 1, "lo": 100, "hi": 640, "lens": 7, "page": 16}, seed)
        s["kvp"], s["idx"] = tab["kvp"].to(DEV), tab["idx"].to(DEV)
        _, kl = _lens({"batch": B, "q": k + 1, "lo": 100, "hi": 640, "lens": 7})
        s["start"] = torch.tensor([n - k - 1 for n in kl], dtype=torch.int32, device=DEV)
    elif kind == "sample":
        g = _gen(seed)
        dt = torch.float32 if case["fp32"] else BF16
        s["logits"] = _normal(g, case["rows"], case["vocab"], std=2.0, dtype=dt)
        s["u"] = torch.rand(case["rows"], generator=g, device=DEV)
    else:
        c = ModelConfig(num_hidden_layers=case["model_layers"])
        D, hkv = c.head_dim, c.num_key_value_heads
        t = _tables(case, seed)
        ql, kl = _lens(case)
        g = _gen(seed)
        s["model"] = CausalLM(c, seed=seed)
        shape = (c.num_hidden_layers, t["pages"], case["page"], hkv, D)
        s["kv"] = (_normal(g, *shape, std=0.5), _normal(g, *shape, std=0.5))
        s["wrapper"] = _planned(case, t, c.num_attention_heads, hkv, D)
        pos = torch.cat([torch.arange(n - q, n) for q, n in zip(ql, kl)])
        row = torch.repeat_interleave(torch.arange(len(ql)), torch.tensor(ql))
        page = t["idx"].long()[t["kvp"].long()[row] + pos // case["page"]]
        s["slots"] = (page * case["page"] + pos % case["page"]).to(DEV)
        s["pos"] = pos.to(DEV)
        s["ids"] = torch.randint(0, c.vocab_size, (len(pos),), generator=g, device=DEV)
        s["call"] = _model_call
    if case.get("graph"):
        _capture(s, lambda: s["call"](s))
    return s


def run(state):
    s, case = state, state["case"]
    if "replay" in s:
        s["replay"]()
        return s["out"]
    kind = s["kind"]
    if kind == "lm_head":
        if case["tokens"]:
            out = torch.empty(case["rows"], dtype=torch.int64, device=DEV)
            return kernels.lm_head_fold(s["x"], s["w"], s["ss"], 1e-6, argmax_out=out)
        return kernels.lm_head_fold(s["x"], s["w"], s["ss"], 1e-6)
    if kind == "accept":
        return kernels.spec_accept(s["target"], s["draft"] if case["temp"] else None, s["tok"],
                                   s["u"], case["temp"], s["kvp"], s["idx"], s["start"])
    if kind == "sample":
        return kernels.sample(s["logits"], case["temp"], case["top_k"], case["top_p"], s["u"])
    return s["call"](s)


# ---------------------------------------------------------------- 64 bits

def _attention64(q, keys, values):
    """Bottom-right causal attention of one request in 64 bits.
    q (n, Hq, D), keys / values (L, Hkv, D)."""
    n, hq, d = q.shape
    L, hkv = keys.shape[:2]
    limit = torch.arange(L - n, L, device=q.device)[:, None]
    cols = torch.arange(L, device=q.device)[None, :]
    out = torch.empty(n, hq, d, dtype=torch.float64, device=q.device)
    for h in range(hq):
        kh, vh = (x[:, h * hkv // hq].double() for x in (keys, values))
        for i in range(0, n, 2048):          # pieces of rows: the scores stay small
            sc = q[i:i + 2048, h].double() @ kh.T.contiguous() / math.sqrt(d)
            sc.masked_fill_(cols > limit[i:i + 2048], -math.inf)
            out[i:i + 2048, h] = torch.softmax(sc, -1) @ vh
    return out


def _paged(t, b, pool, n):
    pages = t["idx"][int(t["kvp"][b]):int(t["kvp"][b + 1])].long().to(pool.device)
    return pool[pages].reshape(-1, *pool.shape[2:])[:n]


def _attn64(case, t, q, k, v):
    ql, kl = _lens(case)
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for b, n in enumerate(kl):
        a, z = int(t["qo"][b]), int(t["qo"][b + 1])
        out[a:z] = _attention64(q[a:z], _paged(t, b, k, n), _paged(t, b, v, n))
    return out


def _norm64(x, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _mlp64(x, gate_up, down):
    y = x @ gate_up.double().T
    gate, up = y.chunk(2, -1)
    return (torch.nn.functional.silu(gate) * up) @ down.double().T


def exact(case, seed):
    kind = case["kind"]
    if kind == "attn":
        ql, kl = _lens(case)
        if case["layers"] * case["batch"] * case["hq"] > 60000:
            return None                      # too many small products in a row
        t, q, k, v = _attn_inputs(case, seed)
        return torch.stack([_attn64(case, t, q[i], k[i], v[i]) for i in range(q.shape[0])])
    if kind == "mlp":
        x, gate_up, down = _mlp_inputs(case, seed)
        H, I = case["hidden"], case["inter"]
        out = []
        for gu, dn in zip(gate_up, down):
            if case["fp8"]:
                # the weights FP8 stands for: bf16(w8 * bf16(scale)) per row
                (g8, gs), (d8, ds) = _fp8(gu, [I, I]), _fp8(dn, [H])
                gu = (g8.float() * gs[:, None]).to(BF16)
                dn = (d8.float() * ds[:, None]).to(BF16)
                out.append(_mlp64(_norm64(x.double()), gu, dn))
            else:
                out.append(x.double() + _mlp64(_norm64(x.double()), gu, dn))
        return torch.stack(out)
    if kind == "lm_head":
        if case["tokens"]:
            return None
        x, w = _lm_inputs(case, seed)
        return _norm64(x.double()) @ w.double().T
    if kind != "model":
        return None
    s = prepare({**case, "graph": False}, seed)
    m, c = s["model"], s["model"].config
    t = _tables(case, seed)
    hq, hkv, D, I = (c.num_attention_heads, c.num_key_value_heads, c.head_dim,
                     c.intermediate_size)
    cos, sin = m.rope_cos.double()[s["pos"]][:, None], m.rope_sin.double()[s["pos"]][:, None]

    def rope(z):
        a, b = z[..., :D // 2], z[..., D // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    x = m.embed.double()[s["ids"]]
    for i, L in enumerate(m.layers):
        y = _norm64(x) @ L["qkv"].double().T + L["qkv_b"].double()
        q, k, v = (z.reshape(len(x), -1, D) for z in y.split([hq * D, hkv * D, hkv * D], -1))
        kp, vp = s["kv"][0][i].double(), s["kv"][1][i].double()
        kp.view(-1, hkv, D)[s["slots"]] = rope(k)
        vp.view(-1, hkv, D)[s["slots"]] = v
        a = _attn64(case, t, rope(q), kp, vp)
        x = x + a.reshape(len(x), hq * D) @ L["o"].double().T
        x = x + _mlp64(_norm64(x), L["gate_up"], L["down"])
    return _norm64(x) @ m.lm_head.double().T
