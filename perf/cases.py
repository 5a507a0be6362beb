"""Performance cases of the k-quant path: the calls a decoder-only language model makes on GGUF weights.

kind     one pass                                                             stands for
linear   kquant.matmul on fp32 rows                                           a single projection: a decode matvec, an odd-sized
                                                                              or biased layer, a batch of sequences
step     per layer norm -> q|k|v, o + residual, norm -> gate|up -> act,       a decode step, a speculative-verify batch, a decode
         down + residual (kquant.matmul_fused), then lm_head and the          step of many sequences at once, a short prompt
         greedy pick (kquant.matmul_argmax); fp32, 1 .. 128 tokens
prefill  the same layer on bf16 activations: kquant.prefill_rows_bf16 in      a prompt or a chunk of one, 32 .. 2048 tokens
         front of kquant.matmul
moe      kquant.moe_route and kquant.moe_ffn                                  the routed-expert block of a mixture model, from one
                                                                              token to a prompt chunk of 2048
embed    kquant.dequant_rows for a list of token ids                          the embedding lookup of a prompt

Attention is not part of this path, so what it would return (the input of o) is an input of a pass.  Weights: random
GGUF superblocks with the field distributions of backpack_amd/synth.py, their super-scales set so that a matrix has
weights of mean 0 and rms 1 / sqrt(K), as a model's have: activations then keep their size through a stack of layers.
"""
from __future__ import annotations

import math

import torch

from backpack_amd import capi, kquant, synth

Q4_K, Q5_K, Q6_K = synth.Q4_K, synth.Q5_K, synth.Q6_K
EPS = 1e-5

# rms of a weight over the rms of a block's super-scale d, for the field distributions used here, and dmin over d: the
# mean of the quants, so that the minima centre the weights
_GAIN = {Q4_K: 258.0, Q5_K: 527.0, Q6_K: 683.0}
_CENTRE = {Q4_K: 7.5, Q5_K: 15.5}


def listed():
    L, E = synth.LLAMA3_8B, synth.QWEN3_30B_A3B
    llama = {"hidden": L["hidden"], "kv": 1024, "inter": 14336, "type": Q4_K, "down": Q6_K}
    qwen = {"experts": E["n_experts"], "top_k": E["top_k"], "hidden": E["hidden"], "inter": E["inter"],
            "type": E["gate_up_type"], "down": E["down_type"]}
    return [
        # the smallest call: one decode projection, where latency and the host's share count
        {"name": "linear_decode", "kind": "linear", "type": Q4_K, "M": 1, "N": 4096, "K": 4096, "bias": False},
        # odd sizes, a bias, the third weight type, three drafted tokens
        {"name": "linear_ragged", "kind": "linear", "type": Q5_K, "M": 3, "N": 5003, "K": 2816, "bias": True},
        # one token of one sequence through layers and lm_head
        {"name": "step_decode", "kind": "step", "M": 1, "layers": 8, "vocab": 128256, **llama},
        # eight drafted tokens verified at once
        {"name": "step_verify", "kind": "step", "M": 8, "layers": 4, "vocab": 128256, **llama},
        # one token of each of 48 sequences
        {"name": "step_batch", "kind": "step", "M": 48, "layers": 2, "vocab": 128256, **llama},
        # a short prompt, a ragged number of tokens
        {"name": "prefill_short", "kind": "prefill", "M": 100, **llama},
        # a full prompt chunk
        {"name": "prefill_long", "kind": "prefill", "M": 2048, **llama},
        # a mixture layer: one token, a few sequences, a short prompt, a prompt chunk
        {"name": "moe_decode", "kind": "moe", "T": 1, **qwen},
        {"name": "moe_batch", "kind": "moe", "T": 24, **qwen},
        {"name": "moe_prompt", "kind": "moe", "T": 256, **qwen},
        {"name": "moe_chunk", "kind": "moe", "T": 2048, **qwen},
        # the embedding lookup of a prompt, from a vocabulary-sized Q6_K matrix
        {"name": "embed_prompt", "kind": "embed", "type": Q6_K, "M": 512, "N": 128256, "K": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _layer(rng):
    hidden = 256 * _log(rng, 4, 16)
    return {"hidden": hidden, "kv": 256 * max(1, hidden // 1024), "inter": 256 * int(hidden * rng.uniform(2.5, 3.5) / 256),
            **rng.choice([{"type": Q4_K, "down": Q6_K}, {"type": Q4_K, "down": Q6_K}, {"type": Q5_K, "down": Q6_K},
                          {"type": Q4_K, "down": Q4_K}, {"type": Q6_K, "down": Q6_K}])}


def draw(rng):
    kind = rng.choice(["linear", "step", "step", "prefill", "prefill", "moe", "moe", "embed"])
    if kind == "linear":
        return {"kind": kind, "type": rng.choice([Q4_K, Q5_K, Q6_K]), "M": _log(rng, 1, 128), "N": _log(rng, 512, 32768),
                "K": 256 * _log(rng, 2, 56), "bias": rng.random() < 0.5}
    if kind == "step":
        c = {"kind": kind, "M": _log(rng, 1, 128), **_layer(rng), "vocab": _log(rng, 32000, 128256)}
        c["layers"] = rng.randint(1, 4)
        while _tokens_times_weights(c) > _tokens_times_weights(next(k for k in listed() if k["name"] == "step_batch")):
            if c["layers"] > 1:
                c["layers"] -= 1
            else:
                c["vocab"] = max(4001, int(c["vocab"] * 0.7))
                c["M"] -= c["M"] // 8
        return c
    if kind == "prefill":
        return {"kind": kind, "M": _log(rng, 32, 2048), **_layer(rng)}
    if kind == "moe":
        experts = rng.choice([8, 16, 32, 64, 128])
        return {"kind": kind, "T": _log(rng, 1, 2048), "experts": experts, "top_k": rng.randint(2, min(8, experts // 2)),
                "hidden": 256 * _log(rng, 4, 8), "inter": 256 * _log(rng, 2, 3),
                **rng.choice([{"type": Q4_K, "down": Q6_K}, {"type": Q4_K, "down": Q6_K}, {"type": Q4_K, "down": Q4_K},
                              {"type": Q5_K, "down": Q6_K}])}
    return {"kind": kind, "type": rng.choice([Q4_K, Q5_K, Q6_K, Q6_K]), "M": _log(rng, 1, 4096), "N": _log(rng, 32000, 128256),
            "K": 256 * _log(rng, 4, 16)}


def _matrices(c):
    """(type, N, K) of a layer: q|k|v, o, gate|up, down."""
    H, I, t = c["hidden"], c["inter"], c["type"]
    return [(t, H + 2 * c["kv"], H), (t, H, H), (t, 2 * I, H), (c["down"], H, I)]


def _tokens_times_weights(c):
    return c["M"] * (c["layers"] * sum(n * k for _, n, k in _matrices(c)) + c["vocab"] * c["hidden"])


# --------------------------------------------------------------------------------------------------------------
def _weight(g, type_, N, K):
    nb, bb, rs = synth.n_blocks(K), synth.BLOCK_BYTES[type_], 4 * synth.row_stride_words(type_, K)
    data = torch.randint(0, 256, (N * rs + 16,), dtype=torch.uint8, device="cuda", generator=g)
    rows = data[: N * rs].view(N, rs)
    rows[:, nb * bb:] = 0
    blk = rows[:, : nb * bb].unflatten(1, (nb, bb))
    sigma = 1.0 / (_GAIN[type_] * math.sqrt(K))

    d = (torch.randn((N, nb, 1), device="cuda", generator=g) * sigma).abs()
    if type_ == Q6_K:
        blk[:, :, 192:208] = torch.randint(-64, 64, (N, nb, 16), dtype=torch.int8, device="cuda", generator=g).view(torch.uint8)
        blk[:, :, 208:210] = d.to(torch.float16).view(torch.uint8)
    else:
        blk[:, :, 0:4] = torch.cat([d, d * _CENTRE[type_]], dim=2).to(torch.float16).view(torch.uint8)
    return kquant.KQuantPacked(data, type_, N, K, rs // 4, nb)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rows(*shape):
        return torch.randn(shape, device="cuda", generator=g)
    kind = case["kind"]
    s = {"case": case}
    if kind == "linear":
        s["w"] = _weight(g, case["type"], case["N"], case["K"])
        s["x"] = rows(case["M"], case["K"])
        s["bias"] = rows(case["N"]) if case["bias"] else None
    elif kind in ("step", "prefill"):
        M, H, I = case["M"], case["hidden"], case["inter"]
        s["layers"] = []
        for _ in range(case.get("layers", 1)):
            qkv, o, gate_up, down = (_weight(g, *m) for m in _matrices(case))
            s["layers"].append({"qkv": qkv, "o": o, "gate_up": gate_up, "down": down, "attn": rows(M, H),
                                "norm1": 1.0 + 0.1 * rows(H), "norm2": 1.0 + 0.1 * rows(H)})
        s["x"] = rows(M, H)
        if kind == "step":
            s["head"] = _weight(g, case["down"], case["vocab"], H)
            n = max(capi.lib().bpk_kq_matmul_fused_workspace_bytes(M, n, k) for n, k in ((H + 2 * case["kv"], H), (I, H), (H, I)))
            s["ws"] = torch.empty(n, dtype=torch.uint8, device="cuda")
    elif kind == "moe":
        E, H, I = case["experts"], case["hidden"], case["inter"]
        s["gate"], s["up"] = (_weight(g, case["type"], E * I, H) for _ in range(2))
        s["down"] = _weight(g, case["down"], E * H, I)
        s["router"] = rows(E, H) / math.sqrt(H)
        s["x"] = rows(case["T"], H)
    else:
        s["w"] = _weight(g, case["type"], case["N"], case["K"])
        s["rows"] = torch.randint(0, case["N"], (case["M"],), dtype=torch.int32, device="cuda", generator=g)
    return s


def run(s):
    return _RUN[s["case"]["kind"]](s)


def _run_linear(s):
    return kquant.matmul(s["x"], s["w"], bias=s["bias"])


def _run_step(s):
    x, ws, out = s["x"], s["ws"], []
    for l in s["layers"]:
        out.append(kquant.matmul_fused(x, l["qkv"], capi.PRO_RMS_NORM, norm_w=l["norm1"], eps=EPS, workspace=ws))
        x = kquant.matmul_fused(l["attn"], l["o"], residual=x, workspace=ws)
        act = kquant.matmul_fused(x, l["gate_up"], capi.PRO_RMS_NORM, norm_w=l["norm2"], eps=EPS, workspace=ws,
                                  epilogue=capi.EPI_SILU_MUL)
        x = kquant.matmul_fused(act, l["down"], residual=x, workspace=ws)
    logits, token, value = kquant.matmul_argmax(x, s["head"])
    return {"qkv": out, "x": x, "logits": logits, "token": token, "value": value}


def _run_prefill(s):
    x, out = s["x"], []
    for l in s["layers"]:
        H, I = l["qkv"].K, l["down"].K
        out.append(kquant.matmul(kquant.prefill_rows_bf16(x, H, capi.PRO_RMS_NORM, norm_w=l["norm1"], eps=EPS), l["qkv"]))
        x = x + kquant.matmul(kquant.prefill_rows_bf16(l["attn"], H), l["o"])
        gate_up = kquant.matmul(kquant.prefill_rows_bf16(x, H, capi.PRO_RMS_NORM, norm_w=l["norm2"], eps=EPS), l["gate_up"])
        x = x + kquant.matmul(kquant.prefill_rows_bf16(gate_up, I, capi.PRO_SILU_MUL), l["down"])
    return {"qkv": out, "x": x}


def _run_moe(s):
    idx, wt = kquant.moe_route(s["x"], s["router"], s["case"]["top_k"])
    y = kquant.moe_ffn(s["x"], s["gate"], s["up"], s["down"], idx, wt, s["case"]["experts"])
    return {"y": y, "experts": idx, "weights": wt}


def _run_embed(s):
    return kquant.dequant_rows(s["w"], s["rows"])


_RUN = {"linear": _run_linear, "step": _run_step, "prefill": _run_prefill, "moe": _run_moe, "embed": _run_embed}


# --------------------------------------------------------------------------------------------------------------
def _dense(w, rows=None):
    """Rows of a packed matrix in float64, as the GGUF formats define them."""
    bb = synth.BLOCK_BYTES[w.type]
    b = w.data[: w.N * w.row_stride_bytes].view(w.N, w.row_stride_bytes)[:, : w.n_blocks * bb]
    b = (b if rows is None else b[rows]).unflatten(1, (w.n_blocks, bb))

    def f16(i):
        return b[:, :, i:i + 2].contiguous().view(torch.float16).double()
    if w.type == Q6_K:
        ql, qh = b[:, :, :128].unflatten(2, (2, 2, 32)), b[:, :, 128:192].unflatten(2, (2, 32))
        q = torch.stack([(ql[:, :, :, t & 1] >> (4 * (t >> 1)) & 15) | (qh >> (2 * t) & 3) << 4 for t in range(4)], 3)
        sc = b[:, :, 192:208].contiguous().view(torch.int8).double().repeat_interleave(16, 2)
        return (f16(208) * sc * (q.flatten(2).double() - 32)).flatten(1)
    s = b[:, :, 4:16].to(torch.int32)
    lo, mid, hi = s[:, :, :4], s[:, :, 4:8], s[:, :, 8:]
    sc = torch.cat([lo & 63, hi & 15 | lo >> 6 << 4], 2).double().repeat_interleave(32, 2)
    mn = torch.cat([mid & 63, hi >> 4 | mid >> 6 << 4], 2).double().repeat_interleave(32, 2)
    qs = b[:, :, -128:].unflatten(2, (4, 32))
    q = torch.stack([qs & 15, qs >> 4], 3).flatten(2)
    if w.type == Q5_K:
        q = q | torch.stack([b[:, :, 16:48] >> i & 1 for i in range(8)], 2).flatten(2) << 4
    return (f16(0) * sc * q.double() - f16(2) * mn).flatten(1)


def _product(x, w, step=16384):
    return torch.cat([x @ _dense(w, slice(i, i + step)).T for i in range(0, w.N, step)], 1)


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(1, keepdim=True) + EPS) * w.double()


def _silu_mul(gate_up):
    gate, up = gate_up.chunk(2, 1)
    return torch.nn.functional.silu(gate) * up


def exact(case, seed):
    """The outputs of a pass in float64; a prefill's activation rows are bf16, which prefill_rows_bf16 returns."""
    s, kind = prepare(case, seed), case["kind"]
    if kind == "embed":
        return _dense(s["w"], s["rows"].long())
    x = s["x"].double()
    if kind == "linear":
        y = _product(x, s["w"])
        return y if s["bias"] is None else y + s["bias"].double()
    if kind == "moe":
        E, H, I = case["experts"], case["hidden"], case["inter"]
        top, idx = torch.topk(x @ s["router"].double().T, case["top_k"], dim=1)
        wt = torch.softmax(top, 1)
        y = torch.zeros_like(x)
        for e in range(E):
            t, slot = (idx == e).nonzero(as_tuple=True)
            if len(t):
                xe = x[t]
                act = _silu_mul(torch.cat([xe @ _dense(w, slice(e * I, e * I + I)).T for w in (s["gate"], s["up"])], 1))
                y.index_add_(0, t, wt[t, slot, None] * (act @ _dense(s["down"], slice(e * H, e * H + H)).T))
        return {"y": y, "experts": idx.int(), "weights": wt}
    rows = (lambda v: v.bfloat16().double()) if kind == "prefill" else (lambda v: v)
    out = []
    for l in s["layers"]:
        out.append(_product(rows(_norm(x, l["norm1"])), l["qkv"]))
        x = x + _product(rows(l["attn"].double()), l["o"])
        x = x + _product(rows(_silu_mul(_product(rows(_norm(x, l["norm2"])), l["gate_up"]))), l["down"])
    if kind == "prefill":
        return {"qkv": out, "x": x}
    logits = _product(x, s["head"])
    value, token = logits.max(1)
    return {"qkv": out, "x": x, "logits": logits, "token": token.int(), "value": value}


def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": synth.weight_bytes(case["type"], N, K) + 4 * M * (K + N) + (4 * N if case["bias"] else 0),
                "flops": 2.0 * M * N * K}
    if kind in ("step", "prefill"):
        M, H, n = case["M"], case["hidden"], case.get("layers", 1)
        mats = _matrices(case) * n
        b = sum(synth.weight_bytes(*m) for m in mats)
        # x in, attention's output in, q|k|v out, per layer; the last x out; logits out
        b += 4 * M * (n * (2 * H + 2 * case["kv"]) + 2 * H) + 8 * H * n
        f = 2.0 * M * sum(N * K for _, N, K in mats)
        if kind == "step":
            b += synth.weight_bytes(case["down"], case["vocab"], H) + 4 * M * case["vocab"] + 8 * M
            f += 2.0 * M * case["vocab"] * H
        return {"bytes": b, "flops": f}
    if kind == "moe":
        T, k, E, H, I = case["T"], case["top_k"], case["experts"], case["hidden"], case["inter"]
        touched = E * (1.0 - (1.0 - k / E) ** T)   # experts expected to be chosen by at least one token
        per = 2 * synth.weight_bytes(case["type"], I, H) + synth.weight_bytes(case["down"], H, I)
        return {"bytes": touched * per + 4 * E * H + 4 * T * 2 * H + 8 * T * k, "flops": 2.0 * T * (k * 3 * H * I + E * H)}
    M, K = case["M"], case["K"]
    return {"bytes": synth.weight_bytes(case["type"], M, K) + 4 * M * K + 4 * M, "flops": 0.0}


def tolerance(case):
    # Four times what the library's kernels differ by among each other (the generic fp32 kernel against the chosen
    # ones; one GEMM tiling against another): 8e-6 through four layers of eight tokens, 2.2e-6 in a mixture layer,
    # 9e-5 where a bf16 activation rounds the other way.  differ: near-ties of the greedy pick and of the router.
    return {"linear": {"rel": 1e-5}, "step": {"rel": 3e-5, "differ": 0.03}, "prefill": {"rel": 4e-4},
            "moe": {"rel": 1e-5, "differ": 1e-3}, "embed": "exact"}[case["kind"]]
