"""The work that a user of this library has it do, as cases that can be timed and compared.

A case names one kind of pass and its sizes; the kinds are the library's call structures:

``project``  one quantized matrix on a few f32 rows, ``QMatMul.forward``: the smallest call of all (a single
             Q8_0 matrix of Qwen3-0.6B on one row), a speech model's heads and adapters, any odd shape.
``token``    one greedy decode step at one token: embedding row, decoder layers (``Qwen3DecodeLayer``: norms,
             q|k|v, attention over the cache, o, gate|up, down), final norm, LM head, argmax.  Chat and TTS
             talkers spend nearly all of their time here.
``rows``     the projections of decoder layers for several f32 rows at once: a batch of sequences that decode
             together, the candidates of a speculative step, a short prompt.  RMSNorm, q|k|v group, o with the
             residual, RMSNorm, MLP.
``prefill``  the same projections on the bf16 rows of a prompt (chat history, an ASR clip's audio tokens).
``moe``      one layer of experts at the Qwen3-30B-A3B shape (128 experts, top 8): routing, sort by expert,
             expert MLPs, combine.  One token is decode, a few are a batch, hundreds and more a prompt.

Weights are N(0, 0.02), quantized, those that add to the residual stream (o, down) smaller by
sqrt(2 layers), as models are initialised; the tied embedding is N(0, 1), so that a layer's share of the
stream is as small as in a trained model.  Activations and router logits are N(0, 1).  ``mix`` is the type mixture of a
Q4_K_M file: Q4_K with Q6_K for attn_v and ffn_down (every other layer here) and for the output matrix.
"""
from __future__ import annotations

import math

import torch

import izwi_amd as qa
from izwi_amd import capi
from izwi_amd.qwen3_layer import Qwen3DecodeLayer

Q8_0, Q4K, Q6K = qa.GgmlDType.Q8_0, qa.GgmlDType.Q4K, qa.GgmlDType.Q6K
TYPES = {"q8_0": Q8_0, "q4k": Q4K, "q6k": Q6K}
BYTES = {"q8_0": 34 / 32, "q4k": 144 / 256, "q6k": 210 / 256}
EPS = 1e-6
HEAD_DIM, KV_HEADS, VOCAB = 128, 8, 151936
# hidden, query heads, MLP width (Qwen3-0.6B and Qwen3-8B)
MODELS = {"0p6b": (1024, 16, 3072), "8b": (4096, 32, 12288)}
EXPERTS, TOP_K, MOE_HIDDEN, MOE_INTER = 128, 8, 2048, 768


def listed():
    return [
        # the smallest call: MLP up projection of Qwen3-0.6B on one row
        {"name": "project_q8_0_m1", "kind": "project", "quant": "q8_0", "n": 3072, "k": 1024, "m": 1},
        # a whole decode step of the small model (TTS talker, ASR decoder), short context
        {"name": "token_0p6b_q8_0", "kind": "token", "model": "0p6b", "quant": "q8_0", "layers": 28, "pos": 299},
        # a decode step of the chat model, longer context; eight of its 36 layers and the LM head
        {"name": "token_8b_q4k", "kind": "token", "model": "8b", "quant": "q4k", "layers": 8, "pos": 1500},
        # eight sequences decoding together
        {"name": "rows_8b_q4k_m8", "kind": "rows", "model": "8b", "quant": "q4k", "layers": 4, "m": 8},
        # 64 sequences of the small model
        {"name": "rows_0p6b_q8_0_m64", "kind": "rows", "model": "0p6b", "quant": "q8_0", "layers": 8, "m": 64},
        # a short prompt (odd length) into the chat model with a Q4_K_M file's types, f32 activations
        {"name": "rows_8b_mix_m101", "kind": "rows", "model": "8b", "quant": "mix", "layers": 2, "m": 101},
        # a prompt of ordinary length, odd
        {"name": "prefill_8b_q8_0_m500", "kind": "prefill", "model": "8b", "quant": "q8_0", "layers": 1, "m": 500},
        # a long prompt
        {"name": "prefill_8b_q4k_m2048", "kind": "prefill", "model": "8b", "quant": "q4k", "layers": 1, "m": 2048},
        # expert layers: one token, sixteen, a prompt, a long prompt
        {"name": "moe_q4k_t1", "kind": "moe", "quant": "q4k", "t": 1},
        {"name": "moe_q4k_t16", "kind": "moe", "quant": "q4k", "t": 16},
        {"name": "moe_q4k_t512", "kind": "moe", "quant": "q4k", "t": 512},
        {"name": "moe_q4k_t4096", "kind": "moe", "quant": "q4k", "t": 4096},
    ]


def _spread(rng, low, high):
    """A whole number, even over the logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(("project", "token", "rows", "rows", "prefill", "prefill", "moe", "moe"))
    if kind == "project":
        quant = rng.choice(("q8_0", "q4k", "q6k"))
        block = TYPES[quant].block_size()
        return {"kind": kind, "quant": quant, "n": _spread(rng, 64, 16384), "k": block * _spread(rng, 256 // block, 12288 // block),
                "m": _spread(rng, 1, 64)}
    if kind == "moe":
        return {"kind": kind, "quant": rng.choice(("q4k", "q4k", "q8_0")), "t": _spread(rng, 1, 4096)}
    model = rng.choice(("0p6b", "8b"))
    quant = rng.choice(("q8_0", "q4k", "mix"))
    if kind == "token":
        return {"kind": kind, "model": model, "quant": quant, "layers": rng.randint(2, 8) if model == "8b" else rng.randint(4, 28),
                "pos": _spread(rng, 1, 4095)}
    if kind == "rows":
        m = _spread(rng, 2, 512)
        # no 129 to 191 rows of the small model: when these cases were written the f32 MLP's results were wrong
        # there (its outputs shared memory with the workspace of the split along k), so none could be compared
        return {"kind": kind, "model": model, "quant": quant, "layers": rng.randint(1, 4),
                "m": m + 63 if model == "0p6b" and 128 < m < 192 else m}
    return {"kind": kind, "model": model, "quant": quant, "layers": 1, "m": _spread(rng, 65, 2048)}


# --- weights ------------------------------------------------------------------


def _q6k_blocks(w):
    """Q6_K block bytes of an f32 [n, k] matrix: a signed 8-bit scale per 16 values, taken from the value of
    the largest magnitude, 6-bit quants."""
    g = w.view(-1, 16, 16)
    far = g.gather(2, g.abs().argmax(2, keepdim=True)).squeeze(2)
    scale = far / -32.0
    d = (scale.abs().amax(1) / 127.0).to(torch.float16)
    df = d.float().unsqueeze(1)
    sc = torch.where(df > 0, torch.round(scale / df.clamp_min(1e-20)), torch.zeros_like(scale)).clamp_(-127, 127)
    step = (df * sc).unsqueeze(2)
    q = torch.where(step != 0, torch.round(g / step), torch.zeros_like(g)).clamp_(-32, 31).add_(32).to(torch.uint8)
    q = q.view(-1, 2, 4, 32)  # half, group, element
    lo, hi = q & 15, q >> 4
    ql = lo[:, :, 0:2] | (lo[:, :, 2:4] << 4)
    qh = hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)
    n = q.shape[0]
    return torch.cat([ql.reshape(n, 128), qh.reshape(n, 64), sc.to(torch.int8).view(torch.uint8), d.view(n, 1).view(torch.uint8)], 1)


def _blocks(quant, n, k, gen, std=0.02):
    """GGUF block bytes of a seeded N(0, std) [n, k] matrix, one row of the result per matrix row."""
    rows = max(1, (1 << 27) // k)
    parts = []
    for at in range(0, n, rows):
        w = torch.randn(min(rows, n - at), k, device="cuda", generator=gen) * std
        if quant == "q6k":
            parts.append(_q6k_blocks(w).view(w.shape[0], -1))
            continue
        out = torch.empty(w.shape[0], qa.quantized_storage_bytes(1, k, TYPES[quant]), dtype=torch.uint8, device="cuda")
        capi.check(capi.lib().izwi_qmm_quantize_weights_f32(int(TYPES[quant]), w.data_ptr(), w.shape[0], k, out.data_ptr(), capi.DEVICE,
                                                            torch.cuda.current_stream().cuda_stream))
        parts.append(out)
    return parts[0] if len(parts) == 1 else torch.cat(parts)


def _matrix(quant, blocks, n, k):
    torch.cuda.synchronize()  # from_blocks reads the bytes on a stream of the library's
    return qa.QMatMul.from_qtensor(qa.QTensor.from_blocks(TYPES[quant], blocks.contiguous().view(-1), (n, k)))


def _shapes(model):
    hidden, heads, inter = MODELS[model]
    q, kv = heads * HEAD_DIM, KV_HEADS * HEAD_DIM
    return {"q": (q, hidden), "k": (kv, hidden), "v": (kv, hidden), "o": (hidden, q), "gate": (inter, hidden), "up": (inter, hidden),
            "down": (hidden, inter)}


def _quant_of(quant, name, layer):
    if quant != "mix":
        return quant
    return "q6k" if name in ("v", "down") and layer % 2 == 0 or name == "head" else "q4k"


def _layers(case, gen):
    """One dict of projections per layer, every one with buffers of its own.  The first layer of a type is
    drawn; the others hold its rows in another order."""
    made, out = {}, []
    for i in range(case["layers"]):
        mm = {}
        for name, (n, k) in _shapes(case["model"]).items():
            quant = _quant_of(case["quant"], name, i)
            if (name, quant) not in made:
                std = 0.02 / math.sqrt(2 * case["layers"]) if name in ("o", "down") else 0.02
                made[name, quant] = _blocks(quant, n, k, gen, std)
            mm[name] = _matrix(quant, made[name, quant].roll(37 * i, 0), n, k)
        out.append(mm)
    return out


# --- states -------------------------------------------------------------------


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape, mean=0.0, std=1.0):
        return torch.randn(*shape, device="cuda", generator=gen) * std + mean

    kind, s = case["kind"], {"case": case}
    if kind == "project":
        n, k = case["n"], case["k"]
        s["mm"] = _matrix(case["quant"], _blocks(case["quant"], n, k, gen), n, k)
        s["x"] = randn(case["m"], k)
        return s
    if kind == "moe":
        def stack(n, k):
            blocks = _blocks(case["quant"], EXPERTS * n, k, gen)
            torch.cuda.synchronize()
            return qa.QTensor.from_blocks(TYPES[case["quant"]], blocks.view(-1), (EXPERTS, n, k))

        s["experts"] = qa.MoeExperts(stack(MOE_INTER, MOE_HIDDEN), stack(MOE_INTER, MOE_HIDDEN), stack(MOE_HIDDEN, MOE_INTER))
        s["x"], s["logits"] = randn(case["t"], MOE_HIDDEN), randn(case["t"], EXPERTS)
        return s

    hidden, heads, inter = MODELS[case["model"]]
    layers = _layers(case, gen)
    if kind == "token":
        s["layers"] = [Qwen3DecodeLayer(randn(hidden, mean=1, std=0.1), randn(hidden, mean=1, std=0.1), w["q"], w["k"], w["v"],
                                        randn(2 * HEAD_DIM, mean=1, std=0.1), w["o"], w["gate"], w["up"], w["down"], heads, KV_HEADS,
                                        HEAD_DIM, EPS) for w in layers]
        quant = _quant_of(case["quant"], "head", 0)
        s["head"] = _matrix(quant, _blocks(quant, VOCAB, hidden, gen, 1.0), VOCAB, hidden)
        s["embed"] = qa.QuantizedEmbedding(s["head"].qtensor)  # a tied checkpoint
        s["norm"] = randn(hidden, mean=1, std=0.1)
        s["token"] = torch.randint(0, VOCAB, (1,), device="cuda", dtype=torch.int32, generator=gen)
        angle = case["pos"] * 1e6 ** (-torch.arange(HEAD_DIM // 2, device="cuda", dtype=torch.float64) / (HEAD_DIM // 2))
        s["cos_sin"] = torch.cat([angle.cos(), angle.sin()]).float().view(1, HEAD_DIM)
        capacity = -(-(case["pos"] + 1) // 256) * 256
        s["caches"] = randn(case["layers"], 2, 1, KV_HEADS, capacity, HEAD_DIM)
        return s
    m = case["m"]
    s["qkv"] = [(w["q"], w["k"], w["v"]) for w in layers]
    s["o"] = [w["o"] for w in layers]
    s["down"] = [w["down"] for w in layers]
    s["x"], s["attn"] = randn(m, hidden), randn(m, heads * HEAD_DIM)  # attn: what the caller's attention gives
    if kind == "rows":
        s["norms"] = [(randn(hidden, mean=1, std=0.1), randn(hidden, mean=1, std=0.1)) for _ in layers]
        s["mlp"] = [qa.Qwen3Mlp(qa.Qwen3GateUpProjection.new_separate(w["gate"], w["up"]), w["down"]) for w in layers]
        return s
    s["gate_up"] = [(w["gate"], w["up"]) for w in layers]
    s["x"], s["attn"], s["mid"] = s["x"].bfloat16(), s["attn"].bfloat16(), randn(m, inter).bfloat16()  # mid: the caller's silu(gate) * up
    return s


# --- passes -------------------------------------------------------------------


def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


def _run_project(s):
    return s["mm"].forward(s["x"])


def _run_moe(s):
    out, ids, weights = s["experts"].layer(s["logits"], s["x"], TOP_K, return_routing=True)
    return {"out": out, "ids": ids, "weights": weights}


def _run_token(s):
    pos = s["case"]["pos"]
    x = s["embed"].forward(s["token"])
    for layer, cache in zip(s["layers"], s["caches"]):
        x = layer.forward(x, s["cos_sin"], cache[0], cache[1], pos)
    logits = s["head"].forward_normed(x, s["norm"], EPS)
    return {"token": qa.argmax(logits), "logits": logits, "hidden": x, "caches": s["caches"]}


def _run_rows(s):
    x, qkv = s["x"], []
    for group, o, mlp, (w_in, w_post) in zip(s["qkv"], s["o"], s["mlp"], s["norms"]):
        qkv.append(qa.forward_group(group, qa.try_fused_rms_norm(x, w_in, EPS)))
        x = o.forward_fused(s["attn"], residual=x)
        x = x + mlp.forward(qa.try_fused_rms_norm(x, w_post, EPS))
    return {"x": x, "qkv": qkv}


def _run_prefill(s):
    out = []
    for group, o, gate_up, down in zip(s["qkv"], s["o"], s["gate_up"], s["down"]):
        x = s["x"]
        out.append((qa.forward_group(group, x), o.forward_fused(s["attn"], residual=x), qa.forward_group(gate_up, x),
                    down.forward_fused(s["mid"], residual=x)))
    return out


# --- what a pass cannot do without ----------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "project":
        n, k, m = case["n"], case["k"], case["m"]
        return {"bytes": n * k * BYTES[case["quant"]] + 4 * m * (k + n), "flops": 2 * m * n * k}
    if kind == "moe":
        t = case["t"]
        used = EXPERTS * (1 - (1 - TOP_K / EXPERTS) ** t)  # experts that some token takes, on average
        per = 3 * MOE_INTER * MOE_HIDDEN
        return {"bytes": used * per * BYTES[case["quant"]] + t * (8 * MOE_HIDDEN + 4 * EXPERTS + 8 * TOP_K), "flops": 2 * t * TOP_K * per}
    hidden, heads, inter = MODELS[case["model"]]
    m = case.get("m", 1)
    size = 4 if kind != "prefill" else 2
    nbytes = flops = 0
    for i in range(case["layers"]):
        for name, (n, k) in _shapes(case["model"]).items():
            nbytes += n * k * BYTES[_quant_of(case["quant"], name, i)]
            flops += 2 * m * n * k
    qkv = (heads + 2 * KV_HEADS) * HEAD_DIM
    if kind == "token":
        kv = 2 * KV_HEADS * HEAD_DIM * (case["pos"] + 1)
        nbytes += case["layers"] * (4 * kv + 16 * hidden) + VOCAB * (hidden * BYTES[_quant_of(case["quant"], "head", 0)] + 4)
        flops += case["layers"] * 4 * heads * HEAD_DIM * (case["pos"] + 1) + 2 * VOCAB * hidden
    elif kind == "rows":
        nbytes += size * m * (2 * hidden + heads * HEAD_DIM + case["layers"] * qkv)
    else:
        nbytes += size * m * (hidden + heads * HEAD_DIM + inter + case["layers"] * (qkv + 2 * hidden + 2 * inter))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what the path differs from itself by with its f32 sums in another order (other kernel
    forms, other splits of k), over the listed cases and thirty drawn ones."""
    if case["kind"] == "project":  # integer block dots: the f32 sums alone, 1.3e-7 measured
        return {"rel": 1e-6, "max": 1e-5}
    if case["kind"] == "token":
        # 7e-3 (K-quants) to 2e-2 (q8_0): a last bit moves an 8-bit activation quant of a later layer across a
        # rounding boundary now and then, and every quantization after that passes it on
        return {"rel": 0.03, "max": 0.3}
    if case["kind"] == "rows":  # the same over up to four layers, 3.9e-3; beyond 64 rows bf16 roundings, 1.3e-3
        return {"rel": 0.016, "max": 0.13} if case["m"] <= 64 else {"rel": 5e-3, "max": 0.04}
    if case["kind"] == "prefill":  # one product each: bf16 results one rounding apart, 5e-5
        return {"rel": 2e-4, "max": 0.03}
    return {"rel": 5e-4, "max": 0.02}  # moe: activation quants of the second product, 1.3e-4
