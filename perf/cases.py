"""What the framework's speed is measured on: the calls its users make, through the public entry points.

`listed()` holds twelve fixed cases, `draw(rng)` gives one more of the same kinds with sizes spread over the same
ranges.  `prepare` makes what a program holds before the call (weights in their resident form, activations, a model
with its caches), `run` is one pass, `work` what that pass cannot do without, `tolerance` how far another correct
implementation of the same precision may be from it.

Kinds of work:
  matmul   QuantizedMatmul (f32 / f16 activations) or QuantizedMatmulBf16: one activation row up to a long prompt
  moe      route_topk and MoEExperts.process: the router and the MXFP4 expert layer
  chat     LlamaQ8: a prompt in f32 (the default), then greedy decode steps from the replayed graph
  prompt   LlamaQ8.prefill(bf16=True): a prompt on the bf16 matrix cores
  step     LlamaQ8.forward_decode: one token at the end of a long context
"""
import math

import torch

from luminal_amd import capi, synth
from luminal_amd.llama import LLAMA3_8B, LlamaQ8, random_weights
from luminal_amd.moe import MoEExperts, Mxfp4Weight, route_topk
from luminal_amd.quantized import Q8Weight, QuantizedMatmul, QuantizedMatmulBf16

DEV = "cuda:0"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}

# Ranges of the drawn cases.
MAX_ROWS = {"f32": 512, "f16": 512, "bf16": 2048}
MIN_N, MAX_N = 256, 14336
MIN_K, MAX_K = 512, 14336
MAX_PROMPT, MAX_CHAT_PROMPT, MAX_CHAT_STEPS, MAX_CONTEXT = 2000, 300, 32, 8000


def _matmul(name, dtype, m, n, k):
    return {"name": name, "kind": "matmul", "dtype": dtype, "m": m, "n": n, "k": k}


def listed():
    gate, down = synth.LLAMA3_8B_PROJ["gate"], synth.LLAMA3_8B_PROJ["down"]
    return [
        # one token through the smallest projection (k or v): nothing but launch and latency
        _matmul("matvec_f32_1_kv", "f32", 1, *synth.LLAMA3_8B_PROJ["k"]),
        # a batch of three sequences decoding in f16, the type the reference's own example runs in
        _matmul("rows_f16_3_qo", "f16", 3, *synth.LLAMA3_8B_PROJ["q"]),
        # a short prompt through a layer whose width is no multiple of a power-of-two tile (the MoE model's)
        _matmul("rows_f32_45_ragged", "f32", 45, synth.MOE_HIDDEN, synth.MOE_HIDDEN),
        # prompts through the reference's operator in its two activation types
        _matmul("rows_f32_256_gate", "f32", 256, *gate),
        _matmul("rows_f16_512_down", "f16", 512, *down),
        # sixteen sequences decoding in bf16: the weights are read for sixteen rows
        _matmul("gemm_bf16_16_gate", "bf16", 16, *gate),
        # a long prompt in bf16
        _matmul("gemm_bf16_2048_gate", "bf16", 2048, *gate),
        # a mixture-of-experts layer for one decoding sequence, and for a prompt
        {"name": "moe_1", "kind": "moe", "mode": "exact", "t": 1},
        {"name": "moe_1024", "kind": "moe", "mode": "exact", "t": 1024},
        # a question and its answer with the engine's defaults
        {"name": "chat_300_32", "kind": "chat", "prompt": 300, "steps": 32, "q8_embed": False},
        # a document read in bf16
        {"name": "prompt_bf16_2000", "kind": "prompt", "prompt": 2000, "q8_embed": False},
        # one more token behind a long document
        {"name": "step_8000", "kind": "step", "context": 8000, "q8_embed": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matmul"] * 6 + ["moe"] * 2 + ["chat", "prompt", "step"])
    if kind == "matmul":
        dtype = rng.choice(["f32", "f16", "bf16"])
        # half the matrices have a width that is a multiple of 1024, the others any the type's operator takes
        step = rng.choice([1024, 64 if dtype == "bf16" else 32])
        k = max(MIN_K, _log_int(rng, MIN_K, MAX_K) // step * step)
        n = _log_int(rng, MIN_N, MAX_N)
        if rng.random() < 0.75:
            n = n // 4 * 4
        m = _log_int(rng, 1, MAX_ROWS[dtype])
        largest = 512 if dtype != "bf16" else 2048
        # no dearer than the largest listed product of the type
        while m * n * k > largest * MAX_N * 4096:
            m = max(1, m // 2)
        return {"kind": kind, "dtype": dtype, "m": m, "n": n, "k": k}
    if kind == "moe":
        return {"kind": kind, "mode": rng.choice(["exact", "exact", "fast"]), "t": _log_int(rng, 1, 1024)}
    q8_embed = rng.random() < 0.5
    if kind == "chat":
        return {"kind": kind, "prompt": _log_int(rng, 2, MAX_CHAT_PROMPT), "steps": rng.randint(4, MAX_CHAT_STEPS),
                "q8_embed": q8_embed}
    if kind == "prompt":
        return {"kind": kind, "prompt": _log_int(rng, 16, MAX_PROMPT), "q8_embed": q8_embed}
    return {"kind": kind, "context": _log_int(rng, 32, MAX_CONTEXT), "q8_embed": q8_embed}


# ---- inputs ---------------------------------------------------------------------------------------------------------

def _generator(seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    return gen


def _q8_weight(n, k, gen):
    """Quants U{-127..127}, block scales |N(0, 0.02)| / 127, as `synth.q8_0_random`, made on the device."""
    blocks = n * k // 32
    raw = torch.empty((blocks, 34), dtype=torch.uint8, device=DEV)
    d = torch.randn((blocks, 1), device=DEV, generator=gen).abs() * (0.02 / 127.0)
    raw[:, :2] = d.to(torch.float16).view(torch.uint8)
    raw[:, 2:] = torch.randint(-127, 128, (blocks, 32), dtype=torch.int8, device=DEV, generator=gen).view(torch.uint8)
    return Q8Weight.from_raw(raw, n, k, DEV)


def _mxfp4_weight(n, k, gen):
    """e2m1 codes uniform over the 16 values, block scales 2^-8 .. 2^0, as `synth.mxfp4_random`."""
    blocks = n * k // 32
    raw = torch.empty((blocks, 17), dtype=torch.uint8, device=DEV)
    raw[:, :16] = torch.randint(0, 256, (blocks, 16), dtype=torch.uint8, device=DEV, generator=gen)
    raw[:, 16] = torch.randint(127 - 8, 127 + 1, (blocks,), dtype=torch.uint8, device=DEV, generator=gen)
    return Mxfp4Weight.from_raw(raw, n, k, DEV)


def _llama(case, seed, gen):
    cfg = LLAMA3_8B
    weights = random_weights(cfg, seed, DEV)
    if case["q8_embed"]:
        weights["embed"] = _q8_weight(cfg.vocab, cfg.dim, gen)
    tokens = case.get("prompt", case.get("context"))
    room = tokens + case.get("steps", 0) + 2
    model = LlamaQ8(cfg, weights, max_seq=(room + 255) // 256 * 256, device=DEV)
    ids = torch.randint(0, cfg.vocab, (tokens,), device=DEV, generator=gen).cpu().numpy()
    return {"case": case, "model": model, "ids": ids}


def prepare(case, seed):
    gen = _generator(seed)
    if case["kind"] == "matmul":
        w = _q8_weight(case["n"], case["k"], gen)
        x = torch.randn((case["m"], case["k"]), device=DEV, generator=gen).to(DTYPES[case["dtype"]])
        op = QuantizedMatmulBf16() if case["dtype"] == "bf16" else QuantizedMatmul()
        return {"case": case, "op": op, "x": x, "w": w}
    if case["kind"] == "moe":
        h, i, e = synth.MOE_HIDDEN, synth.MOE_INTER, synth.MOE_EXPERTS
        experts = MoEExperts(_mxfp4_weight(e * 2 * i, h, gen), _mxfp4_weight(e * h, i, gen), e, h, i)
        x = torch.randn((case["t"], h), device=DEV, generator=gen).to(torch.bfloat16)
        logits = torch.randn((case["t"], e), device=DEV, generator=gen)
        mode = capi.LHIP_MOE_EXACT if case["mode"] == "exact" else capi.LHIP_MOE_FAST
        return {"case": case, "experts": experts, "x": x, "logits": logits, "mode": mode}
    state = _llama(case, seed, gen)
    if case["kind"] == "step":
        state["model"].prefill(state["ids"])
        state["token"] = torch.randint(0, LLAMA3_8B.vocab, (1,), device=DEV, generator=gen).to(torch.float32)
    return state


# ---- one pass -------------------------------------------------------------------------------------------------------

def _caches(model):
    """The updated state: the keys of every layer and the values of the last, which all that was computed before reach."""
    return (*model.k_cache, model.v_cache[-1])


def run(state):
    kind = state["case"]["kind"]
    if kind == "matmul":
        return state["op"].process(state["x"], state["w"])
    if kind == "moe":
        sel, wts = route_topk(state["logits"], synth.MOE_TOPK)
        return state["experts"].process(state["x"], sel, wts, state["mode"]), sel, wts
    model = state["model"]
    if kind == "chat":
        model.reset()
        model.prefill(state["ids"])
        tokens = model.decode(state["case"]["steps"])
        return (tokens, model.decode_step(), model.tok_i, *_caches(model))
    if kind == "prompt":
        model.reset()
        # the logits and caches, not the pick: which of two near ties bf16 rounding leaves ahead is no result
        return (model.prefill(state["ids"], bf16=True), *_caches(model))
    return (model.forward_decode(state["token"]), *_caches(model))


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def _q8_bytes(n, k):
    return n * k * 34 // 32


def _llama_matrices(cfg):
    """(n, k) of the matrices every token passes through, the vocabulary's apart."""
    layer = [(cfg.qkv_rows, cfg.dim), (cfg.dim, cfg.dim), (2 * cfg.ffn, cfg.dim), (cfg.dim, cfg.ffn)]
    return layer * cfg.layers


def _llama_pass(cfg, tokens, before):
    """Bytes and flops of `tokens` tokens behind `before` others, the last one's logits among the results."""
    body, head = _llama_matrices(cfg), (cfg.vocab, cfg.dim)
    kv_row = 2 * cfg.kv_heads * cfg.head_dim * 4  # keys and values are kept in f32
    nbytes = sum(_q8_bytes(n, k) for n, k in body) + _q8_bytes(*head) + 4 * cfg.vocab + tokens * 4 * cfg.dim
    nbytes += cfg.layers * kv_row * (before + tokens)
    flops = tokens * sum(2 * n * k for n, k in body) + 2 * head[0] * head[1]
    seen = tokens * before + tokens * (tokens + 1) // 2
    flops += cfg.layers * cfg.q_heads * seen * 4 * cfg.head_dim
    return nbytes, flops


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _q8_bytes(n, k) + (m * k + m * n) * (4 if case["dtype"] == "f32" else 2), "flops": 2 * m * n * k}
    if kind == "moe":
        t, h, i, e, top = case["t"], synth.MOE_HIDDEN, synth.MOE_INTER, synth.MOE_EXPERTS, synth.MOE_TOPK
        touched = e * (1.0 - (1.0 - top / e) ** t)
        return {"bytes": int(touched * 3 * h * i * 17 // 32) + t * (4 * h + 4 * e + 8 * top), "flops": t * top * 6 * h * i}
    cfg = LLAMA3_8B
    if kind == "chat":
        parts = [_llama_pass(cfg, case["prompt"], 0)]
        parts += [_llama_pass(cfg, 1, case["prompt"] + s) for s in range(case["steps"] + 1)]
    elif kind == "prompt":
        parts = [_llama_pass(cfg, case["prompt"], 0)]
    else:
        parts = [_llama_pass(cfg, 1, case["context"])]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


# Four times the largest difference seen on an MI355X (2-norm, and largest element over the rms): the matmuls and the
# expert layer against the same product in 64 bits over the exactly dequantised weights, the model against the same
# tokens read in two pieces (other kernels' shapes and other orders of additions) and decoded by the unfused operators.
_MATMUL_TOLERANCE = {
    "f32": {"rel": 8.5e-7, "max": 1.1e-5},   # 2.1e-7, 2.7e-6: the order of f32 additions
    "f16": {"rel": 8.3e-4, "max": 6e-3},     # 2.1e-4, 1.5e-3: the f16 result
    "bf16": {"rel": 6.6e-3, "max": 6.8e-2},  # 1.7e-3, 1.7e-2: the bf16 result
}


def tolerance(case):
    kind = case["kind"]
    if kind == "matmul":
        return dict(_MATMUL_TOLERANCE[case["dtype"]])
    if kind == "moe":  # 2.4e-3, 2.0e-2: two roundings to bf16, the SwiGLU rows and the result
        return {"rel": 9.4e-3, "max": 7.9e-2}
    if kind == "prompt":  # 1.3e-2, 6.2e-2: 32 layers of bf16 operands
        return {"rel": 5.2e-2, "max": 2.5e-1}
    return {"rel": 1.1e-5, "max": 5.2e-5}  # 2.7e-6, 1.3e-5: 32 layers of f32 sums; the tokens stay the same
