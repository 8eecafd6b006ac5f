"""Workloads of the GEMM / fused-attention library, for timing it and for comparing two builds of it.

A case is a dict of plain values; ``prepare`` makes the operands a user's program has in hand, ``run`` is one pass through the
public entry points (``Mi355Engine`` operators and ``Mi355Backend`` members).  The kinds:

linear         activation(x W + b) of one dense layer (``FusedLinear``; storage "f16w": fp32 activations on fp16 weights)
matmul         the plain product x W (``TensorMatMul``)
mha            a multi-head attention layer, four projections and an optional padding mask (``MultiHeadAttentionForward``)
sdpa           fp32 scaled dot-product attention, by default with its probabilities (``ScaledDotProductAttention``)
prefill        flash attention with log-sum-exp over whole sequences (``FlashAttention``)
decode_step    one token per sequence: Q and K/V projections with the rotary embedding, attention over the cache, output projection
paged_decode   one query over a block-table cache (``PagedAttentionHalf`` / ``PagedAttentionDecode[Gqa]``)
paged_prefill  a chunk of queries after a prefix that is already in such a cache

The backend is used the way a serving loop uses it: calls only enqueue, and the block tables, which the program itself wrote, are
not read back on every call.
"""
from __future__ import annotations

import math

import torch

from aidotnet.tensors_amd import Mi355Backend, Mi355Engine

_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2}
_ENGINE = []


def _engine() -> Mi355Engine:
    if not _ENGINE:
        _ENGINE.append(Mi355Engine(Mi355Backend(synchronous=False, validate_block_tables=False)))
    return _ENGINE[0]


def listed():
    return [
        # the smallest call: a batch of eight through one 768-wide fp32 layer -- launch and latency
        dict(name="linear_f32_small", kind="linear", dtype="f32", M=8, N=768, K=768, act="ReLU"),
        # the feed-forward up-projection of a 768-wide fp32 encoder over 8 x 512 tokens
        dict(name="linear_f32_ffn", kind="linear", dtype="f32", M=4096, N=3072, K=768, act="GELU"),
        # a batch of prompts whose tokens do not fill whole tiles, through a wide bf16 layer
        dict(name="linear_bf16_ragged", kind="linear", dtype="bf16", M=1000, N=11008, K=4096, act="Swish"),
        # the largest call: a square half-precision product
        dict(name="matmul_f16_8192", kind="matmul", dtype="f16", M=8192, N=8192, K=8192),
        # logits over a vocabulary of odd size for 64 sequences
        dict(name="matmul_bf16_vocab", kind="matmul", dtype="bf16", M=64, N=50257, K=768),
        # an attention layer of a 768-wide encoder over a padded batch
        dict(name="mha_bf16_padded", kind="mha", dtype="bf16", B=8, S=512, dModel=768, H=12, padded=True),
        # the operator with its default of returning the probabilities, causal
        dict(name="sdpa_f32_weights", kind="sdpa", B=4, H=12, Hkv=12, Sq=512, Sk=512, D=64, causal=True, padded=False, softcap=0.0, weights=True),
        # prompt processing: four prompts of 2048 tokens
        dict(name="prefill_bf16", kind="prefill", dtype="bf16", B=4, H=32, Hkv=32, S=2048, D=128, causal=True),
        # fp32 causal attention of a small decoder-only model
        dict(name="prefill_f32", kind="prefill", dtype="f32", B=8, H=12, Hkv=12, S=512, D=64, causal=True),
        # the attention block of one decode step of 32 sequences with grouped-query heads
        dict(name="decode_step_bf16", kind="decode_step", dtype="bf16", B=32, H=32, Hkv=8, D=128, S=4096, dModel=4096),
        # one sequence's token over its paged cache
        dict(name="paged_decode_bf16", kind="paged_decode", dtype="bf16", H=32, Hkv=8, D=128, block=16, S=8191),
        # a chunk of a long prompt after the part that is already in the paged cache
        dict(name="paged_prefill_bf16", kind="paged_prefill", dtype="bf16", H=32, Hkv=8, D=128, block=16, S=512, start=3584),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: mostly a multiple of 64, sometimes any number."""
    n = _log_int(rng, lo, hi)
    return n if rng.random() < 0.25 else max(64, n // 64 * 64)


def _rate(case):
    return 6e13 if case.get("dtype", "f32") in ("f32", "f16w") else 6e14


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 3e12, w["flops"] / _rate(case))


def _heads(rng):
    H = rng.choice([4, 8, 12, 16, 32])
    return H, H // rng.choice([g for g in (1, 2, 4, 8) if H % g == 0])


def _draw_once(rng):
    kind = rng.choice(["linear", "linear", "matmul", "matmul", "mha", "sdpa", "prefill", "decode_step", "paged_decode", "paged_prefill"])
    if kind in ("linear", "matmul"):
        c = dict(kind=kind, dtype=rng.choice(["f32", "f16", "bf16"]), M=_log_int(rng, 1, 8192), N=_width(rng, 64, 16384), K=_width(rng, 64, 16384))
        if kind == "linear":
            c["dtype"] = rng.choice(["f32", "f16", "bf16", "f16w"])
            c["act"] = rng.choice(["None", "ReLU", "GELU", "Swish"])
        elif rng.random() < 0.3:
            c.update(M=_log_int(rng, 1, 512), N=_log_int(rng, 30000, 60000), K=64 * _log_int(rng, 8, 64))
        return c
    if kind == "mha":
        H = rng.choice([4, 8, 12, 16])
        return dict(kind=kind, dtype=rng.choice(["f32", "f16", "bf16"]), B=_log_int(rng, 1, 16), S=_log_int(rng, 16, 1024), dModel=H * rng.choice([32, 64, 64, 128]),
                    H=H, padded=rng.random() < 0.5)
    if kind == "sdpa":
        H, Hkv = _heads(rng)
        S = _log_int(rng, 16, 1024)
        return dict(kind=kind, B=_log_int(rng, 1, 8), H=H, Hkv=Hkv, Sq=S, Sk=S if rng.random() < 0.6 else S + _log_int(rng, 1, 512),
                    D=rng.choice([32, 64, 64, 128]), causal=rng.random() < 0.5, padded=rng.random() < 0.4, softcap=rng.choice([0.0, 0.0, 30.0]),
                    weights=rng.random() < 0.6)
    if kind == "prefill":
        H, Hkv = _heads(rng)
        return dict(kind=kind, dtype=rng.choice(["f32", "f16", "bf16", "bf16"]), B=_log_int(rng, 1, 16), H=H, Hkv=Hkv, S=_log_int(rng, 16, 4096),
                    D=rng.choice([64, 80, 128, 128, 256]), causal=rng.random() < 0.75)
    if kind == "decode_step":
        H, Hkv = _heads(rng)
        D = rng.choice([64, 128])
        return dict(kind=kind, dtype=rng.choice(["f16", "bf16"]), B=_log_int(rng, 1, 64), H=H, Hkv=Hkv, D=D, S=_log_int(rng, 64, 8192), dModel=H * D)
    H, Hkv = _heads(rng)
    c = dict(kind=kind, dtype=rng.choice(["f32", "f16", "bf16", "bf16"]), H=H, Hkv=Hkv, D=rng.choice([64, 128]), block=rng.choice([16, 16, 32, 64]))
    if kind == "paged_decode":
        c["S"] = _log_int(rng, 64, 32768)
    else:
        c.update(S=_log_int(rng, 8, 2048), start=rng.choice([0, _log_int(rng, 16, 8192)]))
    return c


def draw(rng):
    limit = 0.5 * max(_cost(c) for c in listed())
    while True:
        c = _draw_once(rng)
        w = work(c)
        if _cost(c) <= limit and w["bytes"] < 6e8:
            return c


def _seen(Sq, Sk, causal):
    """Logits of one head: query i sees the keys up to i + Sk - Sq under the causal rule."""
    return Sq * (Sk - Sq) + Sq * (Sq + 1) // 2 if causal else Sq * Sk


def work(case):
    k = case["kind"]
    if k in ("linear", "matmul"):
        M, N, K = case["M"], case["N"], case["K"]
        ab, wb = (4, 2) if case["dtype"] == "f16w" else (_BYTES[case["dtype"]],) * 2
        return {"bytes": ab * (M * K + M * N) + wb * K * N + (4 * N if k == "linear" else 0), "flops": 2 * M * N * K}
    if k == "mha":
        B, S, dM, e = case["B"], case["S"], case["dModel"], _BYTES[case["dtype"]]
        return {"bytes": e * (2 * B * S * dM + 4 * dM * dM) + (B * S if case["padded"] else 0), "flops": 8 * B * S * dM * dM + 4 * B * S * S * dM}
    if k == "sdpa":
        B, H, Hkv, Sq, Sk, D = (case[n] for n in ("B", "H", "Hkv", "Sq", "Sk", "D"))
        return {"bytes": 4 * (2 * B * H * Sq * D + 2 * B * Hkv * Sk * D) + (4 * B * H * Sq * Sk if case["weights"] else 0) + (B * Sk if case["padded"] else 0),
                "flops": 4 * B * H * D * _seen(Sq, Sk, case["causal"])}
    if k == "prefill":
        B, H, Hkv, S, D = (case[n] for n in ("B", "H", "Hkv", "S", "D"))
        e = _BYTES[case["dtype"]]
        return {"bytes": B * H * S * D * (e + 4) + 2 * B * Hkv * S * D * e + 4 * B * H * S, "flops": 4 * B * H * D * _seen(S, S, case["causal"])}
    e, H, Hkv, D = _BYTES[case["dtype"]], case["H"], case["Hkv"], case["D"]
    if k == "decode_step":
        B, S, dM = case["B"], case["S"], case["dModel"]
        weights = dM * (2 * H + 2 * Hkv) * D
        return {"bytes": e * (weights + 2 * B * Hkv * S * D + 2 * B * dM + 2 * B * Hkv * D), "flops": 2 * B * weights + 4 * B * H * S * D}
    if k == "paged_decode":
        return {"bytes": e * (2 * Hkv * case["S"] * D + H * D) + 4 * H * D, "flops": 4 * H * case["S"] * D}
    keys = case["start"] + case["S"]
    return {"bytes": e * (2 * Hkv * keys * D + case["S"] * H * D) + 4 * case["S"] * H * D, "flops": 4 * H * D * _seen(case["S"], keys, True)}


def tolerance(case):
    """About four times the error measured against float64 (a hundred drawn cases): fp32 arithmetic 1.1e-6; one rounding to the storage
    type, of the result or of the probabilities, 2.1e-4 (fp16) and 1.7e-3 (bf16); a chain of such roundings 4.8e-4 and 4.0e-3."""
    kind, dtype = case["kind"], case.get("dtype", "f32")
    if dtype in ("f32", "f16w") or kind == "paged_decode":      # (paged decode: 16-bit cache, everything after the load in fp32)
        return {"rel": 4e-6}
    if kind in ("mha", "decode_step"):
        return {"rel": {"f16": 1.5e-3, "bf16": 1e-2}[dtype]}
    return {"rel": {"f16": 8e-4, "bf16": 7e-3}[dtype]}


def _padding_mask(gen, B, S):
    """Keep-mask [B, 1, 1, S] of sequences whose lengths lie between half of S and S."""
    lengths = torch.randint((S + 1) // 2, S + 1, (B,), device="cuda", generator=gen)
    return (torch.arange(S, device="cuda")[None, :] < lengths[:, None])[:, None, None, :]


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    k = case["kind"]
    storage = _TORCH.get(case.get("dtype", "f32"), torch.float32)
    state = {"case": case, "engine": _engine()}

    def randn(*shape, std=1.0, dtype=storage):
        return (std * torch.randn(*shape, device="cuda", generator=gen)).to(dtype)

    if k in ("linear", "matmul"):
        M, N, K = case["M"], case["N"], case["K"]
        state["x"] = randn(M, K)
        state["w"] = randn(K, N, std=1.0 / math.sqrt(K), dtype=torch.float16 if case["dtype"] == "f16w" else storage)
        if k == "linear":
            state["bias"] = randn(N, std=0.1, dtype=torch.float32)
        return state
    if k == "mha":
        B, S, dM = case["B"], case["S"], case["dModel"]
        state["x"] = randn(B, S, dM)
        for name in ("wq", "wk", "wv", "wo"):
            state[name] = randn(dM, dM, std=1.0 / math.sqrt(dM))
        state["mask"] = _padding_mask(gen, B, S) if case["padded"] else None
        return state
    if k == "sdpa":
        B, H, Hkv, Sq, Sk, D = (case[n] for n in ("B", "H", "Hkv", "Sq", "Sk", "D"))
        state["q"], state["k"], state["v"] = randn(B, H, Sq, D), randn(B, Hkv, Sk, D), randn(B, Hkv, Sk, D)
        state["mask"] = _padding_mask(gen, B, Sk) if case["padded"] else None
        return state
    H, Hkv, D, S = case["H"], case["Hkv"], case["D"], case["S"]
    if k == "prefill":
        B = case["B"]
        state["q"], state["k"], state["v"] = randn(B, H, S, D), randn(B, Hkv, S, D), randn(B, Hkv, S, D)
        return state
    if k == "decode_step":
        B, dM = case["B"], case["dModel"]
        std = 1.0 / math.sqrt(dM)
        state["x"] = randn(B, dM)
        state["wq"], state["wkv"], state["wo"] = randn(dM, H * D, std=std), randn(dM, 2 * Hkv * D, std=std), randn(H * D, dM, std=std)
        state["kcache"], state["vcache"] = randn(B, Hkv, S, D), randn(B, Hkv, S, D)
        angle = torch.arange(S, device="cuda", dtype=torch.float32)[:, None] * (10000.0 ** (-torch.arange(D // 2, device="cuda") * 2.0 / D))[None, :]
        state["cos"], state["sin"] = torch.cos(angle).contiguous(), torch.sin(angle).contiguous()
        # the activations of the step, kept across tokens
        for name, width in (("q", H * D), ("kv", 2 * Hkv * D), ("att", H * D), ("y", dM)):
            state[name] = torch.empty(B, width, device="cuda", dtype=storage)
        return state
    queries, start = (1, S - 1) if k == "paged_decode" else (S, case["start"])
    block = case["block"]
    blocks = (start + queries + block - 1) // block
    pool = blocks + blocks // 4 + 1                       # other sequences hold blocks of the pool too
    state["q"] = randn(queries, H, D)
    state["kpool"], state["vpool"] = randn(pool, block, Hkv, D), randn(pool, block, Hkv, D)
    state["table"] = torch.randperm(pool, device="cuda", generator=gen)[:blocks].to(torch.int32)
    return state


def run(state):
    case, eng = state["case"], state["engine"]
    be, W = eng.backend, eng.backend.WrapTensor
    k, kind = case["kind"], case.get("dtype", "f32")
    if k == "matmul":
        return eng.TensorMatMul(state["x"], state["w"])
    if k == "linear":
        layer = eng.FusedLinearFp16WeightB if kind == "f16w" else eng.FusedLinear
        return layer(state["x"], state["w"], state["bias"], case["act"])
    if k == "mha":
        return eng.MultiHeadAttentionForward(state["x"], state["wq"], state["wk"], state["wv"], state["wo"], case["H"], state["mask"])
    if k == "sdpa":
        out, weights = eng.ScaledDotProductAttention(state["q"], state["k"], state["v"], state["mask"], softcap=case["softcap"],
                                                     isCausal=case["causal"], returnWeights=case["weights"])
        return (out, weights) if case["weights"] else out
    if k == "prefill":
        return eng.FlashAttention(state["q"], state["k"], state["v"], isCausal=case["causal"])
    H, Hkv, D, S = case["H"], case["Hkv"], case["D"], case["S"]
    scale = 1.0 / math.sqrt(D)
    if k == "decode_step":
        B, dM = case["B"], case["dModel"]
        x, cos, sin, q, kv, att, y = (W(state[n]) for n in ("x", "cos", "sin", "q", "kv", "att", "y"))
        # Q, then [K | V] of which the K half is rotated; the row they add to the cache is the program's own copy
        be.GemmRope(kind, x, W(state["wq"]), q, B, H * D, dM, cos, sin, D, H * D, 1, S - 1)
        be.GemmRope(kind, x, W(state["wkv"]), kv, B, 2 * Hkv * D, dM, cos, sin, D, Hkv * D, 1, S - 1)
        be.DecodeAttention(kind, q, W(state["kcache"]), W(state["vcache"]), att, B, H, S, D, scale, numKVHeads=Hkv, outputIs16Bit=True)
        (be.Bf16Gemm if kind == "bf16" else be.Hgemm)(att, W(state["wo"]), y, B, dM, H * D)
        return state["q"], state["kv"], state["att"], state["y"]
    operands = tuple(W(state[n]) for n in ("q", "kpool", "vpool", "table"))
    if kind != "f32":
        queries, start = (1, S - 1) if k == "paged_decode" else (S, case["start"])
        out = be.PagedAttentionHalf(kind, *operands, H, Hkv, D, case["block"], queries, start, scale)
    elif k == "paged_decode":
        out = be.PagedAttentionDecodeGqa(*operands, H, Hkv, D, case["block"], S, scale)
    else:
        out = be.PagedAttentionPrefillGqa(*operands, H, Hkv, D, case["block"], S, case["start"], scale)
    return out.tensor
