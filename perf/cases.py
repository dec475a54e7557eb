"""Performance cases of the FP8 linear path: what a model's layers ask of this package, through its public entry
points, from one decoded token to a prefill of thousands.

A case is a dict of plain values.  `listed()` gives the named cases, `draw(rng)` one more of the same ranges,
`prepare(case, seed)` what a program holds before the call (weights, quantisation config, inputs, paged cache),
`run(state)` one pass, `work(case)` the bytes and operations a pass cannot do without, `tolerance(case)` how far two
correct results may be apart.

The kinds:
  linear   `Linear` on bf16 activations: dynamic quantisation and the scaled matmul; scaling "block" (1 x 128 groups
           against 128 x 128 weight blocks), "row" (per token x per channel) or "static" (per tensor, offline scales)
  norm     RMSNorm fused with the per-token quantisation, then the per-channel scaled matmul
  mlp      the gated feed-forward block
  qkv      the fused QKV projection of a ragged batch that stores K and V into the paged cache
  mla      the batched matmul of latent attention (one small weight per head) with its quantiser
  moe      the expert matmuls of a mixture-of-experts layer
"""
from __future__ import annotations

import math

import torch

import modular_amd as mx
from modular_amd import synth

# (K, N) of the linears the benchmark configurations name: Llama-3.1-8B (qkv, o_proj, gate_up, down), DeepSeek-V3
# attention (q_a, q_b, kv_a, kv_b, o_proj, q_a + kv_a stacked), Llama-3.1-70B (qkv, gate_up, down)
LINEARS = [(4096, 6144), (4096, 4096), (4096, 28672), (14336, 4096),
           (7168, 1536), (1536, 24576), (7168, 576), (512, 32768), (16384, 7168), (7168, 2112),
           (8192, 10240), (8192, 57344), (28672, 8192)]
MLPS = [(4096, 14336), (7168, 18432), (8192, 28672)]   # hidden, feed-forward
QKVS = [(4096, 32, 8), (8192, 64, 8), (5120, 40, 8)]   # hidden, query heads, K / V heads (of 128)
# tokens x weight elements of the largest listed dense case: no drawn one does more
MOST_WORK = 4096 * 16384 * 7168


def listed() -> list[dict]:
    return [
        # one sequence decoding, the attention output projection of an 8B model: launch and host latency
        {"name": "linear_block_m1", "kind": "linear", "scaling": "block", "M": 1, "K": 4096, "N": 4096},
        # 70B decode of a few sequences behind the layer's norm: the weight stream (470 MB)
        {"name": "norm_row_m8", "kind": "norm", "M": 8, "K": 8192, "N": 57344},
        # a serving batch in decode, odd size: between the weight stream and the matrix pipe
        {"name": "linear_block_m117", "kind": "linear", "scaling": "block", "M": 117, "K": 4096, "N": 6144},
        # checkpoint with static per-tensor scales, a ragged prefill chunk
        {"name": "linear_static_m1777", "kind": "linear", "scaling": "static", "M": 1777, "K": 4096, "N": 6144},
        # a full prefill batch on the largest attention projection: the matrix pipe
        {"name": "linear_block_m4096", "kind": "linear", "scaling": "block", "M": 4096, "K": 16384, "N": 7168},
        # the feed-forward block of an 8B model, decode batch and prefill batch
        {"name": "mlp_block_m16", "kind": "mlp", "scaling": "block", "M": 16, "hidden": 4096, "inter": 14336},
        {"name": "mlp_block_m2048", "kind": "mlp", "scaling": "block", "M": 2048, "hidden": 4096, "inter": 14336},
        # fused QKV: 64 sequences decode one token each (70B, per channel); a ragged prefill of 5 prompts (8B, block)
        {"name": "qkv_row_decode64", "kind": "qkv", "scaling": "row", "batch": 64, "tokens": 64, "cached": 1500,
         "hidden": 8192, "heads": 64, "kv_heads": 8},
        {"name": "qkv_block_prefill5", "kind": "qkv", "scaling": "block", "batch": 5, "tokens": 2011, "cached": 0,
         "hidden": 4096, "heads": 32, "kv_heads": 8},
        # latent attention in decode: 128 heads absorb 48 tokens' queries into the 512-wide latent space
        {"name": "mla_decode48", "kind": "mla", "M": 48, "K": 128, "N": 512, "heads": 128},
        # the experts of a 256-expert layer: a decode batch (the weights of the experts in use stream by), a prefill
        {"name": "moe_decode64", "kind": "moe", "tokens": 64, "experts": 256, "top_k": 8, "hidden": 7168, "inter": 2048,
         "host_sync": False},
        {"name": "moe_prefill4096", "kind": "moe", "tokens": 4096, "experts": 256, "top_k": 8, "hidden": 7168, "inter": 2048,
         "host_sync": True},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    kind = rng.choice(["linear", "linear", "linear", "norm", "mlp", "qkv", "mla", "moe"])
    if kind in ("linear", "norm"):
        if rng.random() < 0.6:
            K, N = rng.choice(LINEARS)
        else:
            K, N = 128 * _log_int(rng, 4, 128), 16 * _log_int(rng, 32, 1792)
        M = _log_int(rng, 1, min(4096, MOST_WORK // (K * N)))
        case = {"kind": kind, "M": M, "K": K, "N": N}
        if kind == "linear":
            case["scaling"] = rng.choice(["block", "block", "row", "static"])
        return case
    if kind == "mlp":
        hidden, inter = rng.choice(MLPS)
        return {"kind": kind, "scaling": rng.choice(["block", "row"]), "hidden": hidden, "inter": inter,
                "M": _log_int(rng, 1, min(2048, MOST_WORK // (3 * hidden * inter)))}
    if kind == "qkv":
        hidden, heads, kv_heads = rng.choice(QKVS)
        batch = _log_int(rng, 1, 128)
        decode = rng.random() < 0.5
        tokens = batch if decode else max(batch, _log_int(rng, 64, 4096))
        return {"kind": kind, "scaling": rng.choice(["block", "row"]), "batch": batch, "tokens": tokens,
                "cached": rng.randrange(1, 2048) if decode else 0, "hidden": hidden, "heads": heads, "kv_heads": kv_heads}
    if kind == "mla":
        K, N = rng.choice([(128, 512), (512, 128)])
        return {"kind": kind, "M": _log_int(rng, 1, 1024), "K": K, "N": N, "heads": rng.choice([16, 64, 128])}
    hidden, inter, experts, top_k = rng.choice([(7168, 2048, 256, 8), (4096, 1536, 128, 8), (2048, 1408, 64, 6)])
    return {"kind": kind, "tokens": _log_int(rng, 1, 4096), "experts": experts, "top_k": top_k, "hidden": hidden,
            "inter": inter, "host_sync": rng.random() < 0.5}


# ---- inputs -----------------------------------------------------------------------------------------------------------

def _config(scaling: str) -> mx.QuantConfig:
    if scaling == "block":
        return mx.blockwise_fp8_config()
    if scaling == "row":
        return mx.rowwise_fp8_config()
    return mx.QuantConfig(
        input_scale=mx.InputScaleSpec(mx.ScaleGranularity.TENSOR, mx.ScaleOrigin.STATIC, torch.float32),
        weight_scale=mx.WeightScaleSpec(mx.ScaleGranularity.TENSOR, torch.float32),
        format=mx.QuantFormat.COMPRESSED_TENSORS_FP8)


def _weight(N: int, K: int, scaling: str, seed: int):
    w = synth.weights_f32(N, K, seed=seed, device="cuda")
    if scaling == "block":
        return synth.quantize_weight_block(w)
    if scaling == "row":
        return synth.quantize_weight_rowwise(w)
    scale = w.abs().amax() / synth.FP8_MAX
    return (w / scale).to(torch.float8_e4m3fn), scale.cpu()


def _experts(experts: int, N: int, K: int, seed: int):
    """[E, N, K] weights with their block scales, sixteen experts at a time."""
    w = torch.empty((experts, N, K), dtype=torch.float8_e4m3fn, device="cuda")
    s = torch.empty((experts, -(-N // 128), -(-K // 128)), dtype=torch.float32, device="cuda")
    for e in range(0, experts, 16):
        n = min(16, experts - e)
        w[e:e + n], s[e:e + n] = synth.quantize_weight_block(
            synth.weights_f32(n * N, K, seed=seed + e, device="cuda").reshape(n, N, K))
    return w, s


def _routing(case: dict, seed: int) -> torch.Tensor:
    """[tokens, top_k] expert ids, a few experts much more popular than the rest (rank^-1.1)."""
    g = torch.Generator().manual_seed(seed)
    rank = torch.empty(case["experts"])
    rank[torch.randperm(case["experts"], generator=g)] = torch.arange(1, case["experts"] + 1, dtype=torch.float32)
    logits = torch.randn((case["tokens"], case["experts"]), generator=g) - 1.1 * torch.log(rank)
    return logits.topk(case["top_k"], dim=1).indices.to(torch.int32)


def _prompt_lengths(case: dict, seed: int) -> list[int]:
    """`tokens` shared out over `batch` sequences, every one at least one token, uneven where there is room."""
    batch, tokens = case["batch"], case["tokens"]
    share = torch.rand(batch, generator=torch.Generator().manual_seed(seed)) + 0.2
    lens = (1 + (tokens - batch) * share / share.sum()).to(torch.int64).tolist()
    lens[-1] += tokens - sum(lens)
    return lens


def prepare(case: dict, seed: int) -> dict:
    kind, base = case["kind"], 1000 * seed
    state = {"case": case}
    if kind in ("linear", "norm"):
        M, K, N = case["M"], case["K"], case["N"]
        scaling = case.get("scaling", "row")
        cfg = _config(scaling)
        state["x"] = synth.activations(M, K, seed=base, device="cuda")
        w, ws = _weight(N, K, scaling, base + 1)
        if kind == "norm":
            g = torch.Generator().manual_seed(base + 2)
            gamma = (1.0 + 0.1 * torch.randn(K, generator=g)).to(torch.bfloat16).cuda()
            state.update(cfg=cfg, w=w, ws=ws, gamma=gamma)
            return state
        layer = mx.Linear(K, N, cfg, device="cuda")
        layer.load_state_dict({"weight": w, "weight_scale": ws} | (
            {"input_scale": torch.tensor(float(state["x"].abs().max()) / synth.FP8_MAX)} if scaling == "static" else {}))
        state["layer"] = layer
    elif kind == "mlp":
        H, F = case["hidden"], case["inter"]
        state["x"] = synth.activations(case["M"], H, seed=base, device="cuda")
        layer = mx.MLP(H, F, _config(case["scaling"]), device="cuda")
        weights = {}
        for i, (name, n, k) in enumerate((("gate_proj", F, H), ("up_proj", F, H), ("down_proj", H, F))):
            weights[name + ".weight"], weights[name + ".weight_scale"] = _weight(n, k, case["scaling"], base + 1 + i)
        layer.load_state_dict(weights)
        state["layer"] = layer
    elif kind == "qkv":
        page, head = 128, 128
        lens = _prompt_lengths(case, base)
        pages = [-(-(case["cached"] + n) // page) for n in lens]
        kv = mx.KVCacheParams(torch.bfloat16, case["kv_heads"], head, num_layers=2, page_size=page)
        blocks = torch.zeros(kv.blocks_shape(sum(pages) + 3), dtype=torch.bfloat16, device="cuda")
        order = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(base + 3)).tolist()
        table, at = torch.zeros((len(lens), max(pages)), dtype=torch.int32), 0
        for b, n in enumerate(pages):
            table[b, :n] = torch.tensor(order[at:at + n], dtype=torch.int32)
            at += n
        offsets = torch.zeros(len(lens) + 1, dtype=torch.int32)
        offsets[1:] = torch.cumsum(torch.tensor(lens), 0)
        N = (case["heads"] + 2 * case["kv_heads"]) * head
        w, ws = _weight(N, case["hidden"], case["scaling"], base + 1)
        state.update(kv=kv, w=w, ws=ws, cfg=_config(case["scaling"]), offsets=offsets.cuda(),
                     x=synth.activations(case["tokens"], case["hidden"], seed=base, device="cuda"),
                     cache=mx.PagedCacheValues(blocks, torch.full((len(lens),), case["cached"], dtype=torch.int32).cuda(),
                                               table.cuda()))
    elif kind == "mla":
        B, M, K, N = case["heads"], case["M"], case["K"], case["N"]
        # activations as the attention graph holds them: [token, head, channel], read as [head, token, channel]
        state["x"] = synth.activations(M, B * K, seed=base, device="cuda").reshape(M, B, K).transpose(0, 1)
        state["w"], state["ws"] = synth.quantize_weight_block(
            synth.weights_f32(B * N, K, seed=base + 1, device="cuda").reshape(B, N, K))
        state["cfg"] = _config("block")
    else:
        E, H, F = case["experts"], case["hidden"], case["inter"]
        state["x"] = synth.activations(case["tokens"], H, seed=base, device="cuda")
        state["router"] = _routing(case, base).cuda()
        state["gate_up"], state["gate_up_scales"] = _experts(E, 2 * F, H, base + 1)
        state["down"], state["down_scales"] = _experts(E, H, F, base + 501)
        state["cfg"] = _config("block")
    return state


# ---- one pass ---------------------------------------------------------------------------------------------------------

def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind in ("linear", "mlp"):
        return state["layer"](state["x"])
    cfg = state["cfg"]
    if kind == "norm":
        q, scales = mx.rms_norm_fused_quantize_dynamic_scaled_fp8(state["x"], state["gamma"], 1e-5)
        return mx.dynamic_scaled_matmul(q, state["w"], scales, state["ws"], cfg.input_scale, cfg.weight_scale)
    if kind == "qkv":
        q = mx.quantized_fused_qkv_matmul(state["kv"], state["x"], state["w"], state["cache"], 1, state["offsets"],
                                          case["heads"], cfg, state["ws"])
        return q, state["cache"].kv_blocks
    if kind == "mla":
        q, scales = mx.batched_quantize_dynamic_scaled_fp8(state["x"], 128)
        return mx.batched_dynamic_scaled_fp8_matmul(q, state["w"], scales, state["ws"], cfg.input_scale, cfg.weight_scale)
    return mx.expert_matmuls_fp8(state["x"], state["router"], state["gate_up"], state["gate_up_scales"], state["down"],
                                 state["down_scales"], cfg, host_sync=case["host_sync"])


# ---- what a pass cannot do without ------------------------------------------------------------------------------------

def _scale_bytes(N: int, K: int, scaling: str) -> int:
    return 4 * (-(-N // 128)) * (-(-K // 128)) if scaling == "block" else 4 * N if scaling == "row" else 4


def work(case: dict) -> dict:
    """bf16 activations in and results out once, the fp8 weights (of the experts in use) with their scales once."""
    kind = case["kind"]
    if kind in ("linear", "norm", "qkv"):
        scaling = case.get("scaling", "row")
        if kind == "qkv":
            M, K, N = case["tokens"], case["hidden"], 128 * (case["heads"] + 2 * case["kv_heads"])
        else:
            M, K, N = case["M"], case["K"], case["N"]
        return {"flops": 2 * M * N * K, "bytes": N * K + _scale_bytes(N, K, scaling) + 2 * M * (K + N)}
    if kind == "mlp":
        M, H, F = case["M"], case["hidden"], case["inter"]
        scales = _scale_bytes(2 * F, H, case["scaling"]) + _scale_bytes(H, F, case["scaling"])
        return {"flops": 6 * M * H * F, "bytes": 3 * H * F + scales + 4 * M * H}
    if kind == "mla":
        B, M, K, N = case["heads"], case["M"], case["K"], case["N"]
        return {"flops": 2 * B * M * N * K, "bytes": B * (N * K + _scale_bytes(N, K, "block") + 2 * M * (K + N))}
    T, H, F, k = case["tokens"], case["hidden"], case["inter"], case["top_k"]
    used = int(_routing(case, 0).unique().numel())
    expert = 3 * H * F + _scale_bytes(2 * F, H, "block") + _scale_bytes(H, F, "block")
    return {"flops": 6 * T * k * H * F, "bytes": used * expert + 2 * T * H + 4 * T * k + 2 * T * k * H}


def tolerance(case: dict) -> dict:
    """Four times what each path shows against the same steps with the matmuls' sums in 64 bits.  The results are bf16
    (8 bits) of float32 sums of exact fp8 products, which the matrix pipe truncates some 13 bits below the largest:
    other sums flip a share of the last bits (4e-4 of the norm, one bf16 step at most)."""
    if case["kind"] in ("mlp", "moe"):
        # a flipped bit of the intermediate result moves fp8 codes (3 bits) of the second matmul's input: 3e-3
        return {"rel": 1.2e-2}
    if case["kind"] == "qkv" and case["scaling"] == "row":
        # this op rounds the sum, each scale and their products to bf16 on the way: 4e-3, two steps
        return {"rel": 1.6e-2, "max": 6.4e-2}
    return {"rel": 1.6e-3, "max": 3.2e-2}
