"""What this framework is timed on: the W8A8 FP8 work of a served model, through the public entry points.

Six kinds of pass, each as a serving program makes it:

* ``linear``        one block-FP8 projection (``w8a8_block_fp8_linear``, what ``Fp8LinearMethod.apply`` calls for every
                    projection of a layer): group quant of the 16-bit activations, block-scaled GEMM, optional bias.
* ``linear_ue8m0``  the same projection in the power-of-two scale recipe: packed UE8M0 activation scales and a weight that was
                    requantised to power-of-two block scales at load time.
* ``linear_token``  one per-token / per-channel FP8 projection (``apply_fp8_linear``), optional bias.
* ``quant``         the group quantisation alone, as a fused producer or a cache writer calls it, in its scale layouts.
* ``moe``           one block-FP8 mixture-of-experts layer: the grouped sigmoid router, then the fused experts.
* ``mla``           one absorbed product of multi-head latent attention: per-tensor quant of the [heads, tokens, dim] view,
                    then the batched FP8 GEMM with the absorbed weight.

Sizes are those of BASELINE.json's configurations (DeepSeek-V3 and Llama-3-8B projections, the DeepSeek-V3 expert layer) and,
in ``draw``, the ranges around them: one token to a full prefill chunk, tensor-parallel shards of the projections and of the
experts, rows that are no multiple of anything.
"""
from __future__ import annotations

import math

import torch

from sglang_amd import fp8_kernel, fp8_utils, fused_moe, sgl_kernel

BLOCK = [128, 128]
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # a decode step of one request: latency and launches are all there is (gate_up shard at tensor parallel 8)
        {"name": "linear_decode_1", "kind": "linear", "m": 1, "n": 4608, "k": 7168, "dtype": "bf16", "bias": False},
        # a decode step of a small batch
        {"name": "linear_decode_32", "kind": "linear", "m": 32, "n": 4096, "k": 4096, "dtype": "bf16", "bias": False},
        # a decode step of a large batch, the attention output projection
        {"name": "linear_decode_128", "kind": "linear", "m": 128, "n": 7168, "k": 16384, "dtype": "bf16", "bias": False},
        # a ragged prefill chunk through a short-K projection of a float16 model whose projections have biases
        {"name": "linear_chunk_1000", "kind": "linear", "m": 1000, "n": 24576, "k": 1536, "dtype": "fp16", "bias": True},
        # a full prefill chunk, gate_up at tensor parallel 2: the headline of bench.py
        {"name": "linear_prefill_4096", "kind": "linear", "m": 4096, "n": 18432, "k": 7168, "dtype": "bf16", "bias": False},
        # a mid-sized prefill chunk with power-of-two scales (the recipe whose scales the matrix core applies)
        {"name": "ue8m0_prefill_2000", "kind": "linear_ue8m0", "m": 2000, "n": 7168, "k": 18432, "dtype": "bf16"},
        # a decode step of a per-channel quantised model (qkv)
        {"name": "token_decode_8", "kind": "linear_token", "m": 8, "n": 6144, "k": 4096, "dtype": "bf16", "bias": False,
         "per_channel": True},
        # a prefill chunk of it, gate_up, one scale for the whole weight, with bias
        {"name": "token_prefill_2048", "kind": "linear_token", "m": 2048, "n": 28672, "k": 4096, "dtype": "bf16", "bias": True,
         "per_channel": False},
        # the group quantisation of a long prefill on its own (largest)
        {"name": "quant_16384", "kind": "quant", "m": 16384, "k": 7168, "dtype": "bf16", "layout": "row"},
        # a decode batch through the expert layer: most experts are hit by a token or two
        {"name": "moe_decode_32", "kind": "moe", "m": 32, "experts": 256, "hidden": 7168, "inter": 2048, "topk": 8,
         "groups": 8, "topk_group": 4},
        # a prefill chunk through the expert layer: every expert works on some 128 rows
        {"name": "moe_prefill_4096", "kind": "moe", "m": 4096, "experts": 256, "hidden": 7168, "inter": 2048, "topk": 8,
         "groups": 8, "topk_group": 4},
        # decode attention: the query side of the absorbed product of all 128 heads
        {"name": "mla_decode_64", "kind": "mla", "m": 64, "heads": 128, "k": 128, "n": 512, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi, step=1):
    """Whole multiples of step between lo and hi, even over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear_ue8m0", "linear_token", "linear_token", "quant", "moe", "moe", "mla"])
    dtype = "fp16" if rng.random() < 0.25 else "bf16"
    if kind in ("linear", "linear_ue8m0", "linear_token"):
        n, k = _log_int(rng, 512, 28672, 64), _log_int(rng, 512, 18432, 128)
        # no more arithmetic than the full prefill chunk has
        most = max(1, min(8192 if kind == "linear_token" else 4096, 4096 * 18432 * 7168 // (n * k)))
        # the power-of-two recipe is a prefill one here: its kernels begin above a decode batch
        m = _log_int(rng, min(129 if kind == "linear_ue8m0" else 1, most), most)
        case = {"kind": kind, "m": m, "n": n, "k": k, "dtype": dtype}
        if kind != "linear_ue8m0":
            case["bias"] = rng.random() < 0.3
        if kind == "linear_token":
            case["per_channel"] = rng.random() < 0.5
        return case
    if kind == "quant":
        return {"kind": kind, "m": _log_int(rng, 1, 16384), "k": _log_int(rng, 512, 7168, 128), "dtype": dtype,
                "layout": rng.choice(["row", "column", "ue8m0"])}
    if kind == "moe":
        # the whole layer, an expert-parallel share of it, and tensor-parallel shards of the intermediate size
        return {"kind": kind, "m": _log_int(rng, 1, 4096), "experts": rng.choice([64, 128, 256]),
                "hidden": rng.choice([2048, 4096, 7168]), "inter": rng.choice([256, 512, 1024, 2048]), "topk": rng.choice([4, 6, 8]),
                "groups": 8, "topk_group": 4}
    k, n = rng.choice([(128, 512), (512, 128)])  # q_nope . w_kc, and attention output . w_vc
    return {"kind": kind, "m": _log_int(rng, 1, 512), "heads": rng.choice([16, 32, 64, 128]), "k": k, "n": n, "dtype": dtype}


# ---------------------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------------------


def _activation(gen, shape, dtype):
    """N(0, 1) with one value in a thousand fifty times as large: the outliers that group scales exist for."""
    x = torch.randn(shape, generator=gen, device="cuda")
    return torch.where(torch.rand(shape, generator=gen, device="cuda") < 1e-3, x * 50.0, x).to(dtype)


def _weight(gen, n, k):
    return torch.randn((n, k), generator=gen, device="cuda").mul_(0.02)


def _block_quant(w):
    """float32 [n, k] -> e4m3fn and one float32 scale per 128 x 128 block (blockamax / 448), as a checkpoint holds them."""
    n, k = w.shape
    nb, kb = (n + 127) // 128, (k + 127) // 128
    if (n, k) != (nb * 128, kb * 128):
        w = torch.nn.functional.pad(w, (0, kb * 128 - k, 0, nb * 128 - n))
    tiles = w.view(nb, 128, kb, 128)
    scale = tiles.abs().amax(dim=(1, 3)).clamp_(min=1e-12) / 448.0
    q = (tiles / scale[:, None, :, None]).clamp_(-448.0, 448.0).view(nb * 128, kb * 128)[:n, :k]
    return q.to(torch.float8_e4m3fn).contiguous(), scale


def _expert_weights(gen, experts, n, k):
    q = torch.empty((experts, n, k), device="cuda", dtype=torch.float8_e4m3fn)
    scale = torch.empty((experts, (n + 127) // 128, (k + 127) // 128), device="cuda")
    for e in range(experts):
        q[e], scale[e] = _block_quant(_weight(gen, n, k))
    return q, scale


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    kind, m = case["kind"], case["m"]
    state = {"kind": kind}
    if kind == "moe":
        e, hidden, inter = case["experts"], case["hidden"], case["inter"]
        state["x"] = torch.randn((m, hidden), generator=gen, device="cuda").to(torch.bfloat16)
        state["logits"] = torch.randn((m, e), generator=gen, device="cuda")
        state["gate_bias"] = torch.randn((e,), generator=gen, device="cuda").mul_(0.01)
        state["w13"], state["w13_scale"] = _expert_weights(gen, e, 2 * inter, hidden)
        state["w2"], state["w2_scale"] = _expert_weights(gen, e, hidden, inter)
        state["topk"], state["groups"], state["topk_group"] = case["topk"], case["groups"], case["topk_group"]
        return state
    dtype = DTYPES[case["dtype"]]
    k = case["k"]
    if kind == "quant":
        state["x"] = _activation(gen, (m, k), dtype)
        state["column"], state["ue8m0"] = case["layout"] != "row", case["layout"] == "ue8m0"
        return state
    n = case["n"]
    if kind == "mla":
        # attention keeps the tokens outermost; the products run per head
        state["x"] = torch.randn((m, case["heads"], k), generator=gen, device="cuda").to(dtype).transpose(0, 1)
        w = torch.randn((case["heads"], n, k), generator=gen, device="cuda").mul_(0.02)
        w, w_scale = fp8_utils.input_to_float8(w)
        state["w"], state["w_scale"], state["dtype"] = w.transpose(1, 2), w_scale, dtype
        return state
    state["x"] = _activation(gen, (m, k), dtype)
    state["bias"] = torch.randn((n,), generator=gen, device="cuda").to(dtype) if case.get("bias") else None
    w = _weight(gen, n, k)
    if kind == "linear":
        state["w"], state["w_scale"] = _block_quant(w)
    elif kind == "linear_ue8m0":
        state["w"], state["w_scale"] = fp8_utils.requant_weight_ue8m0(*_block_quant(w), BLOCK)
    else:
        amax = w.abs().amax(dim=1, keepdim=True) if case["per_channel"] else w.abs().amax().view(1, 1)
        scale = amax.clamp_(min=1e-12) / 448.0
        # the layer keeps the weight transposed: [k, n], column-major
        state["w"] = (w / scale).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn).t()
        state["w_scale"] = scale if case["per_channel"] else scale.view(1)
    return state


# ---------------------------------------------------------------------------------------------------------------------------
# the pass
# ---------------------------------------------------------------------------------------------------------------------------


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return fp8_utils.w8a8_block_fp8_linear(state["x"], state["w"], BLOCK, state["w_scale"], bias=state["bias"])
    if kind == "linear_ue8m0":
        x = state["x"]
        q, s = fp8_kernel.sglang_per_token_group_quant_fp8(x, 128, column_major_scales=True, scale_tma_aligned=True,
                                                           scale_ue8m0=True)
        return fp8_kernel.w8a8_block_fp8_matmul(q, state["w"], s, state["w_scale"], BLOCK, x.dtype)
    if kind == "linear_token":
        return fp8_utils.apply_fp8_linear(state["x"], state["w"], state["w_scale"], bias=state["bias"],
                                          use_per_token_if_dynamic=True)
    if kind == "quant":
        return fp8_kernel.sglang_per_token_group_quant_fp8(state["x"], 128, column_major_scales=state["column"],
                                                           scale_tma_aligned=state["ue8m0"], scale_ue8m0=state["ue8m0"])
    if kind == "moe":
        weights, ids = fused_moe.biased_grouped_topk(state["x"], state["logits"], state["gate_bias"], state["topk"], True,
                                                     state["groups"], state["topk_group"])
        return fused_moe.fused_experts(state["x"], state["w13"], state["w2"], weights, ids, use_fp8_w8a8=True,
                                       w1_scale=state["w13_scale"], w2_scale=state["w2_scale"], block_shape=BLOCK,
                                       routed_scaling_factor=2.5)
    x = state["x"]
    q, s = fp8_kernel.per_tensor_quant_mla_fp8(x, torch.zeros((1,), device=x.device, dtype=torch.float32))
    return sgl_kernel.bmm_fp8(q, state["w"], s, state["w_scale"], state["dtype"])


# ---------------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------------------


def work(case):
    kind, m = case["kind"], case["m"]
    if kind == "moe":
        e, hidden, inter, topk = case["experts"], case["hidden"], case["inter"], case["topk"]
        hit = e * (1.0 - (1.0 - topk / e) ** m)  # experts that some token picks, on average
        return {"bytes": hit * 3 * inter * hidden * (1 + 4 / 16384) + 2 * 2 * m * hidden + 4 * m * e + 4 * e,
                "flops": 2.0 * m * topk * 3 * inter * hidden}
    k = case["k"]
    if kind == "quant":
        scales = -(-k // 512) * 4 if case["layout"] == "ue8m0" else k // 128 * 4
        return {"bytes": m * (3 * k + scales), "flops": 0}
    n = case["n"]
    if kind == "mla":
        return {"bytes": case["heads"] * (2 * m * k + n * k + 2 * m * n), "flops": 2.0 * case["heads"] * m * n * k}
    bias = 2 * n if case.get("bias") else 0
    if kind == "linear_token":
        scales = 4 * (n if case["per_channel"] else 1)
    else:
        scales = 4 * -(-n // 128) * (k // 128)
    return {"bytes": 2 * m * k + n * k + 2 * m * n + scales + bias, "flops": 2.0 * m * n * k}


def tolerance(case):
    if case["kind"] == "quant":
        return "exact"  # bytes and scales are defined bit for bit
    # 16-bit results of float32 sums; the expert layer also rounds (and requantises) between its two products
    return {"rel": 1e-2 if case["kind"] == "moe" else 5e-3}
