"""The work that a serving engine has this package do, as cases to be timed.

A case is one step's worth of calls on one GPU: a linear layer or the projections of one
transformer layer in the forms the quantization methods call them, an expert layer, or the
activation quantization alone.  ``listed()`` holds the ordinary points of that range,
``draw()`` others of it.

Paths (``case["path"]``):

* ``block_fp8``    w8a8_block_fp8_linear: per-token-group FP8 quantization, block-scaled GEMM, bias
* ``block_ops``    the same linear as a drop-in user calls it: the quantization helper, then the
                   ``sgl_kernel`` GEMM operator
* ``ue8m0``        deepgemm_w8a8_block_fp8_linear_with_fallback with power-of-two scales
* ``fp8_token``    apply_fp8_linear: per-token FP8 quantization, per-channel weight scales
* ``int8_token``   apply_w8a8_int8_linear: per-token INT8 quantization, per-channel weight scales
* ``block_int8``   apply_w8a8_block_int8_linear
* ``experts``      cutlass_fused_experts_fp8: routing tables to weighted combine
* ``group_quant`` / ``token_quant_fp8`` / ``token_quant_int8``: activation quantization alone
"""

from __future__ import annotations

import math

import torch

from sglang_amd.moe.cutlass_moe import cutlass_fused_experts_fp8
from sglang_amd.quantization import fp8_utils
from sglang_amd.quantization.fp8_kernel import sglang_per_token_group_quant_fp8, sglang_per_token_quant_fp8
from sglang_amd.quantization.int8_kernel import per_token_quant_int8
from sglang_amd.quantization.int8_utils import apply_w8a8_block_int8_linear
from sglang_amd.quantization.w8a8_int8 import apply_w8a8_int8_linear
from sglang_amd.sgl_kernel import fp8_blockwise_scaled_mm

# a program whose checkpoints carry power-of-two scales sets this once; only the `ue8m0` path reads it
fp8_utils.DEEPGEMM_SCALE_UE8M0 = True

BLOCK = [128, 128]
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
BLOCK_PATHS = ("block_fp8", "block_ops", "ue8m0", "block_int8")
TOKEN_PATHS = ("fp8_token", "int8_token")
QUANT_PATHS = ("group_quant", "token_quant_fp8", "token_quant_int8")

# (N, K) of the projections of one layer
DEEPSEEK_V3 = "24576x1536,32768x512,7168x16384,4096x7168,2112x7168"
LLAMA_8B = "6144x4096,4096x4096,28672x4096,4096x14336"
LLAMA_70B = "10240x8192,8192x8192,57344x8192,8192x28672"


def _linear(name, path, rows, shapes, dtype="bf16", bias=False):
    return {"name": name, "path": path, "rows": rows, "shapes": shapes, "dtype": dtype, "bias": bias}


def listed():
    return [
        # one token through one narrow projection (DeepSeek-V3's fused q_a/kv_a): the smallest call there is
        _linear("block_fp8_1_token", "block_fp8", 1, "2112x7168"),
        # single-stream decode of a Llama-8B layer with per-token FP8 activations
        _linear("fp8_token_1_token_layer", "fp8_token", 1, LLAMA_8B),
        # batched decode on one INT8 projection with bias
        _linear("int8_token_16_rows_bias", "int8_token", 16, "14336x4096", bias=True),
        # batched decode of a Llama-70B layer through the block-FP8 linear
        _linear("block_fp8_64_rows_layer", "block_fp8", 64, LLAMA_70B),
        # a mixed batch (some prompts being prefilled among decodes) of no round size, called operator by operator
        _linear("block_ops_333_rows_fp16", "block_ops", 333, "4096x7168", dtype="fp16"),
        # a short prompt of ragged length on a block-INT8 checkpoint
        _linear("block_int8_1000_rows_bias", "block_int8", 1000, "5120x5120", bias=True),
        # chunked prefill of a Llama-8B layer
        _linear("fp8_token_2048_rows_layer", "fp8_token", 2048, LLAMA_8B),
        # chunked prefill of the DeepSeek-V3 projections: the benchmark's step
        _linear("block_fp8_4096_rows_layer", "block_fp8", 4096, DEEPSEEK_V3),
        # the largest: prefill of a Llama-70B layer whose scales are powers of two
        _linear("ue8m0_4096_rows_layer", "ue8m0", 4096, LLAMA_70B),
        # a decode batch through one rank's experts (DeepSeek-V3's expert shape, 32 local experts)
        {"name": "experts_16_tokens", "path": "experts", "rows": 16, "experts": 32, "topk": 8, "hidden": 7168, "inter": 2048, "dtype": "bf16"},
        # a prefill chunk of ragged length through the same experts
        {"name": "experts_2500_tokens", "path": "experts", "rows": 2500, "experts": 32, "topk": 8, "hidden": 7168, "inter": 2048, "dtype": "bf16"},
        # a long prompt's activations, quantized once for several GEMMs
        {"name": "group_quant_8192_rows", "path": "group_quant", "rows": 8192, "hidden": 7168, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi, multiple=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi // multiple, max(-(-lo // multiple), round(v / multiple)))) * multiple


def draw(rng):
    path = rng.choice(("block_fp8",) * 3 + ("fp8_token",) * 2 + ("int8_token",) * 2 + ("block_ops", "ue8m0", "block_int8", "experts", "experts", "quant"))
    rows = _log_int(rng, 1, 8192)
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16"))
    if path == "quant":
        return {"path": rng.choice(QUANT_PATHS), "rows": rows, "hidden": _log_int(rng, 512, 16384, 128), "dtype": dtype}
    if path == "experts":
        experts = _log_int(rng, 4, 64)
        hidden, inter = _log_int(rng, 1024, 7168, 128), _log_int(rng, 256, 2048, 128)
        return {"path": path, "rows": min(rows, 4096), "experts": experts, "topk": rng.randint(1, min(8, experts)), "hidden": hidden,
                "inter": inter, "dtype": dtype}
    # K of any multiple of the operators' 16 bytes is taken by the per-token linears; checkpoints mostly have multiples of 128
    n_step = 16 if rng.random() < 0.25 else 64
    k_step = 16 if path in TOKEN_PATHS and rng.random() < 0.15 else 128
    n, k = _log_int(rng, 512, 32768, n_step), _log_int(rng, 512, 16384, k_step)
    rows = max(1, min(rows, int(2e12 / (n * k))))
    if path == "ue8m0":
        dtype = "bf16"
    bias = path != "block_ops" and rng.random() < 0.3
    return {"path": path, "rows": rows, "shapes": "%dx%d" % (n, k), "dtype": dtype, "bias": bias}


def _shapes(case):
    return [tuple(int(v) for v in s.split("x")) for s in case["shapes"].split(",")]


# ---------------------------------------------------------------------------------------------
# inputs


def _activations(rows, hidden, dtype, gen):
    """N(0, 1) with 1 % of the values twenty times as large, as activations have them."""
    x = torch.randn((rows, hidden), generator=gen, device="cuda", dtype=torch.float32)
    outlier = torch.rand((rows, hidden), generator=gen, device="cuda") < 0.01
    return torch.where(outlier, x * 20.0, x).to(dtype)


def _gaussian(shape, gen):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * 0.02


def _block_quant(w, limit, code_dtype, power_of_two=False):
    """w [..., N, K] -> codes and scales [..., ceil(N/128), ceil(K/128)]: absmax / limit per 128 x 128 block."""
    n, k = w.shape[-2:]
    nb, kb = -(-n // 128), -(-k // 128)
    if n % 128 or k % 128:
        w = torch.nn.functional.pad(w, (0, kb * 128 - k, 0, nb * 128 - n))
    blocks = w.view(*w.shape[:-2], nb, 128, kb, 128)
    scale = blocks.abs().amax(dim=(-3, -1), keepdim=True).clamp_(min=1e-12) / limit
    if power_of_two:
        scale = torch.exp2(torch.ceil(torch.log2(scale)))
    q = blocks / scale
    q = q.round_().to(code_dtype) if code_dtype == torch.int8 else q.to(code_dtype)
    q = q.view(*w.shape)[..., :n, :k].contiguous()
    return q, scale.view(*w.shape[:-2], nb, kb).contiguous()


def _channel_quant(w, limit, code_dtype):
    scale = w.abs().amax(dim=-1, keepdim=True).clamp_(min=1e-12) / limit
    q = w / scale
    return (q.round_() if code_dtype == torch.int8 else q).to(code_dtype), scale


def _weight(path, n, k, gen):
    w = _gaussian((n, k), gen)
    if path in ("block_fp8", "block_ops"):
        return _block_quant(w, 448.0, torch.float8_e4m3fn)
    if path == "ue8m0":
        return _block_quant(w, 448.0, torch.float8_e4m3fn, power_of_two=True)
    if path == "block_int8":
        return _block_quant(w, 127.0, torch.int8)
    # the per-token methods keep the transposed view of the stored [N, K] weight after loading
    q, s = _channel_quant(w, 448.0 if path == "fp8_token" else 127.0, torch.float8_e4m3fn if path == "fp8_token" else torch.int8)
    return q.t(), s


def _prepare_experts(case, gen):
    e, topk, hidden, inter, rows = (case[k] for k in ("experts", "topk", "hidden", "inter", "rows"))
    w1q, w1s, w2q, w2s = [], [], [], []
    for _ in range(e):
        q, s = _block_quant(_gaussian((2 * inter, hidden), gen), 448.0, torch.float8_e4m3fn)
        w1q.append(q)
        w1s.append(s)
        q, s = _block_quant(_gaussian((hidden, inter), gen), 448.0, torch.float8_e4m3fn)
        w2q.append(q)
        w2s.append(s)
    # a router prefers some experts over others
    logits = torch.randn((rows, e), generator=gen, device="cuda") + 0.5 * torch.randn((1, e), generator=gen, device="cuda")
    weights, ids = torch.topk(torch.softmax(logits, dim=-1), topk, dim=-1)
    int64 = lambda: torch.empty((e,), dtype=torch.int64, device="cuda")  # noqa: E731
    strides = lambda v: torch.full((e,), v, dtype=torch.int64, device="cuda")  # noqa: E731
    sizes = lambda: torch.empty((e, 3), dtype=torch.int32, device="cuda")  # noqa: E731
    return {
        "path": "experts",
        "args": (
            _activations(rows, hidden, DTYPES[case["dtype"]], gen),
            torch.stack(w1q).transpose(1, 2), torch.stack(w2q).transpose(1, 2),
            torch.stack(w1s).transpose(1, 2), torch.stack(w2s).transpose(1, 2),
            weights / weights.sum(dim=-1, keepdim=True), ids.to(torch.int32),
            strides(hidden), strides(2 * inter), strides(inter), strides(hidden),
            torch.empty((7182 * 1024,), dtype=torch.uint8, device="cuda"),
            int64(), int64(), int64(), int64(), int64(),
            torch.empty((e + 1,), dtype=torch.int32, device="cuda"), sizes(), sizes(),
        ),
    }


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    path, rows = case["path"], case["rows"]
    if path == "experts":
        return _prepare_experts(case, gen)
    dtype = DTYPES[case["dtype"]]
    if path in QUANT_PATHS:
        return {"path": path, "x": _activations(rows, case["hidden"], dtype, gen)}
    inputs, layers = {}, []
    for n, k in _shapes(case):
        if k not in inputs:  # projections of the same width read the same activations
            inputs[k] = _activations(rows, k, dtype, gen)
        weight, scale = _weight(path, n, k, gen)
        bias = (torch.randn((n,), generator=gen, device="cuda") * 0.1).to(dtype) if case["bias"] else None
        layers.append((inputs[k], weight, scale, bias))
    return {"path": path, "layers": layers}


# ---------------------------------------------------------------------------------------------
# one pass


def run(state):
    path = state["path"]
    if path == "block_fp8":
        return [fp8_utils.w8a8_block_fp8_linear(x, w, BLOCK, s, bias=b) for x, w, s, b in state["layers"]]
    if path == "block_ops":
        outs = []
        for x, w, s, _ in state["layers"]:
            q, xs = sglang_per_token_group_quant_fp8(x, 128, column_major_scales=True)
            outs.append(fp8_blockwise_scaled_mm(q, w.t(), xs, s.t(), x.dtype))
        return outs
    if path == "ue8m0":
        return [fp8_utils.deepgemm_w8a8_block_fp8_linear_with_fallback(x, w, BLOCK, s, bias=b) for x, w, s, b in state["layers"]]
    if path == "fp8_token":
        return [fp8_utils.apply_fp8_linear(x, w, s, bias=b) for x, w, s, b in state["layers"]]
    if path == "int8_token":
        return [apply_w8a8_int8_linear(x, w, s, b) for x, w, s, b in state["layers"]]
    if path == "block_int8":
        return [apply_w8a8_block_int8_linear(x, w, BLOCK, s, bias=b) for x, w, s, b in state["layers"]]
    if path == "experts":
        return cutlass_fused_experts_fp8(*state["args"])
    if path == "group_quant":
        return sglang_per_token_group_quant_fp8(state["x"], 128, column_major_scales=True)
    if path == "token_quant_fp8":
        return sglang_per_token_quant_fp8(state["x"])
    if path == "token_quant_int8":
        return per_token_quant_int8(state["x"])
    raise ValueError(path)


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without, and how close another implementation comes


def work(case):
    path, m = case["path"], case["rows"]
    if path in QUANT_PATHS:
        scales = case["hidden"] // 128 if path == "group_quant" else 1
        return {"bytes": m * (3 * case["hidden"] + 4 * scales), "flops": 0}
    if path == "experts":
        e, topk, hidden, inter = (case[k] for k in ("experts", "topk", "hidden", "inter"))
        hit = e * (1.0 - (1.0 - topk / e) ** m)  # experts that some token is routed to, on average
        per_expert = 3 * hidden * inter + 4 * (3 * hidden * inter // 16384)
        return {"bytes": hit * per_expert + 4 * m * hidden + 8 * m * topk, "flops": 6 * m * topk * hidden * inter}
    total = {"bytes": 0, "flops": 0}
    widths = set()
    for n, k in _shapes(case):
        scales = 4 * (-(-n // 128)) * (-(-k // 128)) if path in BLOCK_PATHS else 4 * n
        total["bytes"] += n * k + scales + 2 * m * n + (2 * n if case["bias"] else 0) + (0 if k in widths else 2 * m * k)
        total["flops"] += 2 * m * n * k
        widths.add(k)
    return total


def tolerance(case):
    path = case["path"]
    if path in QUANT_PATHS:
        return "exact"
    if path == "experts":
        # a 16-bit intermediate on the other side of a rounding boundary moves one FP8 code of the second GEMM's input
        return {"rel": 1e-2, "max": 0.15}
    # sums of exact products in fp32 (int32), rounded once (twice with bias) to the 16-bit output
    return {"rel": 5e-3 if case["dtype"] == "bf16" else 1e-3, "max": 2e-2 if case["dtype"] == "bf16" else 4e-3}
