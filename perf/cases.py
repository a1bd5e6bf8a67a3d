"""The work that programs built on this package have it do, as cases that a timing harness can run.

listed() are the cases that are followed, draw() gives further ones of the same kinds and ranges, prepare() makes what a
program holds before the call, run() is one pass through the public entry points, work() what a pass cannot do without
and tolerance() how far two correct implementations of the same precision may lie apart.

Kinds:
  linear       serving with the official operators: act_quant of the activations, fp8_gemm against a quantized weight
  deep_infer   serving with DeepLinear: no gradients, the quantized weight kept between calls, bias
  mlp_infer    serving with Fp8MLP on DeepLinear projections: no gradients, quantized weights kept
  dequant      a quantized weight expanded to bf16 (checkpoint conversion, bf16 fallbacks)
  deep_train   one training step of a DeepLinear layer with bias: output and the gradients of input, weight and bias
  fp8_train    the same for Fp8Linear (the official dialect, either fp8 format)
  mlp_train    one training step of Fp8MLP, memory-saving or not, either dialect and format
  moe_decode   routed experts while decoding: a few tokens per expert, per-token cast and grouped GEMM
  moe_train    one training step of a grouped linear layer from the Megatron operators: padding, both grouped casts, the
               weights' block casts of a first micro-batch, grouped GEMMs forward and for the input gradient, one
               row-scaled GEMM per expert for the weight gradients
"""
import math
import random

import torch

import mdy_triton_amd as m
from mdy_triton_amd import fp8_kernel
from mdy_triton_amd.megatron_patchs.dpsk_grouped_linear import Fp8Padding, Fp8Unpadding
from mdy_triton_amd.megatron_patchs.manger import CustomManger

DEVICE = "cuda"
FORMATS = {"e4m3fn": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
# what a drawn case may take: no more than the largest listed one
MAX_FLOPS = 1.1e12
MAX_BYTES = 1.1e9


def listed():
    return [
        # one token through a routed expert's down projection: the smallest call, launches and host work count
        {"name": "decode_1", "kind": "linear", "M": 1, "N": 7168, "K": 2048},
        # sixteen sequences decoding through a routed expert's up projection: a long K against few columns
        {"name": "decode_16", "kind": "linear", "M": 16, "N": 2048, "K": 7168},
        # a serving batch through a biased layer whose quantized weight is kept
        {"name": "serve_deep_64", "kind": "deep_infer", "M": 64, "N": 7168, "K": 2048},
        # a small batch through a whole SwiGLU MLP (shared-expert size) with kept quantized weights; 200 tokens: ragged
        {"name": "serve_mlp_200", "kind": "mlp_infer", "M": 200, "H": 7168, "I": 2048},
        # the remainder chunk of a chunked prefill through the fused q_a / kv_a projection: odd tokens, ragged columns
        {"name": "prefill_777", "kind": "linear", "M": 777, "N": 2112, "K": 7168},
        # prefill of 4096 tokens through the dense MLP's up/gate projection: the largest GEMM
        {"name": "prefill_4096", "kind": "linear", "M": 4096, "N": 18432, "K": 7168},
        # the dense MLP's down projection expanded to bf16
        {"name": "dequant_down", "kind": "dequant", "N": 7168, "K": 18432},
        # training step of a square layer, DeepLinear dialect, bias
        {"name": "train_deep", "kind": "deep_train", "M": 8192, "N": 4096, "K": 4096},
        # the same layer in the official dialect with its default format
        {"name": "train_fp8_e5m2", "kind": "fp8_train", "M": 8192, "N": 4096, "K": 4096, "format": "e5m2"},
        # memory-saving training step of a SwiGLU MLP, official dialect, e4m3fn
        {"name": "train_mlp", "kind": "mlp_train", "M": 4096, "H": 7168, "I": 2048, "dialect": "official",
         "format": "e4m3fn", "low_memory": True},
        # decoding: 32 routed experts with one to seventeen tokens each, weights streamed
        {"name": "moe_decode_32", "kind": "moe_decode", "experts": 32, "tokens": 270, "N": 4096, "K": 7168, "routing": 1},
        # training: 8 routed experts with about 500 tokens each, ragged
        {"name": "moe_train_8", "kind": "moe_train", "experts": 8, "tokens": 4000, "N": 4096, "K": 7168, "routing": 2},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi, step):
    """A size from lo to hi, spread over its logarithm, in multiples of step."""
    return min(hi, max(lo, int(round(_log_uniform(rng, lo, hi) / step)) * step))


def _rows(rng, lo, hi):
    return min(hi, max(lo, int(_log_uniform(rng, lo, hi + 1))))


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return case


def _draw(rng):
    kind = rng.choice(["linear", "linear", "deep_infer", "mlp_infer", "dequant", "deep_train", "fp8_train", "mlp_train",
                       "moe_decode", "moe_train"])
    if kind == "linear":
        # columns mostly in multiples of 64, one weight in four with a ragged last block
        return {"kind": kind, "M": _rows(rng, 1, 4096), "N": _size(rng, 512, 18432, rng.choice([64, 64, 64, 8])),
                "K": _size(rng, 512, 18432, 128)}
    if kind == "deep_infer":
        return {"kind": kind, "M": _rows(rng, 1, 1024), "N": _size(rng, 512, 18432, 64), "K": _size(rng, 512, 7168, 64)}
    if kind == "mlp_infer":
        return {"kind": kind, "M": _rows(rng, 1, 2048), "H": _size(rng, 1024, 7168, 128), "I": _size(rng, 512, 8192, 128)}
    if kind == "dequant":
        return {"kind": kind, "N": _size(rng, 512, 18432, rng.choice([64, 1])), "K": _size(rng, 512, 18432, 64)}
    if kind == "deep_train":
        return {"kind": kind, "M": _rows(rng, 256, 16384), "N": _size(rng, 512, 8192, 64), "K": _size(rng, 512, 8192, 64)}
    if kind == "fp8_train":
        return {"kind": kind, "M": _rows(rng, 256, 16384), "N": _size(rng, 512, 8192, 128), "K": _size(rng, 512, 8192, 128),
                "format": rng.choice(["e4m3fn", "e5m2"])}
    if kind == "mlp_train":
        dialect = rng.choice(["official", "deeplinear"])
        return {"kind": kind, "M": _rows(rng, 256, 8192), "H": _size(rng, 1024, 7168, 128), "I": _size(rng, 512, 4096, 128),
                "dialect": dialect, "format": "e4m3fn" if dialect == "deeplinear" else rng.choice(["e4m3fn", "e5m2"]),
                "low_memory": rng.choice([True, False])}
    experts = rng.choice([4, 8, 16, 32] if kind == "moe_train" else [8, 16, 32, 64])
    N, K = _size(rng, 512, 4096, 128), _size(rng, 1024, 7168, 128)
    per_expert = _log_uniform(rng, 100, 1000) if kind == "moe_train" else _log_uniform(rng, 1.5, 40)
    if kind == "moe_train":      # the grouped cast with transposed copies takes multiples of 256
        N, K = (N + 255) // 256 * 256, (K + 255) // 256 * 256
    return {"kind": kind, "experts": experts, "tokens": max(1, int(experts * per_expert)), "N": N, "K": K,
            "routing": rng.randrange(1 << 30)}


def _splits(case):
    """Tokens of every expert: a fixed total, shares between a tenth and twice the mean."""
    rng = random.Random(case["routing"])
    share = [rng.uniform(0.1, 1.9) for _ in range(case["experts"])]
    edges, total = [0], 0.0
    for v in share:
        total += v
        edges.append(int(round(case["tokens"] * total / sum(share))))
    return [b - a for a, b in zip(edges, edges[1:])]


class _Source:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device=DEVICE, dtype=torch.float32)

    def activations(self, M, K):
        """N(0, 1) with one value in a hundred ten times as large: the outlier channels that block scales are for."""
        x = self.normal(M, K)
        big = torch.rand(M, K, generator=self.g, device=DEVICE) < 0.01
        return torch.where(big, x * 10, x).bfloat16()

    def weight(self, N, K):
        return self.normal(N, K).mul_(0.02).bfloat16()

    def gradient(self, M, N):
        return self.normal(M, N).mul_(1e-2).bfloat16()


def _set(layer_weight, value):
    with torch.no_grad():
        layer_weight.copy_(value)


def prepare(case, seed):
    src = _Source(seed)
    kind = case["kind"]
    st = {"case": case}
    if kind in ("linear", "dequant"):
        # the checkpoint format: e4m3fn bytes with one fp32 scale per 128x128 block, ragged last blocks allowed
        N, K = case["N"], case["K"]
        NB = -(-N // 128)
        wq, ws = m.weight_quant_block(src.weight(NB * 128, K if K % 128 == 0 else -(-K // 128) * 128), dtype=torch.float8_e4m3fn)
        st["w"], st["ws"] = wq.view(torch.uint8)[:N, :K].contiguous().view(torch.float8_e4m3fn), ws
        if kind == "linear":
            st["x"] = src.activations(case["M"], K)
    elif kind in ("deep_infer", "deep_train"):
        M, N, K = case["M"], case["N"], case["K"]
        lin = m.DeepLinear(K, N, bias=True, device=DEVICE, dtype=torch.bfloat16)
        _set(lin.weight, src.weight(N, K))
        _set(lin.bias, src.normal(N))
        st["layer"], st["x"] = lin, src.activations(M, K)
        if kind == "deep_infer":
            lin.cache_weight = True
            with torch.no_grad():
                lin(st["x"][:1])
        else:
            st["x"].requires_grad_(True)
            st["dy"] = src.gradient(M, N)
    elif kind == "fp8_train":
        M, N, K = case["M"], case["N"], case["K"]
        lin = m.Fp8Linear(K, N, bias=True, device=DEVICE, dtype=torch.bfloat16, fp8_dtype=FORMATS[case["format"]])
        _set(lin.weight, src.weight(N, K))
        _set(lin.bias, src.normal(N))
        st["layer"], st["x"], st["dy"] = lin, src.activations(M, K).requires_grad_(True), src.gradient(M, N)
    elif kind in ("mlp_infer", "mlp_train"):
        M, H, I = case["M"], case["H"], case["I"]
        infer = kind == "mlp_infer"
        mlp = m.Fp8MLP(H, I, device=DEVICE, dtype=torch.bfloat16, dialect="deeplinear" if infer else case["dialect"],
                       fp8_dtype=FORMATS["e4m3fn" if infer else case["format"]], low_memory=False if infer else case["low_memory"])
        _set(mlp.up_gate_proj.weight, src.weight(2 * I, H))
        _set(mlp.down_proj.weight, src.weight(H, I))
        st["layer"], st["x"] = mlp, src.activations(M, H)
        if infer:
            mlp.up_gate_proj.cache_weight = mlp.down_proj.cache_weight = True
            with torch.no_grad():
                mlp(st["x"][:1])
        else:
            st["x"].requires_grad_(True)
            st["dy"] = src.gradient(M, H)
    else:
        N, K, splits = case["N"], case["K"], _splits(case)
        st["splits"], st["x"] = splits, src.activations(sum(splits), K)
        weights = [src.weight(N, K) for _ in splits]
        if kind == "moe_decode":
            st["wq"], st["ws"] = m.per_block_cast_to_fp8(weights)
        else:
            st["weights"], st["dy"] = weights, src.gradient(sum(splits), N)
            st["pad"], st["unpad"] = Fp8Padding(len(splits)), Fp8Unpadding(len(splits))
    return st


def _train(layer, x, dy):
    out = layer(x)
    return [out] + list(torch.autograd.grad(out, [x] + list(layer.parameters()), dy))


def _moe_train(st):
    splits, weights = st["splits"], st["weights"]
    with torch.no_grad():
        CustomManger.set_first_micro_batch(weights, True)
        wq, ws, wq_t, ws_t = CustomManger.get_fp8_weight(weights)
        x, padded = st["pad"](st["x"], splits)
        xq, xs, xq_t, xs_t = CustomManger.group_per_token_cast_to_fp8(x, padded)
        out = st["unpad"](CustomManger.fp8_grouped_matmul(xq, xs, wq, ws, padded), splits)
        dy, _ = st["pad"](st["dy"], splits)
        dq, ds, dq_t, ds_t = CustomManger.group_per_token_cast_to_fp8(dy, padded)
        dx = st["unpad"](CustomManger.fp8_grouped_matmul(dq, ds, wq_t, ws_t, padded), splits)
        dw = [fp8_kernel.fp8_matmul(dq_t[g], xq_t[g], ds_t[g], xs_t[g], have_w=False) for g in range(len(splits)) if splits[g]]
    return [out, dx] + dw


def run(state):
    kind = state["case"]["kind"]
    if kind == "linear":
        q, s = m.act_quant(state["x"])
        return m.fp8_gemm(q, s, state["w"], state["ws"], out_dtype=torch.bfloat16)
    if kind == "dequant":
        return m.weight_dequant(state["w"], state["ws"], out_dtype=torch.bfloat16)
    if kind in ("deep_infer", "mlp_infer"):
        with torch.no_grad():
            return state["layer"](state["x"])
    if kind in ("deep_train", "fp8_train", "mlp_train"):
        return _train(state["layer"], state["x"], state["dy"])
    if kind == "moe_decode":
        M = state["x"].size(0)
        q, s, _, _ = m.per_token_cast_to_fp8(state["x"])
        return m.fp8_grouped_matmul(q[:M], s[:M], state["wq"], state["ws"], state["splits"])
    return _moe_train(state)


def work(case):
    kind = case["kind"]
    if kind == "dequant":
        N, K = case["N"], case["K"]
        return {"bytes": 3 * N * K + 4 * -(-N // 128) * -(-K // 128), "flops": N * K}
    if kind in ("mlp_infer", "mlp_train"):
        M, H, I = case["M"], case["H"], case["I"]
        if kind == "mlp_infer":     # bf16 in and out, the three projections' bytes
            return {"bytes": 4 * M * H + 3 * H * I, "flops": 6 * M * H * I}
        # x, dy and the bf16 weights in, output and all gradients out; memory-saving: the up/gate projection twice
        return {"bytes": 8 * M * H + 12 * H * I, "flops": (22 if case["low_memory"] else 18) * M * H * I}
    M, N, K = case.get("M", case.get("tokens")), case["N"], case["K"]
    G = case.get("experts", 1)
    if kind in ("linear", "deep_infer", "moe_decode"):
        return {"bytes": 2 * M * K + G * N * K + 2 * M * N, "flops": 2 * M * N * K}
    return {"bytes": 4 * M * K + 4 * G * N * K + 4 * M * N, "flops": 6 * M * N * K}


def tolerance(case):
    """About four times what separates a pass from the same pass with every GEMM summed in float64 and rounded to bf16
    (measured, relative / largest: single GEMMs and their gradients 3e-4 / 0.008; MLPs 2.6e-3 / 0.03 serving and 0.5 in
    training, where a bf16 value that rounds the other way can turn an fp8 byte of the next quantizer; DeepLinear 2.7e-3 /
    0.011 between a bias added before and after the product is rounded to bf16)."""
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    if kind in ("linear", "fp8_train", "moe_decode", "moe_train"):
        return {"rel": 0.0012, "max": 0.032}
    if kind in ("deep_infer", "deep_train"):
        return {"rel": 0.004, "max": 0.045}
    return {"rel": 0.01, "max": 0.15 if kind == "mlp_infer" else 0.9}
