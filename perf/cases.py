"""What users of this framework have it compute, as timed cases.

Four kinds of call, each through its public entry point:

* ``linear``:    ``eager.gemm`` - a linear layer with its fused epilogue;
* ``bmm``:       ``eager.bmm`` - a batched product in one of the four operand layouts;
* ``attention``: ``eager.bmm_softmax_bmm_permute`` and ``eager.mem_eff_attention``;
* ``encoder``:   one transformer encoder block built from ``frontend.nn`` modules, compiled by ``compile_model`` and
  run by ``Model.run_with_tensors`` with its weights bound as constants.
"""
import atexit
import math
import os
import shutil
import tempfile

import torch

from aitemplate_amd import eager
from aitemplate_amd.compiler import Model, compile_model
from aitemplate_amd.frontend import Tensor, nn
from aitemplate_amd.testing import detect_target

DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}

# residual operands behind the bias
RESIDUALS = {"gemm_rcr": 0, "gemm_rcr_bias": 0, "gemm_rcr_bias_relu": 0, "gemm_rcr_bias_gelu": 0,
             "gemm_rcr_bias_fast_gelu": 0, "gemm_rcr_bias_swish": 0, "gemm_rcr_bias_sigmoid": 0,
             "gemm_rcr_bias_add": 1, "gemm_rcr_bias_mul": 1, "gemm_rcr_bias_add_relu": 1, "gemm_rcr_bias_add_add": 2}

MOST_FLOPS = 2 * 8192 ** 3  # of the largest listed case
MOST_BYTES = 1 << 30


def listed():
    return [
        # one pooled row through a hidden-size layer: the smallest call a serving loop makes, all latency
        {"name": "linear_one_row", "path": "linear", "op": "gemm_rcr_bias", "dtype": "float16", "M": 1, "N": 768, "K": 768},
        # one short sequence through a layer: benchmark configuration 1
        {"name": "linear_one_sequence", "path": "linear", "op": "gemm_rcr_bias", "dtype": "float16", "M": 256, "N": 1024,
         "K": 1024},
        # decoding: one row against a wide weight whose K is not a multiple of 8 (the GEMM benchmark's shape)
        {"name": "linear_decode_wide", "path": "linear", "op": "gemm_rcr_bias", "dtype": "float16", "M": 1, "N": 6912,
         "K": 8314},
        # the same layer over a prompt of 2048 rows, with a ReLU
        {"name": "linear_prefill_ragged", "path": "linear", "op": "gemm_rcr_bias_relu", "dtype": "bfloat16", "M": 2048,
         "N": 6912, "K": 8314},
        # BERT-base feed-forward up-projection, 64 sequences of 384: configuration 2, the benchmark's headline
        {"name": "ffn_up", "path": "linear", "op": "gemm_rcr_bias_gelu", "dtype": "float16", "M": 24576, "N": 3072,
         "K": 768},
        # ViT-L MLP down-projection with two residuals, 64 images of 197 tokens: configuration 3
        {"name": "mlp_down", "path": "linear", "op": "gemm_rcr_bias_add_add", "dtype": "float16", "M": 12608, "N": 1024,
         "K": 4096},
        # the largest dense product
        {"name": "square_large", "path": "linear", "op": "gemm_rcr", "dtype": "bfloat16", "M": 8192, "N": 8192,
         "K": 8192},
        # attention scores of 64 sequences and 12 heads, not fused: configuration 4
        {"name": "bmm_scores", "path": "bmm", "layout": "rcr", "dtype": "float16", "B": 768, "M": 384, "N": 384, "K": 64},
        # self-attention of a diffusion UNet at 64 x 64 latents: configuration 5
        {"name": "attention_unet", "path": "attention", "op": "bmm_softmax_bmm_permute", "dtype": "float16", "batch": 2,
         "heads": 8, "seq_q": 4096, "seq_kv": 4096, "head_dim": 40, "causal": False, "lengths": False},
        # 64 sequences padded to 384 tokens, with their key lengths on the device (BERT-base heads)
        {"name": "attention_padded", "path": "attention", "op": "mem_eff_attention", "dtype": "float16", "batch": 64,
         "heads": 12, "seq_q": 384, "seq_kv": 384, "head_dim": 64, "causal": False, "lengths": True},
        # causal self-attention over a long prompt, wide heads
        {"name": "attention_causal_long", "path": "attention", "op": "mem_eff_attention", "dtype": "bfloat16", "batch": 2,
         "heads": 16, "seq_q": 4096, "seq_kv": 4096, "head_dim": 128, "causal": True, "lengths": False},
        # a compiled BERT-base encoder block answering one request of 384 tokens
        {"name": "encoder_one_request", "path": "encoder", "dtype": "float16", "batch": 1, "seq": 384, "hidden": 768,
         "heads": 12},
    ]


# ---- drawn cases -----------------------------------------------------------------------------------------------

def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _multiple(rng, low, high, of):
    return max(of, _log(rng, low, high) // of * of)


def _draw_linear(rng):
    ragged = rng.random() < 0.3  # any N and K; otherwise the multiples of 16 that hidden sizes are
    return {"path": "linear", "op": rng.choice(sorted(RESIDUALS)), "dtype": rng.choice(sorted(DTYPES)),
            "M": _log(rng, 1, 24576),
            "N": _log(rng, 64, 8400) if ragged else _multiple(rng, 64, 8192, 16),
            "K": _log(rng, 64, 8400) if ragged else _multiple(rng, 64, 8192, 16)}


def _draw_bmm(rng):
    ragged = rng.random() < 0.3
    size = (lambda: _log(rng, 16, 1024)) if ragged else (lambda: _multiple(rng, 16, 1024, 8))
    return {"path": "bmm", "layout": rng.choice(("rcr", "rrr", "ccr", "crr")), "dtype": rng.choice(sorted(DTYPES)),
            "B": _log(rng, 1, 1024), "M": size(), "N": size(), "K": size()}


def _draw_attention(rng):
    op = rng.choice(("bmm_softmax_bmm_permute", "mem_eff_attention"))
    seq = _log(rng, 16, 8192)
    return {"path": "attention", "op": op, "dtype": rng.choice(sorted(DTYPES)), "batch": _log(rng, 1, 64),
            "heads": rng.choice((4, 8, 12, 16)), "seq_q": seq, "seq_kv": 77 if rng.random() < 0.15 else seq,
            "head_dim": rng.choice((32, 40, 64, 64, 80, 128, 160)), "causal": rng.random() < 0.3,
            "lengths": op == "mem_eff_attention" and rng.random() < 0.5}


def _draw_encoder(rng):
    hidden = rng.choice((256, 512, 768, 1024))
    return {"path": "encoder", "dtype": rng.choice(sorted(DTYPES)), "batch": _log(rng, 1, 64), "seq": _log(rng, 8, 512),
            "hidden": hidden, "heads": hidden // 64}


def draw(rng):
    kinds = (_draw_linear,) * 10 + (_draw_attention,) * 4 + (_draw_bmm,) * 3 + (_draw_encoder,) * 3
    while True:
        case = rng.choice(kinds)(rng)
        w = work(case)
        # attention reaches a third of a plain product's rate
        cost = w["flops"] * (3 if case["path"] == "attention" else 1)
        if cost <= MOST_FLOPS and w["bytes"] <= MOST_BYTES:
            return case


# ---- work and tolerance ----------------------------------------------------------------------------------------

def _kv_lengths(case):
    """Key lengths of a padded batch: spread evenly from a quarter of the keys to all of them."""
    n, b = case["seq_kv"], case["batch"]
    return [max(1, n - (3 * n // 4) * i // max(1, b - 1)) for i in range(b)]


def work(case):
    if case["path"] == "linear":
        M, N, K, nres = case["M"], case["N"], case["K"], RESIDUALS[case["op"]]
        bias = 0 if case["op"] == "gemm_rcr" else N
        return {"bytes": 2 * (M * K + N * K + bias + (1 + nres) * M * N), "flops": 2 * M * N * K}
    if case["path"] == "bmm":
        B, M, N, K = case["B"], case["M"], case["N"], case["K"]
        return {"bytes": 2 * B * (M * K + N * K + M * N), "flops": 2 * B * M * N * K}
    if case["path"] == "attention":
        h, sq, d = case["heads"], case["seq_q"], case["head_dim"]
        keys = _kv_lengths(case) if case["lengths"] else [case["seq_kv"]] * case["batch"]
        pairs = 0
        for n in keys:
            if case["causal"]:  # query i sees keys 0 .. i
                full = min(sq, n)
                pairs += full * (full + 1) // 2 + max(0, sq - n) * n
            else:
                pairs += sq * n
        return {"bytes": 2 * h * d * (2 * case["batch"] * sq + 2 * sum(keys)), "flops": 4 * h * d * pairs}
    B, S, D = case["batch"], case["seq"], case["hidden"]
    rows = B * S
    weights = 12 * D * D + 9 * D
    return {"bytes": 2 * (2 * rows * D + weights), "flops": 2 * rows * 12 * D * D + 4 * B * S * S * D}


def tolerance(case):
    # the inputs and the result have 11 (float16) or 8 (bfloat16) bits, sums are 32-bit; the encoder block rounds
    # between its five kernels
    half = case["dtype"] == "float16"
    if case["path"] == "encoder":
        return {"rel": 3e-3 if half else 2e-2, "max": 3e-2 if half else 2e-1}
    return {"rel": 1e-3 if half else 8e-3, "max": 1e-2 if half else 8e-2}


# ---- prepare and run -------------------------------------------------------------------------------------------

_compiled = {}  # (dtype, batch, seq, hidden, heads) -> the compiled block, as a program keeps it
_workdir = None


def _encoder_library(case):
    global _workdir
    key = tuple(case[k] for k in ("dtype", "batch", "seq", "hidden", "heads"))
    if key not in _compiled:
        if _workdir is None:
            _workdir = tempfile.mkdtemp(prefix="encoder_")
            atexit.register(shutil.rmtree, _workdir, ignore_errors=True)
            os.environ.setdefault("CACHE_DIR", _workdir)  # of profiling results
        dtype, B, S, D, H = key
        attention = nn.MultiheadAttention(D, B, S, H, qkv_bias=True, has_residual=True, dtype=dtype)
        up = nn.Linear(D, 4 * D, specialization="fast_gelu", dtype=dtype)
        down = nn.Linear(4 * D, D, specialization="add", dtype=dtype)
        for prefix, module in (("attention", attention), ("up", up), ("down", down)):
            module.name_parameter_tensor(prefix)
        x = Tensor(shape=[B, S, D], dtype=dtype, name="x", is_input=True)
        residual = Tensor(shape=[B * S, D], dtype=dtype, name="residual", is_input=True)
        h = attention(x, residual)
        y = down(up(h), h)
        y._attrs["name"], y._attrs["is_output"] = "y", True
        _compiled[key] = compile_model(y, detect_target(), _workdir, "block_" + "_".join(str(k) for k in key))
    return _compiled[key].lib_path


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]

    def normal(*shape, scale=1.0):
        return torch.randn(*shape, device="cuda", generator=g, dtype=torch.float32).mul_(scale).to(dtype)

    if case["path"] == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        x, w = normal(M, K), normal(N, K, scale=K ** -0.5)
        bias = None if case["op"] == "gemm_rcr" else normal(N, scale=0.1)
        return {"path": "linear", "args": (case["op"], x, w, bias, *(normal(M, N) for _ in range(RESIDUALS[case["op"]])))}
    if case["path"] == "bmm":
        B, M, N, K = case["B"], case["M"], case["N"], case["K"]
        a = normal(B, K, M) if case["layout"][0] == "c" else normal(B, M, K)
        b = normal(B, N, K, scale=K ** -0.5) if case["layout"][1] == "c" else normal(B, K, N, scale=K ** -0.5)
        return {"path": "bmm", "args": (case["layout"], a, b)}
    if case["path"] == "attention":
        B, H, d = case["batch"], case["heads"], case["head_dim"]
        lead = (B * H,) if case["op"] == "bmm_softmax_bmm_permute" else (B, H)
        q = normal(*lead, case["seq_q"], d)
        k, v = (normal(*lead, case["seq_kv"], d) for _ in range(2))
        state = {"path": case["op"], "args": (q, k, v), "heads": H, "scale": d ** -0.5, "causal": case["causal"]}
        if case["op"] == "mem_eff_attention":
            lengths = _kv_lengths(case)
            state["lengths"] = torch.tensor(lengths, dtype=torch.int32, device="cuda") if case["lengths"] else None
        return state
    B, S, D = case["batch"], case["seq"], case["hidden"]
    module = Model(_encoder_library(case))
    weights = {}
    for name, n, k in (("attention_qkv", 3 * D, D), ("attention_proj", D, D), ("up", 4 * D, D), ("down", D, 4 * D)):
        weights[name + "_weight"] = normal(n, k, scale=k ** -0.5)
        weights[name + "_bias"] = normal(n, scale=0.1)
    module.set_many_constants_with_tensors(weights)
    x = normal(B, S, D)
    return {"path": "encoder", "module": module, "feed": {"x": x, "residual": x.view(B * S, D)},
            "out": [torch.empty(B, S, D, device="cuda", dtype=dtype)]}


def run(state):
    if state["path"] == "linear":
        return eager.gemm(*state["args"])
    if state["path"] == "bmm":
        return eager.bmm(*state["args"])
    if state["path"] == "bmm_softmax_bmm_permute":
        return eager.bmm_softmax_bmm_permute(*state["args"], shape=(state["heads"],), scale=state["scale"],
                                             causal=state["causal"])
    if state["path"] == "mem_eff_attention":
        return eager.mem_eff_attention(*state["args"], causal=state["causal"], lengths_kv=state["lengths"])
    return state["module"].run_with_tensors(state["feed"], state["out"])
