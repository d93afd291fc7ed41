"""The extension module of the eager calls and model runs against the Python path it shortens: the same results bit
for bit where it takes a call, and the Python path's answer where it declines one."""
import types

import pytest
import torch

from aitemplate_amd import eager

pytestmark = pytest.mark.gpu


def _rand(*shape, dtype=torch.float16, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def _both(monkeypatch, call):
    taken = []

    def counting(fn):
        def wrapped(*args):
            result = fn(*args)
            taken.append(result is not NotImplemented)
            return result
        return wrapped

    names = ("gemm", "bmm", "bmm_softmax_bmm_permute", "mem_eff_attention")
    native = eager._native
    monkeypatch.setattr(eager, "_native", types.SimpleNamespace(**{n: counting(getattr(native, n)) for n in names}))
    here = call()
    monkeypatch.setattr(eager, "_native", types.SimpleNamespace(**{n: lambda *a: NotImplemented for n in names}))
    there = call()
    assert here.shape == there.shape and here.stride() == there.stride() and here.dtype == there.dtype
    assert torch.equal(here, there)
    return taken[0]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case,native", [
    ("one_row", True), ("three_dims", True), ("pitched_a", True), ("residuals", True), ("out_view", True),
    ("transposed_rows", False), ("bmm_broadcast", True), ("bmm_crr_d1", True), ("attention", True), ("mem_eff", True)])
def test_same_results_as_the_python_path(monkeypatch, case, native, dtype):
    w, bias = _rand(72, 64, dtype=dtype, seed=1), _rand(72, dtype=dtype, seed=2)
    x = _rand(6, 64, dtype=dtype)
    wide = _rand(6, 200, dtype=dtype, seed=3)
    q = _rand(4, 40, 64, dtype=dtype, seed=4)
    calls = {
        "one_row": lambda: eager.gemm("gemm_rcr_bias", x[:1], w, bias),
        "three_dims": lambda: eager.gemm("gemm_rcr_bias_gelu", x.view(2, 3, 64), w, bias),
        "pitched_a": lambda: eager.gemm("gemm_rcr", wide[:, 8:72], w),
        "residuals": lambda: eager.gemm("gemm_rcr_bias_add_add", x, w, bias, wide[:, :72], wide[:, 100:172]),
        "out_view": lambda: eager.gemm("gemm_rcr", x, w, out=wide.clone()[:, 16:88]),
        "transposed_rows": lambda: eager.gemm("gemm_rcr_bias", x.view(2, 3, 64).transpose(0, 1), w, bias),
        "bmm_broadcast": lambda: eager.bmm_rcr(q, q[0]),
        "bmm_crr_d1": lambda: eager.bmm("crr", q, q, d1=2),
        "attention": lambda: eager.bmm_softmax_bmm_permute(q, q, q, shape=(2,), scale=0.125, causal=True),
        "mem_eff": lambda: eager.mem_eff_attention(q[None], q[None], q[None], lengths_kv=torch.tensor([17], dtype=torch.int32).cuda()),
    }
    assert _both(monkeypatch, calls[case]) is native


def test_refused_arguments_are_worded_by_the_python_path():
    x, w = _rand(6, 64), _rand(72, 64)
    with pytest.raises(ValueError, match="b must be"):
        eager.gemm("gemm_rcr", x, _rand(72, 32))
    with pytest.raises(ValueError, match="bias must be"):
        eager.gemm("gemm_rcr_bias", x, w)
    with pytest.raises(ValueError, match="no CPU path"):
        eager.gemm("gemm_rcr", x.cpu(), w)
    with pytest.raises(RuntimeError, match="out of range"):
        eager.gemm("gemm_rcr", x, w, algo=10000)
