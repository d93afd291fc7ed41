"""The extension module of the eager calls and model runs against the Python path it shortens: the same results bit
for bit where it takes a call, and the Python path's answer where it declines one."""
import os
import types

import pytest
import torch

from aitemplate_amd import _kernels, eager
from aitemplate_amd.compiler import compile_model, ops
from aitemplate_amd.frontend import IntImm, IntVar, Tensor
from aitemplate_amd.testing import detect_target

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
    ("workspace", True), ("small_workspace", True), ("transposed_rows", False), ("bmm_broadcast", True), ("bmm_crr_d1", True), ("attention", True), ("mem_eff", True)])
def test_same_results_as_the_python_path(monkeypatch, case, native, dtype):
    w, bias = _rand(72, 64, dtype=dtype, seed=1), _rand(72, dtype=dtype, seed=2)
    x = _rand(6, 64, dtype=dtype)
    wide = _rand(6, 200, dtype=dtype, seed=3)
    q = _rand(4, 40, 64, dtype=dtype, seed=4)
    long_x, long_w = _rand(16, 2048, dtype=dtype, seed=5), _rand(72, 2048, dtype=dtype, seed=6)
    splitk = next(i for i, n in enumerate(_kernels.gemm_algo_names(0, 0)) if "splitk" in n)
    need = eager.gemm_workspace_bytes("gemm_rcr", splitk, 16, 72, 2048, dtype)
    assert need > 0
    calls = {
        "one_row": lambda: eager.gemm("gemm_rcr_bias", x[:1], w, bias),
        "three_dims": lambda: eager.gemm("gemm_rcr_bias_gelu", x.view(2, 3, 64), w, bias),
        "pitched_a": lambda: eager.gemm("gemm_rcr", wide[:, 8:72], w),
        "residuals": lambda: eager.gemm("gemm_rcr_bias_add_add", x, w, bias, wide[:, :72], wide[:, 100:172]),
        "out_view": lambda: eager.gemm("gemm_rcr", x, w, out=wide.clone()[:, 16:88]),
        "workspace": lambda: eager.gemm("gemm_rcr", long_x, long_w, algo=splitk, workspace=eager.new_workspace(need)),
        "small_workspace": lambda: eager.gemm("gemm_rcr", long_x, long_w, algo=splitk, workspace=eager.new_workspace(need // 2)),
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


def test_wrapper_tensors_are_refused_as_before():
    """torch.func's wrappers have no memory that a kernel could read: an error, from a process that lives on."""
    x, w = _rand(3, 6, 64), _rand(72, 64)
    with pytest.raises(RuntimeError, match="data pointer|storage"):
        torch.vmap(lambda t: eager.gemm("gemm_rcr", t, w))(x)
    with pytest.raises(RuntimeError, match="data pointer|storage"):
        torch.vmap(lambda t: eager.mem_eff_attention(t[None, None], t[None, None], t[None, None]))(x)
    assert eager.gemm("gemm_rcr", x, w).shape == (3, 6, 72)


def _calls_on_late_inputs():
    """name -> (inputs, call): each call takes the inputs that it is to read."""
    w = _rand(72, 64, seed=1)
    q = [_rand(4, 40, 64, seed=s) for s in (2, 3, 4)]
    return {
        "gemm": ([_rand(6, 64)], lambda x: eager.gemm("gemm_rcr", x, w)),
        "gemm_workspace": ([_rand(16, 64)], lambda x: eager.gemm("gemm_rcr", x, w, workspace=eager.new_workspace(1 << 20))),
        "bmm": (q[:2], lambda a, b: eager.bmm("rcr", a, b)),
        "attention": (q, lambda a, b, c: eager.bmm_softmax_bmm_permute(a, b, c, (2,), scale=0.125)),
        "mem_eff": (q, lambda a, b, c: eager.mem_eff_attention(a[None], b[None], c[None])),
    }


def _on_another_stream(inputs, call):
    """call's result where its inputs are written on a side stream, behind other work there."""
    want = call(*inputs)
    late = [torch.zeros_like(t) for t in inputs]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torch.cuda._sleep(1_000_000)
        for to, t in zip(late, inputs):
            to.copy_(t)
        got = call(*late)
    side.synchronize()
    return want, got


@pytest.mark.parametrize("name", ["gemm", "gemm_workspace", "bmm", "attention", "mem_eff"])
def test_calls_go_to_the_current_stream(name):
    want, got = _on_another_stream(*_calls_on_late_inputs()[name])
    assert torch.equal(want, got)


@pytest.fixture(scope="module")
def model():
    m = IntVar([1, 64], name="m")
    x = Tensor(shape=[m, IntImm(40)], name="x", is_input=True)
    w, v = (Tensor(shape=[IntImm(n), IntImm(40)], name=name, is_input=True) for n, name in ((72, "w"), (24, "v")))
    y, z = ops.gemm_rcr()(x, w), ops.gemm_rcr()(x, v)
    for t, name in ((y, "y"), (z, "z")):
        t._attrs["name"] = name
        t._attrs["is_output"] = True
    module = compile_model([y, z], detect_target(), os.environ.get("AIT_TEST_WORKDIR", "/tmp/aitemplate_amd_tests"), "native_calls")
    yield module
    module.close()


@pytest.mark.parametrize("kind", ["dict", "reversed dict", "list", "tuple"])
@pytest.mark.parametrize("rows", [1, 17, 64])
@pytest.mark.parametrize("options", [{}, {"graph_mode": True}, {"sync": False}])
def test_model_runs_as_the_python_path_does(model, kind, rows, options):
    """The same names, order, shapes, memory and values, also where outputs are larger than a run's result."""
    inputs = {"x": _rand(rows, 40), "w": _rand(72, 40, seed=1), "v": _rand(24, 40, seed=2)}

    def run():
        outputs = {"y": torch.full((64, 72), 3.0).half().cuda(), "z": torch.full((64, 24), 3.0).half().cuda()}
        if kind in ("list", "tuple"):
            index = model.get_input_name_to_index_map()
            make = list if kind == "list" else tuple
            ins = make(sorted(inputs.values(), key=lambda t: index[next(n for n, i in inputs.items() if i is t)]))
            outs = make(outputs[n] for n in sorted(outputs, key=model.get_output_name_to_index_map().get))
        else:
            ins = inputs
            outs = outputs if kind == "dict" else dict(reversed(outputs.items()))
        result = model.run_with_tensors(ins, outs, **options)
        torch.cuda.synchronize()
        return result, outputs

    taken = []
    model._native_run = None
    run()   # looks the extension function up
    native, address = model._native_run
    try:
        model._native_run = (lambda *args: (taken.append(native(*args)), taken[-1])[1], address)
        here, here_out = run()
        model._native_run = (lambda *args: NotImplemented, address)
        there, there_out = run()
    finally:
        model._native_run = None
    assert taken and taken[0] is not NotImplemented
    assert list(here) == list(there)
    for name in here:
        assert here[name].shape == there[name].shape == (rows, {"y": 72, "z": 24}[name])
        assert here[name].data_ptr() == here_out[name].data_ptr() and there[name].data_ptr() == there_out[name].data_ptr()
        assert torch.equal(here[name], there[name]) and torch.equal(here_out[name], there_out[name])


@pytest.mark.parametrize("graph_mode", [False, True])
def test_model_runs_on_the_current_stream(model, graph_mode):
    w, v = _rand(72, 40, seed=1), _rand(24, 40, seed=2)

    def call(x):
        outputs = {"y": torch.zeros(64, 72, dtype=torch.float16, device="cuda"), "z": torch.zeros(64, 24, dtype=torch.float16, device="cuda")}
        return model.run_with_tensors({"x": x, "w": w, "v": v}, outputs, sync=False, graph_mode=graph_mode)["y"]
    want, got = _on_another_stream([_rand(17, 40)], call)
    assert torch.equal(want, got)
