"""The extension module of the eager calls and model runs (csrc/native_calls.cpp) up to its launches, without a GPU: the
source is built with host memory for the device (native_host/) and entry points that launch nothing.  Every case runs in a
process of its own, since what these cases guard against ends the interpreter."""
import os
import shutil
import subprocess
import sys
import sysconfig
import textwrap

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "aitemplate_amd", "csrc")
HOST = os.path.join(ROOT, "tests", "native_host")

PRELUDE = """
import ctypes, importlib.util, sys, threading
import torch
spec = importlib.util.spec_from_file_location("_native", sys.argv[1])
native = importlib.util.module_from_spec(spec)
spec.loader.exec_module(native)
stub = ctypes.CDLL(sys.argv[1])
launches = lambda: ctypes.c_int.in_dll(stub, "stub_launches").value
x, w, q = torch.randn(6, 64).half(), torch.randn(72, 64).half(), torch.randn(2, 5, 64).half()
# each entry point on a tensor t of q's shape
CALLS = {
    "gemm": lambda t: native.gemm("gemm_rcr", t, w, None, None, None, None, -1, None),
    "gemm_weight": lambda t: native.gemm("gemm_rcr", x, t[0], None, None, None, None, -1, None),
    "gemm_workspace": lambda t: native.gemm("gemm_rcr", x, w, None, None, None, None, -1, t.to(torch.uint8)),
    "gemm_out": lambda t: native.gemm("gemm_rcr", x[:2], w[:5], None, None, None, t[0, :, :2].t().contiguous(), -1, None),
    "bmm": lambda t: native.bmm(0, t, t, None, 0, -1, "bmm_rcr"),
    "attention": lambda t: native.bmm_softmax_bmm_permute(t, t, t, 1, 0.125, False, None),
    "mem_eff": lambda t: native.mem_eff_attention(t[None], t[None], t[None], False, None, None, None),
}
"""


@pytest.fixture(scope="module")
def module(tmp_path_factory):
    build = tmp_path_factory.mktemp("native_host")
    # beside its own native_device.h, which the quoted include finds first
    shutil.copy(os.path.join(CSRC, "native_calls.cpp"), build)
    shutil.copy(os.path.join(HOST, "native_device.h"), build)
    torch_dir = os.path.dirname(torch.__file__)
    so = str(build / "_native.so")
    subprocess.run(["g++", "-O0", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-shared", "-w", "-I" + CSRC,
                    "-I" + sysconfig.get_paths()["include"], f"-I{torch_dir}/include",
                    f"-I{torch_dir}/include/torch/csrc/api/include", str(build / "native_calls.cpp"),
                    os.path.join(HOST, "kernels.cpp"), "-o", so, f"-L{torch_dir}/lib", "-ltorch_python", "-ltorch_cpu", "-lc10"],
                   check=True)
    return so


def _run(module, body):
    done = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body), module], cwd=ROOT, text=True,
                          stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=120)
    assert done.returncode == 0, done.stdout


def test_ordinary_calls_launch(module):
    _run(module, """
        for n, (name, call) in enumerate(CALLS.items()):
            assert call(q) is not NotImplemented, name
            assert launches() == n + 1, name
    """)


def test_op_table_is_the_python_paths(module):
    _run(module, """
        from aitemplate_amd import _kernels
        bias, d = torch.zeros(72).half(), torch.zeros(6, 72).half()
        for op, epilogue in _kernels.EPILOGUE_OF_OP.items():
            if op == "bmm_rcr":
                continue
            residuals = _kernels.NUM_RESIDUALS_OF_EPILOGUE[epilogue]
            args = [bias if epilogue else None, d if residuals >= 1 else None, d if residuals >= 2 else None]
            assert native.gemm(op, x, w, *args, None, -1, None) is not NotImplemented, op
            assert ctypes.c_int.in_dll(stub, "stub_epilogue").value == epilogue, op
            if residuals:
                assert native.gemm(op, x, w, bias, None, None, None, -1, None) is NotImplemented, op
    """)


@pytest.mark.parametrize("transform", ["vmap", "grad", "functionalize"])
def test_wrappers_without_memory_of_their_own_are_declined(module, transform):
    """torch.func's tensors are of the exact type torch.Tensor and have no storage: the Python path words the error."""
    _run(module, f"""
        def declined(t):
            for name, call in CALLS.items():
                assert call(t) is NotImplemented, name
            return t.float().sum()
        t = torch.randn(3, 2, 5, 64).half()
        if "{transform}" == "vmap":
            torch.vmap(declined)(t)
        elif "{transform}" == "grad":
            torch.func.grad(declined)(q)
        else:
            torch.func.functionalize(declined)(q)
        assert launches() == 0
    """)


@pytest.mark.parametrize("kind", ["dict", "list"])
@pytest.mark.parametrize("change", ["replace", "remove", "clear"])
def test_a_run_keeps_what_it_was_given(module, kind, change):
    """The caller's containers may change while a run is on (the run gives up the interpreter lock): the
    run's tensors live on, and the results are the ones it wrote."""
    _run(module, f"""
        import gc
        RUN = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p, ctypes.c_size_t,
                               ctypes.c_void_p, ctypes.c_bool, ctypes.c_bool, ctypes.POINTER(ctypes.POINTER(ctypes.c_int64)))
        class AITData(ctypes.Structure):
            _fields_ = [("ptr", ctypes.c_void_p), ("shape", ctypes.c_void_p), ("rank", ctypes.c_size_t), ("dtype", ctypes.c_int)]
        names = {{"y": 1, "z": 0}}
        fresh = lambda: {{"y": torch.zeros(4, 8), "z": torch.zeros(4)}}
        outputs = fresh() if "{kind}" == "dict" else [fresh()["z"], fresh()["y"]]
        inputs = {{"x": torch.ones(3)}} if "{kind}" == "dict" else [torch.ones(3)]
        def run(handle, ins, n_in, outs, n_out, stream, sync, graph, shapes):
            if "{change}" == "replace":
                for key in (list(outputs) if "{kind}" == "dict" else range(2)):
                    outputs[key] = torch.full((64,), 7.0)
                for key in (list(inputs) if "{kind}" == "dict" else range(1)):
                    inputs[key] = None
            elif "{change}" == "remove":
                outputs.pop("z" if "{kind}" == "dict" else 0)
            else:
                outputs.clear()
                inputs.clear()
            gc.collect()
            hold.extend(torch.full((64,), 9.0) for _ in range(64))   # takes up memory that was given back
            data = ctypes.cast(outs, ctypes.POINTER(AITData))
            for i, numel in ((0, 2), (1, 16)):
                ctypes.memmove(data[i].ptr, (ctypes.c_float * numel)(*[float(i + 1)] * numel), 4 * numel)
            shapes[0][0], shapes[1][0], shapes[1][1] = 2, 2, 8
            return 0
        hold, callback = [], RUN(run)
        result = native.model_run(ctypes.cast(callback, ctypes.c_void_p).value, 1, {{"x": 0}}, names, [1, 2], inputs, outputs,
                                  None, True, False)
        assert list(result) == ["y", "z"], result
        assert torch.equal(result["y"], torch.full((2, 8), 2.0)) and torch.equal(result["z"], torch.ones(2))
        assert all((t == 9).all() for t in hold)
    """)


def test_a_run_keeps_the_shapes_it_was_given(module):
    """A tensor that is given another shape while a run is on: the run's pointers to shapes stay what they were."""
    _run(module, """
        RUN = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p, ctypes.c_size_t,
                               ctypes.c_void_p, ctypes.c_bool, ctypes.c_bool, ctypes.POINTER(ctypes.POINTER(ctypes.c_int64)))
        class AITData(ctypes.Structure):
            _fields_ = [("ptr", ctypes.c_void_p), ("shape", ctypes.POINTER(ctypes.c_int64)), ("rank", ctypes.c_size_t),
                        ("dtype", ctypes.c_int)]
        a, b, y = torch.ones(3, 4), torch.ones(5), torch.zeros(4, 8)
        seen = []
        def run(handle, ins, n_in, outs, n_out, stream, sync, graph, shapes):
            a.resize_(1, 2, 3, 2, 1, 1, 1)
            b.resize_(5, 1)
            y.resize_(2, 2, 2, 2, 2, 1, 1)
            data = ctypes.cast(ins, ctypes.POINTER(AITData))
            for d in (data[0], data[1], ctypes.cast(outs, ctypes.POINTER(AITData))[0]):
                seen.append([d.shape[i] for i in range(d.rank)])
            shapes[0][0], shapes[0][1] = 3, 8
            return 0
        callback = RUN(run)
        result = native.model_run(ctypes.cast(callback, ctypes.c_void_p).value, 1, {"a": 0, "b": 1}, {"y": 0}, [2], [a, b], [y],
                                  None, True, False)
        assert seen == [[3, 4], [5], [4, 8]], seen
        assert result["y"].shape == (3, 8)
    """)


@pytest.mark.parametrize("mode", ["dispatch", "fake", "function", "vmap", "trace"])
def test_calls_under_a_mode_are_declined(module, mode):
    """The Python path's torch calls (its allocation, reshapes and views) are what a mode sees, refuses or records."""
    _run(module, f"""
        from torch._subclasses.fake_tensor import FakeTensorMode
        from torch.overrides import TorchFunctionMode
        from torch.utils._python_dispatch import TorchDispatchMode
        class Dispatch(TorchDispatchMode):
            def __torch_dispatch__(self, func, types, args=(), kwargs=None):
                return func(*args, **(kwargs or {{}}))
        class Function(TorchFunctionMode):
            def __torch_function__(self, func, types, args=(), kwargs=None):
                return func(*args, **(kwargs or {{}}))
        nowhere = 8   # an address that must not be called
        y = torch.zeros(6, 72).half()
        q4 = q[None]   # (arguments made outside of the mode)
        def calls():
            yield native.gemm("gemm_rcr", x, w, None, None, None, None, -1, None)
            yield native.gemm("gemm_rcr", x, w, None, None, None, y, -1, None)
            yield native.bmm(0, q, q, None, 0, -1, "bmm_rcr")
            yield native.bmm_softmax_bmm_permute(q, q, q, 1, 0.125, False, None)
            yield native.mem_eff_attention(q4, q4, q4, False, None, None, None)
            yield native.model_run(nowhere, 1, {{"x": 0}}, {{"y": 0}}, [2], [x], [y], None, True, False)
        declined = lambda: all(result is NotImplemented for result in calls())
        if "{mode}" == "vmap":
            seen = []
            torch.vmap(lambda t: (seen.append(declined()), t)[1])(torch.zeros(2, 3))
            assert seen == [True]
        elif "{mode}" == "trace":
            seen = []
            torch.jit.trace(lambda t: (seen.append(declined()), t + 1)[1], (torch.zeros(3),), check_trace=False)
            assert all(seen) and seen
        else:
            with dict(dispatch=Dispatch, fake=FakeTensorMode, function=Function)["{mode}"]():
                assert declined()
        assert launches() == 0
        # and no longer once it is over, nor in what autograd and autocast modes leave to the kernels as before
        with torch.inference_mode(), torch.autocast("cpu"):
            assert native.gemm("gemm_rcr", x, w, None, None, None, None, -1, None).is_inference()
        with torch.no_grad():
            assert native.bmm(0, q, q, None, 0, -1, "bmm_rcr") is not NotImplemented
        assert launches() == 2
    """)


def test_declined_calls_leave_no_error_behind(module):
    """An integer that C cannot take: raised where the call ends with it, and nothing left set where it is declined (the
    interpreter makes a SystemError of a result with an error set)."""
    _run(module, """
        for heads in (2 ** 70, -2 ** 70):   # (2 ** 64 + 1 taken modulo 2 ** 64 would be one head of an empty result)
            try:
                native.bmm_softmax_bmm_permute(q, q, q, heads, 0.125, False, None)
            except OverflowError:
                pass
            else:
                assert False, heads
        y = torch.zeros(6, 72).half()
        run = lambda index, ranks: native.model_run(8, 1, {"x": index}, {"y": 0}, ranks, [x], [y], None, True, False)
        for index, ranks in ((0, [2 ** 70]), (0, ["2"]), (0, [None]), (2 ** 70, [2]), ("0", [2]), (-1, [2])):
            assert run(index, ranks) is NotImplemented, (index, ranks)
            by_name = native.model_run(8, 1, {"x": index}, {"y": 0}, ranks, {"x": x}, [y], None, True, False)
            assert by_name is NotImplemented, (index, ranks)
        assert launches() == 0
    """)


def test_an_op_name_without_utf8_is_declined(module):
    """(The Python path has no such op and says so.)"""
    _run(module, """
        assert native.gemm("\\ud800", x, w, None, None, None, None, -1, None) is NotImplemented
        assert launches() == 0
    """)


@pytest.mark.parametrize("first", ["context", "default"])
def test_a_default_device_changes_nothing(module, first):
    """`with torch.device(...)` and torch.set_default_device say where tensors go whose device is not named: the calls name
    it.  A class of that mode's that does more, or a mode beside it, is as any other mode."""
    _run(module, f"""
        from torch.overrides import TorchFunctionMode
        from torch.utils._device import DeviceContext
        class Derived(DeviceContext):
            pass
        class Function(TorchFunctionMode):
            def __torch_function__(self, func, types, args=(), kwargs=None):
                return func(*args, **(kwargs or {{}}))
        call = lambda: native.gemm("gemm_rcr", x, w, None, None, None, None, -1, None)
        def within():
            out = call()
            assert out is not NotImplemented and out.device == x.device
            with Function():
                assert call() is NotImplemented
        if "{first}" == "context":
            with torch.device("meta"):
                within()
        else:
            torch.set_default_device("meta")
            within()
            torch.set_default_device(None)
        assert launches() == 1
        with Derived("meta"):
            assert call() is NotImplemented
        assert call() is not NotImplemented
    """)


def test_errors_keep_their_types(module):
    """What torch raises through its own bindings: an allocation that fails is an OutOfMemoryError, without a C++ trace."""
    _run(module, """
        try:
            native.gemm("gemm_rcr", x.bfloat16(), w.bfloat16(), None, None, None, None, -1, None)
        except torch.OutOfMemoryError as e:
            assert str(e) == "host memory is out of bfloat16", str(e)
        else:
            assert False
    """)


@pytest.mark.parametrize("why", ["not built", "built for another torch"])
def test_without_the_extension_module_the_python_path_takes_every_call(why):
    """The module saves host time and computes nothing: without it, calls and model runs do as before it was there."""
    body = f"""
        import ctypes, sys, types, warnings
        import torch
        sys.modules["aitemplate_amd._native"] = None
        if "{why}" != "not built":
            sys.modules["aitemplate_amd._native"] = types.ModuleType("aitemplate_amd._native")
            sys.modules["aitemplate_amd._native"].torch_version = "1.0.0"
            import aitemplate_amd
            aitemplate_amd._native = sys.modules["aitemplate_amd._native"]
        with warnings.catch_warnings(record=True) as seen:
            warnings.simplefilter("always")
            from aitemplate_amd import eager
        assert any("_native" in str(w.message) for w in seen), seen
        from aitemplate_amd.compiler import Model
        x, q = torch.randn(2, 64).half(), torch.randn(1, 2, 5, 64).half()
        calls = dict(gemm=lambda: eager.gemm("gemm_rcr", x, x), bmm_rcr=lambda: eager.bmm_rcr(q[0], q[0]),
                     bmm=lambda: eager.bmm("rrr", q[0], q[0]), mem_eff=lambda: eager.mem_eff_attention(q, q, q),
                     attention=lambda: eager.bmm_softmax_bmm_permute(q[0], q[0], q[0], (2,)))
        for name, call in calls.items():
            try:
                call()
            except ValueError as e:
                assert "no CPU path" in str(e), (name, e)
            else:
                assert False, name
        model = object.__new__(Model)
        model.DLL = types.SimpleNamespace(is_open=True, close=lambda: None, DLL=types.SimpleNamespace(
            AITemplateModelContainerRun=ctypes.CFUNCTYPE(ctypes.c_int)(lambda: 1)))
        model.handle = model.allocator_handle = ctypes.c_void_p()
        model._native_run, model._input_name_to_index, model._output_name_to_index, model._output_ndims = None, {{"x": 0}}, {{"y": 0}}, [2]
        try:
            model.run_with_tensors([x], [x])
        except ValueError as e:
            assert "contiguous and on GPU" in str(e), e
        else:
            assert False
    """
    done = subprocess.run([sys.executable, "-c", textwrap.dedent(body)], cwd=ROOT, text=True, stdout=subprocess.PIPE,
                          stderr=subprocess.STDOUT, timeout=120)
    assert done.returncode == 0, done.stdout


@pytest.mark.parametrize("built,here,used", [
    ("2.10.0", "2.10.0", True), ("2.10.0+rocm7.0", "2.10.0+rocm7.0", True), ("2.10.0+rocm7.0", "2.10.0+local", True),
    ("2.10.0", "2.11.0", False), ("2.11.0a0+git0123abc", "2.11.0a0+git0123abc", True), ("2.11.0a0", "2.11.0", False),
    ("2.11.0.dev20260101", "2.11.0.dev20260101+rocm7.0", True), ("2.11.0.dev20260101", "2.11.0.dev20260102", False)])
def test_the_module_is_used_with_the_torch_it_was_built_for(monkeypatch, built, here, used):
    """Pre-releases too: the version that torch names at run time, not the three numbers of its headers."""
    import types
    import warnings

    import aitemplate_amd
    from aitemplate_amd import _kernels

    there = types.ModuleType("aitemplate_amd._native")
    there.torch_version, there.torch_build = built.split("a0")[0].split(".dev")[0].split("+")[0], built
    monkeypatch.setitem(sys.modules, "aitemplate_amd._native", there)
    monkeypatch.setattr(aitemplate_amd, "_native", there, raising=False)
    monkeypatch.setattr(torch, "__version__", here)
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        assert (_kernels.load_native() is there) is used
    assert bool(seen) is not used


def test_the_built_module_fits_this_torch():
    from aitemplate_amd import _kernels

    native = _kernels.load_native()
    assert native.torch_version == torch.__version__.split("+")[0]
    assert native.torch_build == torch.__version__


def test_the_kernel_library_builds_without_torch(tmp_path):
    """`make` builds everything but the extension module where python has no torch (or there is no python)."""
    no_torch = tmp_path / "python3"
    no_torch.write_text(f"#!/bin/sh\nexec {sys.executable} -S \"$@\"\n")   # (-S: no site-packages)
    no_torch.chmod(0o755)
    for python, built in ((sys.executable, True), (str(no_torch), False), (str(tmp_path / "none"), False)):
        out = subprocess.run(["make", "-B", "-n", "-C", CSRC, f"PYTHON={python}"], text=True, stdout=subprocess.PIPE,
                             stderr=subprocess.STDOUT)
        assert out.returncode == 0, out.stdout[-2000:]
        assert ("native_calls.cpp" in out.stdout) is built
        assert "profiler_main.cpp" in out.stdout and "gemm_inst_0_0.o" in out.stdout
        assert ("_native.so is not built" in out.stdout) is not built
