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
