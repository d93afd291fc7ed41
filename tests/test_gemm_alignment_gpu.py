"""Instances for operands at any element and for few rows, at the edges of their tiles, slabs and pieces."""
import os
import subprocess

import pytest
import torch

from aitemplate_amd import _kernels, eager
from oracle import oracle

pytestmark = pytest.mark.gpu


def _rand(shape, seed, scale=1.0, dtype=torch.float16):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).to(dtype)


def _instances(epi, dtype):
    return [(i, n) for i, n in enumerate(_kernels.gemm_algo_names(epi, dtype)) if n.endswith("_v1") or "rows" in n]


# K around the 8-element pieces, the 64- and 128-deep slabs and the 1024 that a few-rows workgroup takes together
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (1, 33, 7), (16, 16, 127), (17, 15, 129), (5, 100, 1025), (40, 31, 1151),
                                   (65, 129, 63), (255, 65, 65), (130, 257, 191), (64, 64, 64), (3, 50, 2050)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_operands_at_any_element(M, N, K, dtype):
    lib = _kernels.load()
    dt = 0 if dtype == torch.float16 else 1
    # views one element into their buffers; what lies before, behind and between the rows must not count
    x, w = _rand((M, K), 1, dtype=dtype), _rand((N, K), 2, K ** -0.5, dtype)
    b, d = _rand((N,), 3, dtype=dtype), _rand((M, N), 4, dtype=dtype)
    want = oracle.torch_gemm("gemm_rcr_bias_add", x, w, b, d).to(dtype).float()
    for pitch in (K, K + 3):
        xb = torch.full((M * pitch + 1,), float("nan"), dtype=dtype, device="cuda")
        wb = torch.full((N * pitch + 1,), float("nan"), dtype=dtype, device="cuda")
        xv, wv = (t[1:].view(-1, pitch)[:, :K] for t in (xb, wb))
        xv.copy_(x)
        wv.copy_(w)
        ran = 0
        for algo, name in _instances(4, dt):
            if not lib.aitamd_gemm_algo_supported(4, dt, algo, M, N, K, pitch, pitch, 2):
                continue
            print(f"case instance={name} M={M} N={N} K={K} pitch={pitch}", flush=True)
            got = eager.gemm("gemm_rcr_bias_add", xv, wv, b.cuda(), d.cuda(), algo=algo)
            tol = 1e-2 if dt == 0 else 3e-2
            torch.testing.assert_close(got.cpu().float(), want, atol=tol, rtol=tol)
            ran += 1
        assert ran >= 4


@pytest.mark.parametrize("layout", ["rcr", "rrr", "ccr", "crr"])
@pytest.mark.parametrize("B,M,N,K", [(3, 127, 129, 65), (2, 257, 33, 1), (5, 9, 255, 130), (1, 64, 64, 64)])
def test_layouts_at_any_element(layout, B, M, N, K):
    lib = _kernels.load()
    lay = _kernels.LAYOUT_ID[layout]
    a = _rand((B, K, M) if layout[0] == "c" else (B, M, K), 1)
    b = _rand((B, N, K) if layout[1] == "c" else (B, K, N), 2, K ** -0.5)
    want = oracle.torch_bmm(layout, a, b).half().float()
    ad, bd = a.cuda(), b.cuda()
    ran = 0
    for algo, name in _instances(0, 0):
        if not lib.aitamd_gemm_algo_supported_layout(0, 0, lay, algo, M, N, K, a.shape[2], b.shape[2], 2):
            continue
        print(f"case bmm_{layout} instance={name} B={B} M={M} N={N} K={K}", flush=True)
        torch.testing.assert_close(eager.bmm(layout, ad, bd, algo=algo).cpu().float(), want, atol=1e-2, rtol=1e-2)
        ran += 1
    assert ran >= 3


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("layout", ["rcr", "rrr", "ccr", "crr"])
@pytest.mark.parametrize("B,M,N,K", [(3, 127, 129, 65), (2, 33, 255, 7), (2, 64, 64, 128)])
def test_layouts_between_guards(layout, B, M, N, K, dtype):
    """Operands one element into their buffers, rows 3 and batches 5 elements apart, NaN in every gap: only the operands
    count.  The result's buffer keeps what lies around and between its rows."""
    lib = _kernels.load()
    lay, dt = _kernels.LAYOUT_ID[layout], 0 if dtype == torch.float16 else 1
    a = _rand((B, K, M) if layout[0] == "c" else (B, M, K), 1, dtype=dtype)
    b = _rand((B, N, K) if layout[1] == "c" else (B, K, N), 2, K ** -0.5, dtype)
    want = oracle.torch_bmm(layout, a, b).to(dtype).float()
    tol = 1e-2 if dt == 0 else 3e-2

    def placed(shape, fill):
        pitch = shape[2] + 3
        stride = shape[1] * pitch + 5
        buffer = torch.full((1 + shape[0] * stride,), fill, dtype=dtype, device="cuda")
        return buffer, buffer[1:].as_strided(shape, (stride, pitch, 1), 1), pitch, stride

    _, av, lda, sa = placed(a.shape, float("nan"))
    _, bv, ldb, sb = placed(b.shape, float("nan"))
    av.copy_(a)
    bv.copy_(b)
    ran = 0
    for algo, name in _instances(0, dt):
        if not lib.aitamd_gemm_algo_supported_layout(0, dt, lay, algo, M, N, K, lda, ldb, 2):
            continue
        print(f"case bmm_{layout} instance={name} B={B} M={M} N={N} K={K} {dtype}", flush=True)
        buffer, cv, ldc, sc = placed((B, M, N), 7.0)
        rc = lib.aitamd_bmm(lay, dt, algo, av.data_ptr(), bv.data_ptr(), cv.data_ptr(), B, M, N, K, lda, ldb, ldc, sa, sb, sc, 0,
                            torch.cuda.current_stream().cuda_stream)
        _kernels.check(rc, name)
        torch.testing.assert_close(cv.cpu().float(), want, atol=tol, rtol=tol)
        cv.fill_(7.0)
        assert (buffer == 7.0).all(), name
        ran += 1
    assert ran >= 3


# AITAMD_PROF_ALGO asks for one instance: it is timed also where the profiler by itself would leave it out
@pytest.mark.parametrize("part,M,N,K", [("_k2", 64, 128, 256), ("rows", 128, 128, 256)])
def test_profiler_times_the_instance_asked_for(part, M, N, K):
    lib = _kernels.load()
    name = next(n for i, n in enumerate(_kernels.gemm_algo_names(0, 0)) if part in n and "splitk" not in n
                and lib.aitamd_gemm_algo_supported(0, 0, i, M, N, K, K, K, 16))
    out = subprocess.run([os.path.join(os.path.dirname(_kernels.KERNEL_LIB_PATH), "aitamd_profiler"), "gemm", "gemm_rcr", "0", str(M),
                          str(N), str(K)], env={**os.environ, "AITAMD_PROF_ALGO": name}, stdout=subprocess.PIPE, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.startswith(f"OP:{name},TIME:") and out.stdout.count("OP:") == 1, out.stdout
