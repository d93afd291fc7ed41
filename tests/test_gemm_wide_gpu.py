"""The four-wave GEMM instances at the edges of their tiles, slab pairs and column units: K around the pairs of 64, rows
and columns around 16, 112, 128 and the tiles, fewer and more tiles than CUs, padded operands, batches, and the outputs
that the launcher sends to another instance."""
import pytest
import torch

from aitemplate_amd import _kernels, eager
from oracle import oracle

pytestmark = pytest.mark.gpu

ALIGNED = [n for n in _kernels.gemm_algo_names(2, 0) if n.endswith("_wide")]
DWORDS = [n for n in _kernels.gemm_algo_names(2, 0) if n.endswith("_wide_k2")]
assert ALIGNED and DWORDS


def _rand(shape, seed, dtype, scale=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).to(dtype)


def _algo(op, name, dtype):
    name = name.replace("_f16_", "_bf16_") if dtype == torch.bfloat16 else name
    algo = _kernels.load().aitamd_gemm_find_algo(_kernels.EPILOGUE_OF_OP[op], int(dtype == torch.bfloat16), name.encode())
    assert algo >= 0, f"{op} has no instance {name}"  # (-1 would be the automatic choice)
    return algo


def _check(op, name, M, N, K, dtype=torch.float16, pitch=0, seed=0):
    """Operands as views into NaN-filled buffers of row pitch K + `pitch`: nothing outside of them may count."""
    print(f"case op={op} instance={name} M={M} N={N} K={K} dtype={dtype} pitch=K+{pitch}", flush=True)
    x, w = _rand((M, K), seed, dtype), _rand((N, K), seed + 1, dtype, K ** -0.5)
    b, d0, d1 = (_rand(s, seed + 2 + i, dtype) for i, s in enumerate(((N,), (M, N), (M, N))))
    nres = _kernels.NUM_RESIDUALS_OF_EPILOGUE[_kernels.EPILOGUE_OF_OP[op]]
    xv, wv = (torch.full((t.shape[0], K + pitch), float("nan"), dtype=dtype, device="cuda")[:, :K] for t in (x, w))
    xv.copy_(x)
    wv.copy_(w)
    got = eager.gemm(op, xv, wv, None if op == "gemm_rcr" else b.cuda(), d0.cuda() if nres >= 1 else None,
                     d1.cuda() if nres >= 2 else None, algo=_algo(op, name, dtype))
    want = oracle.torch_gemm(op, x, w, b, d0, d1)
    # one rounding of a 32-bit result, and sums of K products of N(0, 1) x N(0, 1/K) in another order
    eps = 2.0 ** (-11 if dtype == torch.float16 else -8)
    torch.testing.assert_close(got.cpu().float(), want.float(), rtol=2 * eps, atol=2 * eps)


@pytest.mark.parametrize("name", ALIGNED)
@pytest.mark.parametrize("M,N,K", [
    (1, 8, 136),         # the smallest: three pairs, the last of 8
    (256, 256, 192),     # one tile, whole pairs
    (255, 248, 200), (257, 264, 248),  # a row or a piece short of a tile, and past it; pairs cut at every chunk
    (129, 232, 320), (127, 104, 376), (113, 120, 1024),
    (700, 120, 4104),    # many pairs, the last of 8
    (4100, 4200, 136),   # more tiles than CUs: the ring runs from tile to tile, the toggled tail with it
    (8200, 2056, 192),   # the same without a tail
])
def test_wide_shapes(name, M, N, K):
    seed = M + N + K
    _check("gemm_rcr_bias_relu", name, M, N, K, seed=seed)
    _check("gemm_rcr_bias_add_add", name, M, N, K, torch.bfloat16, pitch=8, seed=seed)
    _check("gemm_rcr_bias_add", name, M, N, K, pitch=24, seed=seed)


@pytest.mark.parametrize("name", DWORDS)
@pytest.mark.parametrize("M,N,K", [(1, 8, 138), (256, 256, 196), (255, 248, 206), (257, 264, 254), (130, 216, 1030),
                                   (4100, 4200, 142), (300, 440, 8314)])
def test_wide_dword_rows(name, M, N, K):
    _check("gemm_rcr_bias_gelu", name, M, N, K, seed=K)
    _check("gemm_rcr_bias_relu", name, M, N, K, torch.bfloat16, pitch=4, seed=K)
    _check("gemm_rcr_bias_mul_add", name, M, N, K, pitch=2, seed=K)


@pytest.mark.parametrize("name", ALIGNED + DWORDS)
@pytest.mark.parametrize("op", sorted(set(_kernels.EPILOGUE_OF_OP) - {"bmm_rcr"}))
def test_wide_every_epilogue(name, op):
    # (the bias alone: of halves below)
    dtype = torch.bfloat16 if _kernels.EPILOGUE_OF_OP[op] == 1 else torch.float16
    _check(op, name, 500, 472, 322 if name in DWORDS else 320, dtype, seed=7)


@pytest.mark.parametrize("name", ALIGNED + DWORDS)
def test_wide_bias_of_halves(name):
    for M, N, K in ((500, 472, 320), (257, 264, 136), (4100, 4200, 200)):
        _check("gemm_rcr_bias", name, M, N, K + 2 if name in DWORDS else K, pitch=8, seed=K)


@pytest.mark.parametrize("name", ALIGNED + DWORDS)
def test_wide_supported_problems(name):
    lib, k = _kernels.load(), 2 if name in DWORDS else 8
    ok = lambda N, K, align: lib.aitamd_gemm_algo_supported(2, 0, _algo("gemm_rcr_bias_relu", name, torch.float16), 64, N, K, K, K, align)
    assert ok(64, 136, 2 * k) and not ok(64, 136 + k // 2, 2 * k) and not ok(64, 136, k)
    # short K and columns that are no whole pieces: handed on to an instance that takes them
    for M, N, K in ((64, 64, 128), (300, 60, 136), (70, 59, 48)):
        assert ok(N, K, 2 * k)
        _check("gemm_rcr_bias_relu", name, M, N, K, seed=8)


@pytest.mark.parametrize("name", ALIGNED)
def test_wide_batches(name):
    for B, M, N, K in ((3, 300, 264, 200), (70, 260, 520, 192)):  # the second: more tiles than CUs
        a, b = _rand((B, M, K), 1, torch.float16), _rand((B, N, K), 2, torch.float16, K ** -0.5)
        got = eager.bmm_rcr(a.cuda(), b.cuda(), algo=_algo("gemm_rcr", name, torch.float16))
        torch.testing.assert_close(got.cpu().float(), oracle.torch_bmm_rcr(a, b).float(), rtol=2 ** -10, atol=2 ** -10)


@pytest.mark.parametrize("name", ALIGNED + DWORDS)
def test_wide_other_outputs(name):
    # odd output pitch, output and residual at an odd element: stored by the instance that takes any output
    M, N, K = 300, 264, 200
    op = "gemm_rcr_bias_add"
    x, w = _rand((M, K), 1, torch.float16), _rand((N, K), 2, torch.float16, K ** -0.5)
    b, d = _rand((N,), 3, torch.float16), _rand((M, N), 4, torch.float16)
    want = oracle.torch_gemm(op, x, w, b, d).half().float()
    for pitch, first in ((N + 1, 0), (N + 2, 1), (N, 1)):
        for odd_d in (False, True):
            buf = torch.zeros(M * pitch + 8, dtype=torch.float16, device="cuda")
            out = buf[first:first + M * pitch].view(M, pitch)[:, :N]
            dbuf = torch.zeros(M * N + 8, dtype=torch.float16, device="cuda")
            dv = dbuf[int(odd_d):int(odd_d) + M * N].view(M, N)
            dv.copy_(d)
            eager.gemm(op, x.cuda(), w.cuda(), b.cuda(), dv, out=out, algo=_algo(op, name, torch.float16))
            torch.testing.assert_close(out.cpu().float(), want, rtol=1e-2, atol=1e-2)
            assert buf[:first].abs().sum() == 0 and (pitch == N or buf[first:].view(-1)[:M * pitch].view(M, pitch)[:, N:].abs().sum() == 0)
