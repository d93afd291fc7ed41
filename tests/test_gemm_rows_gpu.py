"""The kernel for few output elements (csrc/gemm_kernel_rows.hpp): exact sums at the edges of its 16 x 16 tiles and of its
128- and 120-deep groups of K, with operands at any element in memory that is NaN around them."""
import pytest
import torch

from aitemplate_amd import _kernels, eager

pytestmark = pytest.mark.gpu


def _rows_algos(epi, dtype, M, N, K, align):
    lib = _kernels.load()
    algos = [(i, n) for i, n in enumerate(_kernels.gemm_algo_names(epi, dtype)) if "rows16x16" in n]
    assert len(algos) == 2
    return [(i, n) for i, n in algos if lib.aitamd_gemm_algo_supported(epi, dtype, i, M, N, K, K, K, align)]


def _integers(offset, *shape, dtype):
    """Integers from -2 to 2 (exact in both types, and so are their sums in 32 bits), `offset` elements into a buffer of NaN."""
    n = 1
    for s in shape:
        n *= s
    buffer = torch.full((n + 64,), float("nan"), device="cuda", dtype=dtype)
    t = buffer[offset:offset + n].view(*shape)
    return t.copy_(torch.randint(-2, 3, shape, device="cuda"))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K", [1, 2, 7, 8, 119, 120, 121, 127, 128, 129, 130, 480, 482, 511, 512, 513, 514, 960, 961, 1026, 2049])
def test_exact_sums_at_the_edges(K, dtype):
    torch.manual_seed(K)
    ran = set()
    for M, N in ((1, 1), (4, 17), (5, 16), (16, 33), (17, 100)):
        for off_a, off_b in ((0, 0), (1, 1), (1, 0), (2, 2)):
            a, b = _integers(off_a, M, K, dtype=dtype), _integers(off_b, N, K, dtype=dtype)
            bias, d0, d1 = (torch.randint(-2, 3, s, device="cuda").to(dtype) for s in ((N,), (M, N), (M, N)))
            align = 2 if K % 2 or off_a % 2 or off_b % 2 else 4
            for op, epi, more in (("gemm_rcr", 0, ()), ("gemm_rcr_bias_add_add", 5, (bias, d0, d1))):
                want = (a.double() @ b.double().t() + sum(x.double() for x in more)).to(dtype)
                for algo, name in _rows_algos(epi, 0 if dtype == torch.float16 else 1, M, N, K, align):
                    got = eager.gemm(op, a, b, *more, algo=algo)
                    assert torch.equal(got, want), (name, M, N, K, off_a, off_b, op)
                    ran.add(name)
    assert len(ran) == (1 if K % 2 else 2)


@pytest.mark.parametrize("B,M,N,K", [(3, 5, 40, 200), (2, 33, 17, 121)])
def test_batches(B, M, N, K):
    torch.manual_seed(0)
    a, b = _integers(0, B, M, K, dtype=torch.float16), _integers(0, B, N, K, dtype=torch.float16)
    want = (a.double() @ b.double().transpose(1, 2).contiguous()).half()
    for algo, name in _rows_algos(0, 0, M, N, K, 4 if K % 2 == 0 else 2):
        assert torch.equal(eager.bmm("rcr", a, b, algo=algo), want), name


def test_an_infinity_behind_a_group_stays_in_its_place():
    """The last piece of a group of rows at odd elements belongs to the next one: it is not multiplied twice."""
    a, b = (torch.ones(n, 241, device="cuda", dtype=torch.float16) for n in (2, 3))
    a[0, 125], b[1, 125] = float("inf"), 0.5
    a[1, 126], b[2, 126] = float("nan"), 0.0
    want = a.float() @ b.float().t()
    for algo, name in _rows_algos(0, 0, 2, 3, 241, 2):
        torch.testing.assert_close(eager.gemm("gemm_rcr", a, b, algo=algo).float(), want, equal_nan=True, atol=0, rtol=0)
