"""What the library takes for a product when nothing was timed (heuristic, csrc/gemm_api.hip).  Without a device it reckons for
256 CUs."""
import pytest

from aitemplate_amd import _kernels


def _choice(epi, layout, batch, M, N, K, align):
    lda, ldb = (M if layout & 2 else K), (N if layout & 1 else K)
    algo = _kernels.load().aitamd_gemm_heuristic_algo_layout(epi, 0, layout, batch, M, N, K, lda, ldb, align)
    assert algo >= 0
    return _kernels.gemm_algo_names(epi, 0)[algo]


@pytest.mark.parametrize("epi,layout,batch,M,N,K", [
    (4, 0, 1, 6029, 3143, 3123), (5, 0, 1, 6674, 1079, 1091), (4, 0, 1, 5796, 2898, 511), (0, 1, 19, 536, 553, 995),
    (0, 1, 59, 452, 219, 109), (17, 1, 59, 452, 219, 109)])
def test_sixteen_waves_through_registers_only_with_a_cu_for_every_tile(epi, layout, batch, M, N, K):
    """A grid of more 128 x 128 tiles than CUs whose epilogue or operands a second workgroup per CU hides."""
    assert "128x128x64_w4x4_reg2" not in _choice(epi, layout, batch, M, N, K, 2)


@pytest.mark.parametrize("epi,layout,batch,M,N,K", [(4, 0, 1, 1900, 2039, 2049), (1, 0, 1, 1900, 2039, 2049)])
def test_sixteen_waves_through_registers_with_a_cu_for_every_tile(epi, layout, batch, M, N, K):
    assert "128x128x64_w4x4_reg2" in _choice(epi, layout, batch, M, N, K, 2)


@pytest.mark.parametrize("M,N,K", [(9419, 1124, 115), (9737, 3454, 217), (5900, 1527, 105), (6592, 1286, 76)])
def test_no_large_tiles_through_registers_for_few_slabs(M, N, K):
    """The fill and the store of a 256 x 256 tile have nothing beside them."""
    assert "256x256x64_w4x4_reg2" not in _choice(1, 0, 1, M, N, K, 4 if K % 2 == 0 else 2)


@pytest.mark.parametrize("M,N,K", [(8192, 4097, 2049), (4096, 4095, 6001)])
def test_large_tiles_through_registers_for_many_slabs(M, N, K):
    assert "256x256x64_w4x4_reg2" in _choice(1, 0, 1, M, N, K, 2)


def test_large_tiles_through_registers_for_many_rounds():
    assert "256x256x64_w4x4_reg2" in _choice(0, 0, 321, 684, 403, 42, 4)


@pytest.mark.parametrize("M,N,K,align", [(79, 1625, 6950, 4), (1596, 76, 4274, 4), (84, 1192, 2314, 4), (51, 1389, 7242, 4)])
def test_few_outputs_kernel_not_for_several_tiles_per_cu(M, N, K, align):
    """16 x 16 tiles of more than a few hundred fetch every row of the operands many times over."""
    assert "rows16x16" not in _choice(1, 0, 1, M, N, K, align)


@pytest.mark.parametrize("M,N,K,align", [(1, 768, 768, 16), (1, 6912, 8314, 4), (8, 4096, 4096, 16), (16, 1001, 3001, 2)])
def test_few_outputs_kernel_for_one_tile_of_rows(M, N, K, align):
    assert "rows16x16" in _choice(1, 0, 1, M, N, K, align)


@pytest.mark.parametrize("M,N,K,align", [(2048, 2048, 2048, 16), (2164, 1592, 864, 16), (3785, 856, 4576, 16),
                                         (1511, 2456, 3378, 4)])
def test_a_ring_of_128_x_128_runs_on_eight_waves(M, N, K, align):
    """One 128 x 128 tile per CU at most: sixteen waves take up to 1.06 times as long."""
    assert "128x128x64_w2x4_dma4" in _choice(1, 0, 1, M, N, K, align)
