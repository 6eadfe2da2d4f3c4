"""The kernels that the dense GEMM chooses by size: few rows of A (up to 32) and tiles of 64x64 and 128x128, at the edges of
their tiles and of their rules, against the CPU oracle.

fp32 results: the products of FP4 values and power-of-two scales are exact, so only the order of the fp32 sums differs: 1e-5
(as in test_gpu_gemm.py).  bf16 results: one rounding, at most 2^-8 of the value: 4e-3.
"""
import pytest
import torch

import oracle as O
from tests.helpers import randn_outliers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = {torch.float32: 1e-5, torch.bfloat16: 4e-3}


@pytest.fixture(scope="module")
def m():
    import alto_amd.mxfp4 as mod
    assert torch.cuda.is_available()
    return mod


def check(m, M, N, K, b_2d, dtype, strided_scales=False):
    aq, as_ = O.quantize(randn_outliers((M, K), torch.bfloat16, seed=M + K))
    bq, bs = O.quantize(randn_outliers((N, K), torch.bfloat16, seed=N + K) * 0.02, is_2d_block=b_2d)
    ref = O.gemm_ref(aq, as_, bq, bs, use_2dblock_b=b_2d, trans_b=True)
    das, dbs = as_.to(DEV), bs.to(DEV)
    if strided_scales:   # scale rows without unit stride along K
        das, dbs = das.t().contiguous().t(), dbs.t().contiguous().t()
    print(f"gemm {M}x{N}x{K} 2d={b_2d} {dtype} strided={strided_scales}", flush=True)
    for out_scale in (1.0, 0.75):
        c = m.blockwise_mxfp4_gemm(aq.to(DEV), das, bq.to(DEV), dbs, use_2dblock_b=b_2d, trans_b=True, output_dtype=dtype, out_scale=out_scale)
        assert c.shape == (M, N) and c.dtype == dtype
        assert O.rel_frobenius(c.cpu(), ref * out_scale) < TOL[dtype]


@pytest.mark.parametrize("M", [1, 15, 16, 17, 32])
@pytest.mark.parametrize("N,K,b_2d", [(16, 32, False), (64, 512, True), (77, 544, False), (5, 2080, False), (96, 1504, True), (6160, 64, False), (10304, 96, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gemm_few_rows(m, M, N, K, b_2d, dtype):
    check(m, M, N, K, b_2d, dtype, strided_scales=(M == 17))


# (33..127 rows, short reductions and narrow results ran on the fallback kernel alone)
@pytest.mark.parametrize("M,N,K,b_2d", [(33, 64, 32, True), (64, 72, 480, False), (65, 64, 512, True), (129, 136, 544, False), (40, 8, 2880, False),
                                        (500, 264, 736, False), (1100, 1064, 64, False), (1100, 1088, 1056, True), (2100, 1000, 288, False), (96, 4104, 2528, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gemm_small_tiles(m, M, N, K, b_2d, dtype):
    check(m, M, N, K, b_2d, dtype)


@pytest.mark.parametrize("K", [512, 608, 1376])
@pytest.mark.parametrize("packed", [False, True])
def test_gemm_tiles_of_every_size_give_the_same_bits(m, K, packed):
    """Rows of one product: 2304 x 2560 takes the 256x256 tile, its first 1000 rows the 128x128 tile, its first 500 the 64x64 tile."""
    from alto_amd.mxfp4.linear import gemm_packed, pack_scales
    N = 2560
    aq, as_ = m.convert_to_mxfp4(randn_outliers((2304, K), torch.bfloat16, seed=K).to(DEV))
    bq, bs = m.convert_to_mxfp4(randn_outliers((N, K), torch.bfloat16, seed=7).to(DEV))
    def product(rows):
        if packed:
            return gemm_packed(aq[:rows], pack_scales(as_[:rows], rows, K), bq, pack_scales(bs, N, K))
        return m.blockwise_mxfp4_gemm(aq[:rows], as_[:rows], bq, bs, trans_b=True, output_dtype=torch.bfloat16)
    whole = product(2304)
    assert torch.equal(product(1000), whole[:1000])
    assert torch.equal(product(500), whole[:500])


# Every ending of the reduction that the 256x128 tile has a kernel for, ragged rows and columns
@pytest.mark.parametrize("K", [512, 544, 640, 704, 768, 832, 864, 960, 1024, 1184])
def test_gemm_narrow_tile(m, K):
    """Packed scales: 2304 x 4104 takes the 256x256 tile (297 tiles of 256x128), its first 1791 rows the 256x128 tile (231)."""
    from alto_amd.mxfp4.linear import gemm_packed, pack_scales
    M, N, rows = 2304, 4104, 1791
    a, b = randn_outliers((M, K), torch.bfloat16, seed=K), randn_outliers((N, K), torch.bfloat16, seed=K + 1)
    aq, as_ = m.convert_to_mxfp4(a.to(DEV))
    bq, bs = m.convert_to_mxfp4(b.to(DEV))
    def product(r, out_scale=1.0):
        return gemm_packed(aq[:r], pack_scales(as_[:r], r, K), bq, pack_scales(bs, N, K), out_scale)
    print(f"narrow {rows}x{N}x{K}", flush=True)
    got = product(rows)
    assert torch.equal(got, product(M)[:rows])
    for i0 in (0, rows - 96):   # (the oracle takes a while for all of it)
        ref = O.gemm_ref(aq[i0:i0 + 96].cpu(), as_[i0:i0 + 96].cpu(), bq.cpu(), bs.cpu(), trans_b=True)
        assert O.rel_frobenius(got[i0:i0 + 96].cpu(), ref) < TOL[torch.bfloat16]
        assert O.rel_frobenius(product(rows, 0.75)[i0:i0 + 96].cpu(), ref * 0.75) < TOL[torch.bfloat16]


@pytest.mark.parametrize("K", [512, 544, 640, 704, 768, 832, 864, 960, 1024, 1184])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,b_2d", [(4104, False), (4128, True)])
def test_gemm_narrow_tile_plain_scales(m, K, dtype, N, b_2d):
    """1791 rows take the 256x128 tile, 100 of them at a time the 64x64 tile."""
    rows = 1791
    a, b = randn_outliers((rows, K), torch.bfloat16, seed=K), randn_outliers((N, K), torch.bfloat16, seed=K + 1)
    aq, as_ = m.convert_to_mxfp4(a.to(DEV))
    bq, bs = m.convert_to_mxfp4(b.to(DEV), is_2d_block=b_2d)
    def product(i, j):
        return m.blockwise_mxfp4_gemm(aq[i:j], as_[i:j], bq, bs, use_2dblock_b=b_2d, trans_b=True, output_dtype=dtype)
    print(f"narrow {rows}x{N}x{K}", flush=True)
    got = product(0, rows)
    for i0 in range(0, rows, 100):
        assert torch.equal(got[i0:i0 + 100], product(i0, i0 + 100)), i0
    ref = O.gemm_ref(aq[-96:].cpu(), as_[-96:].cpu(), bq.cpu(), bs.cpu(), use_2dblock_b=b_2d, trans_b=True)   # (the oracle takes a while for all of it)
    assert O.rel_frobenius(got[-96:].cpu(), ref) < TOL[dtype]


# Both sides of the lines where a short reduction goes to the direct kernel, to the kernel for few rows (16, 32 or 64 columns per
# workgroup) or to the small tiles
@pytest.mark.parametrize("M,N,K", [(16, 6144, 288), (16, 6144, 320), (17, 6144, 384), (17, 6144, 416), (1, 6160, 480), (1, 6160, 512), (32, 6160, 544),
                                   (32, 6160, 576), (16, 10256, 512), (17, 10256, 512), (16, 10256, 544), (17, 10256, 544), (16, 10256, 992), (32, 10256, 1056),
                                   (3328, 1024, 256), (3456, 1024, 256), (3456, 1024, 384), (3328, 1024, 416), (3456, 1024, 416), (3456, 2048, 224),
                                   (3328, 2048, 288), (3456, 2048, 288), (3456, 2048, 384), (3328, 2048, 416), (3456, 2048, 416)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gemm_short_reductions(m, M, N, K, dtype):
    check(m, M, N, K, N % 32 == 0, dtype, strided_scales=(M == 17))


def test_gemm_short_reduction_of_many_rows(m):
    """More rows than a grid dimension of the direct kernel has 64-row groups for."""
    M, N, K = 65535 * 64 + 96, 8, 32
    aq = torch.randint(0, 256, (M, K // 2), dtype=torch.uint8, device=DEV, generator=torch.Generator(DEV).manual_seed(1))
    as_ = torch.full((M, 1), 126, dtype=torch.uint8, device=DEV)
    bq, bs = m.convert_to_mxfp4(randn_outliers((N, K), torch.bfloat16, seed=7).to(DEV))
    c = m.blockwise_mxfp4_gemm(aq, as_, bq, bs, trans_b=True)
    for lo in (0, M - 200):
        part = m.blockwise_mxfp4_gemm(aq[lo:lo + 200], as_[lo:lo + 200], bq, bs, trans_b=True)
        assert O.rel_frobenius(c[lo:lo + 200].cpu(), part.cpu()) < TOL[torch.float32]
