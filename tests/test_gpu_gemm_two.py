"""Two products in one call: the bits of a call each, for every tile, ending of K, scale form and pairing."""
import ctypes

import pytest
import torch

from alto_amd import _lib

pytestmark = pytest.mark.gpu

_P, _I = ctypes.c_void_p, ctypes.c_int64


class Product(ctypes.Structure):
    _fields_ = ([(n, _P) for n in ("a", "a_scales", "b", "b_scales")]
                + [(n, _I) for n in ("lda", "a_ss_r", "a_ss_k", "ldb", "b_ss_r", "b_ss_k", "M", "N", "K")]
                + [("c", _P), ("ldc", _I), ("out_scale", ctypes.c_float)]
                + [(n, ctypes.c_int) for n in ("a_is_2d", "b_is_2d", "c_dtype", "packed")])


def operand(rows, K, packed, g):
    rows = max(rows, 1)   # (an empty operand still has an address)
    codes = torch.randint(0, 256, (rows, K // 2), device="cuda", dtype=torch.uint8, generator=g)
    scales = torch.randint(118, 132, (rows, K // 32), device="cuda", dtype=torch.uint8, generator=g)
    scales[rows // 2, K // 32 - 1] = 255   # one NaN scale in the last block of K: it stays in its row
    if packed:
        flat = torch.empty((K // 32 + 15) // 16 * rows * 16, device="cuda", dtype=torch.uint8)
        _lib.check(_lib.load().alto_mxfp4_pack_scales(scales.data_ptr(), K // 32, 1, 0, rows, K, flat.data_ptr(), stream()), "pack_scales")
        scales = flat
    return codes, scales


def stream():
    return torch.cuda.current_stream().cuda_stream


def product(M, N, K, packed, dtype, scale, g):
    (a, sa), (b, sb) = operand(M, K, packed, g), operand(N, K, packed, g)
    c = torch.full((max(M, 1), N), 7.0, device="cuda", dtype=dtype)
    p = Product(a.data_ptr(), sa.data_ptr(), b.data_ptr(), sb.data_ptr(), K // 2, K // 32, 1, K // 2, K // 32, 1, M, N, K, c.data_ptr(), N, scale, 0, 0,
                {torch.bfloat16: 0, torch.float32: 1}[dtype], int(packed))
    return p, c, (a, sa, b, sb)


def alone(p):
    lib = _lib.load()
    if p.packed:
        _lib.check(lib.alto_mxfp4_gemm_ps(p.a, p.lda, p.a_scales, p.b, p.ldb, p.b_scales, p.M, p.N, p.K, p.c, p.ldc, p.out_scale, stream()), "gemm_ps")
    else:
        _lib.check(lib.alto_mxfp4_gemm(p.a, p.lda, p.a_scales, p.a_ss_r, p.a_ss_k, 0, p.b, p.ldb, p.b_scales, p.b_ss_r, p.b_ss_k, 0, p.M, p.N, p.K, p.c,
                                       p.c_dtype, p.ldc, p.out_scale, stream()), "gemm")


BF, F32 = torch.bfloat16, torch.float32


@pytest.mark.parametrize("T,K,N,packed,dtype,tile", [   # tile: of the launch they share, 0: a launch each
    (512, 512, 512, (1, 1), BF, 64),       # one block of K
    (544, 520, 1056, (1, 1), BF, 64),      # ragged in every direction
    (1024, 2048, 4096, (1, 1), BF, 128),   # K a multiple of 512 in both
    (672, 2528, 7488, (1, 1), BF, 128),    # ragged
    (1024, 4096, 4096, (1, 1), BF, 256),   # K a multiple of 512 in both
    (2048, 4096, 4096, (1, 1), BF, 256),
    (4096, 2592, 2592, (1, 1), BF, 256),   # the last block of one reduction half empty
    (2144, 5696, 3008, (1, 1), BF, 256),   # both reductions end inside a block
    (2336, 4096, 4608, (1, 1), BF, 256),   # one of them
    (512, 1024, 13440, (1, 1), BF, 0),     # reductions more than 16 times apart
    (512, 10208, 13440, (1, 1), BF, 256),  # ... but both ask for the large tile
    (512, 1024, 1024, (0, 0), BF, 64),     # plain scales
    (1376, 2880, 2144, (0, 0), F32, 128),
    (2048, 4096, 4096, (0, 0), BF, 0),     # both on the large tile
    (96, 64, 1024, (0, 0), BF, 0),         # few rows and the direct kernel
    (544, 1024, 512, (1, 0), BF, 0),       # one of each
    (0, 512, 512, (0, 0), BF, 0),          # an empty product
])
def test_two_products_are_the_two_calls(T, K, N, packed, dtype, tile):
    g = torch.Generator(device="cuda").manual_seed(T + K + N)
    x, dx, keep_x = product(T, K, N, packed[0], dtype, 1.0, g)
    w, dw, keep_w = product(N, K, T, packed[1], dtype, 0.25, g) if T else product(N, K, 512, packed[1], dtype, 0.25, g)
    alone(x)
    alone(w)
    want = dx.clone(), dw.clone()
    for first, second in ((x, w), (w, x)):
        assert _lib.load().alto_mxfp4_gemm_two_tile(ctypes.byref(first), ctypes.byref(second)) == tile
        dx.fill_(7.0)
        dw.fill_(7.0)
        _lib.check(_lib.load().alto_mxfp4_gemm_two(ctypes.byref(first), ctypes.byref(second), stream()), "gemm_two")
        for got, ref in zip((dx, dw), want):
            assert torch.equal(got.view(torch.uint8), ref.view(torch.uint8))
    assert want[1].isnan().any() and not want[1].isnan().all()


def test_a_refused_product_launches_nothing():
    g = torch.Generator(device="cuda").manual_seed(1)
    x, dx, keep_x = product(512, 512, 512, 1, BF, 1.0, g)
    w, dw, keep_w = product(512, 512, 512, 1, BF, 1.0, g)
    w.ldc = 256
    with pytest.raises(AssertionError, match="ldc"):
        _lib.check(_lib.load().alto_mxfp4_gemm_two(ctypes.byref(x), ctypes.byref(w), stream()), "gemm_two")
    assert bool((dx == 7.0).all()) and bool((dw == 7.0).all())
