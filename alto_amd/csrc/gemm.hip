// Block-scaled MXFP4 GEMM entry point (dense): C[M][N] = A[M][K] . B[N][K]^T on gfx950 scaled MFMA.
#include "common.h"
#include "gemm_simple.h"
#include "gemm_tiled.h"

namespace alto {
namespace {

template <typename OutT>
__global__ __launch_bounds__(256) void gemm_simple_kernel(OperandView A, OperandView B, int64_t M, int64_t N, int G,
                                                          OutT* c, int64_t ldc, float out_scale) {
  const int wave = threadIdx.x >> 6;
  const int64_t m0 = (int64_t)blockIdx.y * 64 + (wave >> 1) * 32;
  const int64_t n0 = (int64_t)blockIdx.x * 64 + (wave & 1) * 32;
  if (m0 >= M || n0 >= N) return;
  v16f_t acc = mma_tile_32x32(A, B, m0, n0, 0, M, N, 0, G);
  store_tile_32x32<OutT>(acc, c, ldc, m0, n0, 0, M, N, out_scale);
}

// Reductions shorter than the 512 of the 256x256 tile take the direct kernel, which starts its MFMAs after one trip to memory,
// until there is enough work to fill the ring of the 64x64 or 128x128 tile and empty it again.  us, direct / tiles:
//   M x N \ K, bf16          64          192         256         320         416         480
//   33 x 4096            3.1/4.3     3.3/4.3     3.8/4.3     3.7/4.5     4.1/4.5     4.3/4.5
//   500 x 4096           3.7/5.8     4.1/5.8     5.6/5.8     4.9/6.2     5.6/6.2     6.0/6.3
//   1024 x 4096          4.9/7.8     5.9/7.9     8.5/7.8     7.4/8.4     9.0/8.4     9.7/8.6     256 tiles of 128
//   2048 x 4096          7.9/11.0    8.9/11.1   13.9/11.1   11.8/11.5   14.9/11.6   16.4/12.1    512
//   8192 x 4096         19.2/31.3   23.9/31.3   43.5/31.6   39.6/34.2   55.3/34.7   62.6/34.8
//   2048 x 4096, fp32    8.7/14.9    9.8/15.1   15.4/15.1   12.8/15.7   16.2/16.1   17.8/16.4
//   8192 x 4096, fp32   22.9/43.9   24.8/44.3   45.5/44.3   41.1/47.5   57.5/48.0   64.5/48.7
// (K = 256: the direct kernel's lanes read rows that are all exactly one 128-byte line apart.)
bool direct_pays(int64_t M, int64_t N, int64_t K, int c_dtype) {
  if (K >= 512) return false;
  const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128);
  if (c_dtype == ALTO_DT_F32) return tiles < 432 || K < 416;
  if (K == 256 || K >= 416) return tiles < 216;
  return tiles < 432 || K < 256;
}

}  // namespace
}  // namespace alto

extern "C" int alto_mxfp4_gemm(const uint8_t* a, int64_t lda, const uint8_t* a_scales, int64_t a_ss_r, int64_t a_ss_k, int a_is_2d,
                               const uint8_t* b, int64_t ldb, const uint8_t* b_scales, int64_t b_ss_r, int64_t b_ss_k, int b_is_2d,
                               int64_t M, int64_t N, int64_t K, void* c, int c_dtype, int64_t ldc, float out_scale, void* stream) {
  using namespace alto;
  ALTO_REQUIRE(a && b && a_scales && b_scales && c, "gemm: NULL pointer");
  ALTO_REQUIRE(M >= 0 && N >= 0 && K >= 0, "gemm: negative size");
  ALTO_REQUIRE(K % 32 == 0, "gemm: K (%lld) must be a multiple of 32", (long long)K);
  ALTO_REQUIRE(!a_is_2d || M % 32 == 0, "gemm: 2D scales for A need M (%lld) %% 32 == 0", (long long)M);
  ALTO_REQUIRE(!b_is_2d || N % 32 == 0, "gemm: 2D scales for B need N (%lld) %% 32 == 0", (long long)N);
  ALTO_REQUIRE(lda >= K / 2 && ldb >= K / 2 && lda % 16 == 0 && ldb % 16 == 0, "gemm: lda/ldb must be >= K/2 and multiples of 16 bytes");
  ALTO_REQUIRE(((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15) == 0, "gemm: a and b must be 16-byte aligned");
  ALTO_REQUIRE(ldc >= N, "gemm: ldc < N");
  ALTO_REQUIRE(a_ss_r >= 0 && a_ss_k >= 0 && b_ss_r >= 0 && b_ss_k >= 0, "gemm: negative scale stride");
  ALTO_REQUIRE(c_dtype == ALTO_DT_BF16 || c_dtype == ALTO_DT_F32, "gemm: bad c_dtype %d", c_dtype);
  ALTO_REQUIRE((reinterpret_cast<uintptr_t>(c) & (c_dtype == ALTO_DT_F32 ? 3 : 1)) == 0, "gemm: c must be aligned to its element size");
  ALTO_REQUIRE(M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31), "gemm: size out of range");
  if (M == 0 || N == 0) return ALTO_MXFP4_OK;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  OperandView A{a, lda, a_scales, a_ss_r, a_ss_k, a_is_2d};
  OperandView B{b, ldb, b_scales, b_ss_r, b_ss_k, b_is_2d};

  if (gemm_skinny_supported(A, B, M, N, K) && gemm_skinny_pays(M, N, K)) {
    gemm_skinny_launch(A, B, M, N, K, c, c_dtype, ldc, out_scale, st);
    return check_launch("gemm(skinny)");
  }
  if (!(direct_pays(M, N, K, c_dtype) && (M + 63) / 64 <= 65535)) {
    const bool tiled = gemm_tiled_supported(A, B, M, N, K, c, c_dtype, ldc);
    int tile = gemm_mid_tile_size(M, N, c_dtype);
    if (tile == 256 && !tiled) tile = 128;   // (a long, narrow result or a short reduction)
    if (tile != 256 && gemm_mid_supported(A, B, M, N, K, c, ldc)) {
      gemm_mid_launch(tile, A, B, M, N, K, c, c_dtype, ldc, out_scale, false, st);
      return check_launch("gemm(mid)");
    }
    if (tiled) {
      gemm_tiled_launch(A, B, M, N, K, c, c_dtype, ldc, out_scale, st);
      return check_launch("gemm(tiled)");
    }
  }
  dim3 grid((unsigned)((N + 63) / 64), (unsigned)((M + 63) / 64));
  ALTO_REQUIRE(grid.y <= 65535u, "gemm: M too large for the fallback kernel");
  if (c_dtype == ALTO_DT_BF16)
    hipLaunchKernelGGL(gemm_simple_kernel<__bf16>, grid, dim3(256), 0, st, A, B, M, N, (int)(K / 32), (__bf16*)c, ldc, out_scale);
  else
    hipLaunchKernelGGL(gemm_simple_kernel<float>, grid, dim3(256), 0, st, A, B, M, N, (int)(K / 32), (float*)c, ldc, out_scale);
  return check_launch("gemm");
}

extern "C" int64_t alto_mxfp4_packed_scales_bytes(int64_t rows, int64_t K) {
  if (rows < 0 || K < 0 || K % 32 != 0) return 0;
  const int64_t blocks = (K / 32 + 15) / 16;
  return alto::product_below(INT64_MAX, blocks, rows, 16) ? blocks * rows * 16 : 0;
}

extern "C" int alto_mxfp4_pack_scales(const uint8_t* scales, int64_t ss_r, int64_t ss_k, int is_2d, int64_t rows, int64_t K, uint8_t* packed, void* stream) {
  using namespace alto;
  ALTO_REQUIRE(scales && packed, "pack_scales: NULL pointer");
  ALTO_REQUIRE(rows >= 0 && K >= 0 && K % 32 == 0, "pack_scales: K (%lld) must be a multiple of 32", (long long)K);
  ALTO_REQUIRE(!is_2d || rows % 32 == 0, "pack_scales: 2D scales need rows (%lld) %% 32 == 0", (long long)rows);
  ALTO_REQUIRE((reinterpret_cast<uintptr_t>(packed) & 15) == 0, "pack_scales: packed must be 16-byte aligned");
  ALTO_REQUIRE((K / 32 + 15) / 16 <= 65535 && rows < (1ll << 31), "pack_scales: size out of range");
  if (rows == 0 || K == 0) return ALTO_MXFP4_OK;
  pack_scales_launch(scales, ss_r, ss_k, is_2d, rows, K / 32, packed, reinterpret_cast<hipStream_t>(stream));
  return check_launch("pack_scales");
}

extern "C" int alto_mxfp4_gemm_ps(const uint8_t* a, int64_t lda, const uint8_t* a_packed, const uint8_t* b, int64_t ldb, const uint8_t* b_packed,
                                  int64_t M, int64_t N, int64_t K, void* c, int64_t ldc, float out_scale, void* stream) {
  using namespace alto;
  ALTO_REQUIRE(a && b && a_packed && b_packed && c, "gemm_ps: NULL pointer");
  ALTO_REQUIRE(M >= 0 && N >= 0 && K >= 0 && K % 32 == 0, "gemm_ps: K (%lld) must be a multiple of 32", (long long)K);
  ALTO_REQUIRE(lda >= K / 2 && ldb >= K / 2 && lda % 16 == 0 && ldb % 16 == 0, "gemm_ps: lda/ldb must be >= K/2 and multiples of 16 bytes");
  ALTO_REQUIRE(((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(a_packed) | reinterpret_cast<uintptr_t>(b_packed)) & 15) == 0,
               "gemm_ps: a, b and their packed scales must be 16-byte aligned");
  ALTO_REQUIRE(ldc >= N, "gemm_ps: ldc < N");
  ALTO_REQUIRE(M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31), "gemm_ps: size out of range");
  if (M == 0 || N == 0) return ALTO_MXFP4_OK;
  const int64_t KB = (K / 32 + 15) / 16;
  OperandView A{a, lda, a_packed, 16, M * 16, 0};
  OperandView B{b, ldb, b_packed, 16, N * 16, 0};
  // All three tile sizes read packed scales; the shapes are those that the 256x256 tile can serve (which of the three runs is a matter
  // of speed: same bits).  Fewer than 128 rows or 512 K take plain scales.
  OperandView Ap{a, lda, a_packed, 1, 1, 0}, Bp{b, ldb, b_packed, 1, 1, 0};
  if (!(gemm_tiled_supported(Ap, Bp, M, N, K, c, ALTO_DT_BF16, ldc) && product_below(1ll << 31, KB, M, 16) && product_below(1ll << 31, KB, N, 16))) {
    set_error("gemm_ps: shape (%lld, %lld, %lld) is not served by the tile kernels; use alto_mxfp4_gemm with plain scales", (long long)M, (long long)N, (long long)K);
    return ALTO_MXFP4_ENOTIMPL;
  }
  const int tile = gemm_mid_tile_size(M, N, ALTO_DT_BF16);
  if (tile != 256) gemm_mid_launch(tile, A, B, M, N, K, c, ALTO_DT_BF16, ldc, out_scale, true, reinterpret_cast<hipStream_t>(stream));
  else gemm_tiled_launch_ps(A, B, M, N, K, c, ldc, out_scale, reinterpret_cast<hipStream_t>(stream));
  return check_launch("gemm_ps");
}
