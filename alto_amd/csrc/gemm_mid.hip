// MXFP4 GEMM for gfx950 on 128x128 and 64x64 tiles (dense entry): see gemm_mid.h.
#include "gemm_mid.h"
#include "gemm_tiled.h"

namespace alto {
namespace {

template <typename OutT, typename T, bool PS>
__global__ __launch_bounds__(T::THREADS, 2) void gemm_mid_kernel(OperandView A, OperandView B, int64_t M, int64_t N, int G, OutT* c, int64_t ldc,
                                                                 float out_scale, int tiles_m, int tiles_n) {
  __shared__ __align__(16) uint8_t smem[T::LDS];
  int tm, tn;
  if (!tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn)) return;
  TileArgs ta{A, B, (int64_t)tm * T::TM, (int64_t)tn * T::TN, 0, M, N, G, out_scale, (M - 1) * A.ld + G * 16, (N - 1) * B.ld + G * 16, 0, 0, 0, G};
  gemm_mid_tile<OutT, T, PS>(ta, c, ldc, smem);
}

template <typename OutT, typename T, bool PS>
void launch_mid(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int64_t ldc, float out_scale, hipStream_t st) {
  const int tiles_m = (int)((M + T::TM - 1) / T::TM), tiles_n = (int)((N + T::TN - 1) / T::TN);
  const int per_xcd = (tiles_m * tiles_n + 7) / 8;
  hipLaunchKernelGGL((gemm_mid_kernel<OutT, T, PS>), dim3((unsigned)(per_xcd * 8)), dim3(T::THREADS), 0, st, A, B, M, N, (int)(K / 32), (OutT*)c, ldc,
                     out_scale, tiles_m, tiles_n);
}

template <typename T>
void launch_types(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int c_dtype, int64_t ldc, float out_scale,
                  bool packed, hipStream_t st) {
  if (packed) launch_mid<__bf16, T, true>(A, B, M, N, K, c, ldc, out_scale, st);
  else if (c_dtype == ALTO_DT_BF16) launch_mid<__bf16, T, false>(A, B, M, N, K, c, ldc, out_scale, st);
  else launch_mid<float, T, false>(A, B, M, N, K, c, ldc, out_scale, st);
}

}  // namespace

bool gemm_mid_supported(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, const void* c, int64_t ldc) {
  if (K <= 0 || A.ss_k != 1 || B.ss_k != 1) return false;   // scale rows with unit stride along K
  if (!product_below(1ll << 31, M, A.ld) || !product_below(1ll << 31, N, B.ld)) return false;   // 32-bit buffer offsets
  if (N % 8 != 0 || ldc % 8 != 0 || (reinterpret_cast<uintptr_t>(c) & 15) != 0) return false;   // C in aligned 16-byte groups
  return ((M + 63) / 64) * ((N + 63) / 64) < (1ll << 28);
}

// Which tile an M x N result takes.  Times in us at 256x256 / 128x128 / 64x64, packed scales, bf16 result:
//   M x N x K          tiles of 64   of 128     256     128      64
//   512 x 1024 x 1024          128       32      8.9     6.1     4.0
//   256 x 4096 x 14336         256       64     61.9    41.7    24.1
//   500 x 4096 x 4096          512      128     21.8    16.2    11.2   (plain scales)
//   768 x 4096 x 2880          768      192     17.4    12.5    14.5
//   1024 x 4096 x 4096        1024      256     23.3    16.5    20.3
//   512 x 14336 x 4096        1792      448     25.2    24.0    32.2
//   2048 x 4096 x 4096        2048      512     25.5    24.5    34.0
//   3000 x 3072 x 1536        2256      576     13.8    17.2    19.6
// A smaller tile reads its operands from L2 more often and does less with each byte, so it pays while it is what lets
// (nearly) every compute unit work: two 64x64 tiles per compute unit, then one 128x128 tile.  Beyond that the 256x256
// kernel is as fast with half of the units idle.  With fp32 results its stores are slower and the 128x128 tile holds on
// for twice as long (2048 x 4096 x 4096: 33.3 / 30.6; 4096 x 4096 x 2048, 1024 tiles: 31.2 / 35.8).
int gemm_mid_tile_size(int64_t M, int64_t N, int c_dtype) {
  const int64_t t64 = ((M + 63) / 64) * ((N + 63) / 64), t128 = ((M + 127) / 128) * ((N + 127) / 128);
  if (t64 <= 512) return 64;
  if (t128 <= (c_dtype == ALTO_DT_F32 ? 512 : 256)) return 128;
  return 256;
}

void gemm_mid_launch(int tile, const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int c_dtype, int64_t ldc, float out_scale,
                     bool packed, hipStream_t st) {
  if (tile == 128) launch_types<Mid128>(A, B, M, N, K, c, c_dtype, ldc, out_scale, packed, st);
  else launch_types<Mid64>(A, B, M, N, K, c, c_dtype, ldc, out_scale, packed, st);
}

}  // namespace alto
