// MXFP4 GEMM for gfx950 on 128x128 and 64x64 tiles (dense entry): see gemm_mid.h.
#include "gemm_mid.h"
#include "gemm_tiled.h"

namespace alto {
namespace {

template <typename OutT, typename T, bool PS>
__device__ __forceinline__ void mid_tile_of(const GemmProblem& q, int wg, int tiles_m, int tiles_n, uint8_t* smem) {
  int tm, tn;
  if (!tile_coords(wg, tiles_m, tiles_n, tm, tn)) return;
  TileArgs ta{q.A, q.B, (int64_t)tm * T::TM, (int64_t)tn * T::TN, 0, q.M, q.N, q.G, q.out_scale, (q.M - 1) * q.A.ld + q.G * 16, (q.N - 1) * q.B.ld + q.G * 16, 0, 0, 0, q.G};
  gemm_mid_tile<OutT, T, PS>(ta, static_cast<OutT*>(q.c), q.ldc, smem);
}

template <typename OutT, typename T, bool PS>
__global__ __launch_bounds__(T::THREADS, 2) void gemm_mid_kernel(GemmProblem q, int tiles_m, int tiles_n) {
  __shared__ __align__(16) uint8_t smem[T::LDS];
  mid_tile_of<OutT, T, PS>(q, (int)blockIdx.x, tiles_m, tiles_n, smem);
}

// (a kernel of its own: the choice of the product costs a single one 0.3 us, 3..5 % of the small ones)
template <typename OutT, typename T, bool PS>
__global__ __launch_bounds__(T::THREADS, 2) void gemm_mid_two_kernel(GemmPair p) {
  __shared__ __align__(16) uint8_t smem[T::LDS];
  const int k = (int)blockIdx.x >= p.before;
  mid_tile_of<OutT, T, PS>(p.g[k], (int)blockIdx.x - (k ? p.before : 0), p.tiles_m[k], p.tiles_n[k], smem);
}

template <typename OutT, typename T, bool PS>
void launch_mid(const GemmProblem& p, const GemmProblem* q, hipStream_t st) {
  if (q) {
    unsigned workgroups;
    const GemmPair pair = pair_of(p, *q, T::TM, T::TN, workgroups);
    hipLaunchKernelGGL((gemm_mid_two_kernel<OutT, T, PS>), dim3(workgroups), dim3(T::THREADS), 0, st, pair);
    return;
  }
  const int tiles_m = (int)((p.M + T::TM - 1) / T::TM), tiles_n = (int)((p.N + T::TN - 1) / T::TN);
  const int per_xcd = (tiles_m * tiles_n + 7) / 8;
  hipLaunchKernelGGL((gemm_mid_kernel<OutT, T, PS>), dim3((unsigned)(per_xcd * 8)), dim3(T::THREADS), 0, st, p, tiles_m, tiles_n);
}

template <typename T>
void launch_types(const GemmProblem& p, const GemmProblem* q, int c_dtype, bool packed, hipStream_t st) {
  if (packed) launch_mid<__bf16, T, true>(p, q, st);
  else if (c_dtype == ALTO_DT_BF16) launch_mid<__bf16, T, false>(p, q, st);
  else launch_mid<float, T, false>(p, q, st);
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
// kernel is as fast with half of the units idle (and up to 256 tiles of 256x128 run there, see gemm_narrow_pays:
// 512 x 14336 x 4096 in 20.6, 2048 x 4096 x 4096 in 21.7).  With fp32 results its stores are slower and the 128x128 tile holds on
// for twice as long (2048 x 4096 x 4096: 33.3 / 30.6; 4096 x 4096 x 2048, 1024 tiles: 31.2 / 35.8).
int gemm_mid_tile_size(int64_t M, int64_t N, int c_dtype) {
  const int64_t t64 = ((M + 63) / 64) * ((N + 63) / 64), t128 = ((M + 127) / 128) * ((N + 127) / 128);
  if (t64 <= 512) return 64;
  if (t128 <= (c_dtype == ALTO_DT_F32 ? 512 : 256)) return 128;
  return 256;
}

void gemm_mid_launch(int tile, const GemmProblem& first, const GemmProblem* second, int c_dtype, bool packed, hipStream_t st) {
  if (tile == 128) launch_types<Mid128>(first, second, c_dtype, packed, st);
  else launch_types<Mid64>(first, second, c_dtype, packed, st);
}

}  // namespace alto
