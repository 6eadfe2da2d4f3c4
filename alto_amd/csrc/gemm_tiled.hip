// Tuned LDS-tiled MXFP4 GEMM for gfx950: dense entry (one 256x256 tile per 512-thread workgroup or 256x128 per 256-thread one, XCD-aware tile order).

#include "gemm_tiled.h"
#include "gemm_tile.h"

namespace alto {
namespace {

template <typename OutT, bool KTAIL, int LMS, int NST, bool PS, int WN>
__global__ __launch_bounds__(TileOf<WN>::THREADS) void gemm_tiled_kernel(OperandView A, OperandView B, int64_t M, int64_t N, int G,
                                                         OutT* c, int64_t ldc, float out_scale, int tiles_m, int tiles_n) {
  extern __shared__ __align__(16) uint8_t smem[];
  int tm, tn;
  if (!tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn)) return;
  const int KB = (G + 15) / 16;
  TileArgs ta{A, B, (int64_t)tm * GT_TM, (int64_t)tn * TileOf<WN>::TN, 0, M, N, G, out_scale,
              (M - 1) * A.ld + G * 16, (N - 1) * B.ld + G * 16,
              PS ? KB * A.ss_k : ((A.is_2d ? M / 32 : M) - 1) * A.ss_r + G, PS ? KB * B.ss_k : ((B.is_2d ? N / 32 : N) - 1) * B.ss_r + G, 0, G};
  gemm_tile_product<OutT, KTAIL, LMS, NST, PS, WN>(ta, c, ldc, smem);
}

// Two products on packed scales, bf16 results (no KTAIL: K a multiple of 512 in both).  The tiles of the second fill the units that
// the first one's last round leaves idle: 128 + 256 tiles of 2048 x 4096 x 4096 take 50.7 us in two launches, 41.6 in
// one.  Where K ends differs between the two, so a reduction runs its last 256-K stage in full (LMS = -2).
template <bool KTAIL>
__global__ __launch_bounds__(GT_THREADS) void gemm_tiled_two_kernel(GemmPair p) {
  extern __shared__ __align__(16) uint8_t smem[];
  const int k = (int)blockIdx.x >= p.before;
  const GemmProblem& q = p.g[k];
  int tm, tn;
  if (!tile_coords((int)blockIdx.x - (k ? p.before : 0), p.tiles_m[k], p.tiles_n[k], tm, tn)) return;
  const int KB = (q.G + 15) / 16;
  TileArgs ta{q.A, q.B, (int64_t)tm * GT_TM, (int64_t)tn * GT_TN, 0, q.M, q.N, q.G, q.out_scale, (q.M - 1) * q.A.ld + q.G * 16, (q.N - 1) * q.B.ld + q.G * 16,
              KB * q.A.ss_k, KB * q.B.ss_k, 0, q.G};
  gemm_tile_product<__bf16, KTAIL, -2, 4, 1>(ta, static_cast<__bf16*>(q.c), q.ldc, smem);
}

// Plain scales of one operand -> the packed form the PS kernels read: dst[(kb * rows + row) * 16 + 4 (2 h + ms) + j] =
// scale of group 16 kb + 8 ms + 2 j + h of that row, 127 beyond G.  One thread per (row, block).
__global__ __launch_bounds__(256) void pack_scales_kernel(const uint8_t* __restrict__ src, int64_t ss_r, int64_t ss_k, int is_2d, int64_t rows, int G,
                                                          uint8_t* __restrict__ dst) {
  const int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int kb = blockIdx.y;
  if (row >= rows) return;
  const uint8_t* sr = src + (is_2d ? (row >> 5) : row) * ss_r;
  uint32_t w[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const int h = d >> 1, ms = d & 1;
    uint32_t v = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int g = 16 * kb + 8 * ms + 2 * j + h;
      v |= (uint32_t)(g < G ? sr[g * ss_k] : (uint8_t)127) << (8 * j);
    }
    w[d] = v;
  }
  *reinterpret_cast<uint4*>(dst + ((int64_t)kb * rows + row) * 16) = make_uint4(w[0], w[1], w[2], w[3]);
}

template <typename OutT, bool KTAIL, int LMS = -1, int NST = 4, bool PS = false, int WN = 4>
int launch_tiled(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int64_t ldc, float out_scale, hipStream_t st) {
  using W = TileOf<WN>;
  auto kern = gemm_tiled_kernel<OutT, KTAIL, LMS, NST, PS, WN>;
  static LdsLimit lds;
  if (const int rc = lds.raise(reinterpret_cast<const void*>(kern), W::LDS, "gemm")) return rc;
  const int tiles_m = (int)((M + GT_TM - 1) / GT_TM), tiles_n = (int)((N + W::TN - 1) / W::TN);
  const int T = tiles_m * tiles_n;
  const int per_xcd = (T + 7) / 8;
  hipLaunchKernelGGL(kern, dim3((unsigned)(per_xcd * 8)), dim3(W::THREADS), W::LDS, st, A, B, M, N, (int)(K / 32), (OutT*)c, ldc, out_scale, tiles_m, tiles_n);
  return check_launch("gemm");
}

}  // namespace

bool gemm_tiled_supported(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, const void* c, int c_dtype, int64_t ldc) {
  (void)c_dtype;
  // small problems do not fill 256x256 tiles; the direct kernel handles them
  if (M < 128 || N < 128 || K < 512) return false;   // (scale rows are read 16 bytes = 512 K at a time)
  // the tile kernel reads scale rows with unit stride along K and stores C in aligned 16-byte groups
  if (A.ss_k != 1 || B.ss_k != 1) return false;
  if (!product_below(1ll << 31, M, A.ld) || !product_below(1ll << 31, N, B.ld)) return false;   // 32-bit buffer offsets
  if (!product_below(1ll << 31, M, A.ss_r) || !product_below(1ll << 31, N, B.ss_r)) return false;
  if (N % 8 != 0 || ldc % 8 != 0 || (reinterpret_cast<uintptr_t>(c) & 15) != 0) return false;
  const int64_t tiles = ((M + GT_TM - 1) / GT_TM) * ((N + GT_TN - 1) / GT_TN);
  return tiles < (1ll << 28);
}

template <int WN>   // (see TileOf)
static int launch_plain(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int c_dtype, int64_t ldc, float out_scale,
                        hipStream_t st) {
  const bool tail = (K / 32) % 16 != 0;   // K not a multiple of 512: the last scale block of a row is partial
#define ALTO_TILED_LAUNCH(T, ...) launch_tiled<T, __VA_ARGS__, false, WN>(A, B, M, N, K, c, ldc, out_scale, st)
  if (!tail) {
    if (c_dtype == ALTO_DT_BF16) return ALTO_TILED_LAUNCH(__bf16, false, -1, 4);
    else return ALTO_TILED_LAUNCH(float, false, -1, 4);
  }
  // K is known here: the kernel that ends the reduction exactly where K ends
  int lms, nst;
  gemm_tile_last_stage(K / 32, lms, nst);
#define ALTO_TILED_ENDINGS(T)                             \
  switch (lms * 4 + nst - 1) {                            \
    case 0: return ALTO_TILED_LAUNCH(T, true, 0, 1);      \
    case 1: return ALTO_TILED_LAUNCH(T, true, 0, 2);      \
    case 2: return ALTO_TILED_LAUNCH(T, true, 0, 3);      \
    case 3: return ALTO_TILED_LAUNCH(T, true, 0, 4);      \
    case 4: return ALTO_TILED_LAUNCH(T, true, 1, 1);      \
    case 5: return ALTO_TILED_LAUNCH(T, true, 1, 2);      \
    case 6: return ALTO_TILED_LAUNCH(T, true, 1, 3);      \
    default: return ALTO_TILED_LAUNCH(T, true, 1, 4);     \
  }
  if (c_dtype == ALTO_DT_BF16) {
    ALTO_TILED_ENDINGS(__bf16)
  }
  // fp32: the 256x256 tile has no registers for these; the 256x128 tile needs them: with whole blocks of 512 the products beyond K (1280 x 512 of
  // 1536) made short reductions slower than the 128x128 tile they had before, 1408 x 5160 x 1280 15.4 -> 16.1 us (now 14.5), 3585 x 2048 x 1664
  // 18.5 -> 19.4; over 187 shapes 0.92 of the time of whole blocks.
  if constexpr (WN == 2) {
    ALTO_TILED_ENDINGS(float)
  } else {
    return ALTO_TILED_LAUNCH(float, true, -1, 4);
  }
#undef ALTO_TILED_ENDINGS
#undef ALTO_TILED_LAUNCH
}

// Both operands with packed scales (A.scales / B.scales = packed base, ss_k = bytes per block), bf16 output.
template <int WN>
static int launch_ps(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int64_t ldc, float out_scale, hipStream_t st) {
  const bool tail = (K / 32) % 16 != 0;
#define ALTO_TILED_LAUNCH(...) launch_tiled<__bf16, __VA_ARGS__, true, WN>(A, B, M, N, K, c, ldc, out_scale, st)
  if (!tail) {
    return ALTO_TILED_LAUNCH(false, -1, 4);
  } else {
    int lms, nst;
    gemm_tile_last_stage(K / 32, lms, nst);
    switch (lms * 4 + nst - 1) {
      case 0: return ALTO_TILED_LAUNCH(true, 0, 1);
      case 1: return ALTO_TILED_LAUNCH(true, 0, 2);
      case 2: return ALTO_TILED_LAUNCH(true, 0, 3);
      case 3: return ALTO_TILED_LAUNCH(true, 0, 4);
      case 4: return ALTO_TILED_LAUNCH(true, 1, 1);
      case 5: return ALTO_TILED_LAUNCH(true, 1, 2);
      case 6: return ALTO_TILED_LAUNCH(true, 1, 3);
      default: return ALTO_TILED_LAUNCH(true, 1, 4);
    }
  }
#undef ALTO_TILED_LAUNCH
}

// Up to 256 tiles of 256x128, one per compute unit, that tile: each 256x256 tile's work is then done by two units at once, where the
// 256x256 tile leaves half of them idle or more.  us at 256x256 / 256x128 (same bits):
//   M x N x K             tiles of 256x128                   M x N x K             tiles of 256x128
//   1100 x 4096 x 512           160   7.9 /  6.4             1536 x 4096 x 14336         192  64.6 / 51.5
//   1376 x 4096 x 2880          192  18.3 / 15.1             2560 x 3072 x 14336         240  72.7 / 59.0
//   512 x 14336 x 4096          224  25.1 / 20.6             2048 x 4224 x 4096          264  26.6 / 36.3
//   2048 x 4096 x 1024          256  11.3 / 11.2             3000 x 3072 x 1536          288  14.4 / 19.0
//   2048 x 4096 x 4096          256  25.1 / 21.7             4096 x 4096 x 4096          512  35.9 / 41.1
// (From 257 tiles on a second round begins, and a narrow tile reads 1.5 times the bytes per product.)  Plain scales, as the inference and
// the fp32 entry points bring them: bf16 results at 256x256 / 256x128, fp32 results at 128x128 / 256x128, which is what they had:
//   M x N x K             tiles     bf16          fp32                  M x N x K             tiles     bf16          fp32
//   2048 x 4096 x 4096     256   28.3 / 23.9   30.9 / 26.8              1000 x 6144 x 1440     192   13.4 / 11.0   18.7 / 15.7
//   1376 x 4096 x 2880     192   22.1 / 17.3   25.1 / 20.9              333 x 14336 x 7200     224   54.1 / 39.2   52.7 / 40.4
//   1536 x 4096 x 14336    192   72.4 / 59.6   71.9 / 62.2              1100 x 4096 x 512      160    8.4 /  6.8   10.8 / 10.3
bool gemm_narrow_pays(int64_t M, int64_t N) { return ((M + GT_TM - 1) / GT_TM) * ((N + TileOf<2>::TN - 1) / TileOf<2>::TN) <= 256; }

int gemm_tiled_launch_ps(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int64_t ldc, float out_scale,
                         hipStream_t st) {
  return gemm_narrow_pays(M, N) ? launch_ps<2>(A, B, M, N, K, c, ldc, out_scale, st) : launch_ps<4>(A, B, M, N, K, c, ldc, out_scale, st);
}

int gemm_tiled_launch(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int c_dtype, int64_t ldc, float out_scale, hipStream_t st) {
  return gemm_narrow_pays(M, N) ? launch_plain<2>(A, B, M, N, K, c, c_dtype, ldc, out_scale, st) : launch_plain<4>(A, B, M, N, K, c, c_dtype, ldc, out_scale, st);
}

template <bool KTAIL>
static int launch_two(const GemmProblem& p, const GemmProblem& q, hipStream_t st) {
  auto kern = gemm_tiled_two_kernel<KTAIL>;
  static LdsLimit lds;
  if (const int rc = lds.raise(reinterpret_cast<const void*>(kern), GT_LDS_BYTES, "gemm_two")) return rc;
  unsigned workgroups;
  const GemmPair pair = pair_of(p, q, GT_TM, GT_TN, workgroups);
  hipLaunchKernelGGL(kern, dim3(workgroups), dim3(GT_THREADS), GT_LDS_BYTES, st, pair);
  return check_launch("gemm_two");
}

int gemm_tiled_launch_two(const GemmProblem& first, const GemmProblem& second, hipStream_t st) {
  return first.G % 16 == 0 && second.G % 16 == 0 ? launch_two<false>(first, second, st) : launch_two<true>(first, second, st);
}

void pack_scales_launch(const uint8_t* src, int64_t ss_r, int64_t ss_k, int is_2d, int64_t rows, int64_t G, uint8_t* dst, hipStream_t st) {
  const int KB = (int)((G + 15) / 16);
  hipLaunchKernelGGL(pack_scales_kernel, dim3((unsigned)((rows + 255) / 256), (unsigned)KB), dim3(256), 0, st, src, ss_r, ss_k, is_2d, rows, (int)G, dst);
}

}  // namespace alto
