// Block-scaled MXFP4 GEMM entry point (dense): C[M][N] = A[M][K] . B[N][K]^T on gfx950 scaled MFMA.
#include <algorithm>

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

// Which kernel a product past its checks takes.
enum class Route { NONE, DIRECT, SKINNY, MID64, MID128, TILED };
struct GemmCall {
  GemmProblem q;
  int64_t K;
  int c_dtype;
  bool packed;
  Route route;
  bool narrow = false;   // MID128, but 256x128 tiles where the product has a launch to itself
};

int plan_gemm(const alto_mxfp4_product& p, GemmCall& g) {
  ALTO_REQUIRE(p.a && p.b && p.a_scales && p.b_scales && p.c, "gemm: NULL pointer");
  ALTO_REQUIRE(p.M >= 0 && p.N >= 0 && p.K >= 0, "gemm: negative size");
  ALTO_REQUIRE(p.K % 32 == 0, "gemm: K (%lld) must be a multiple of 32", (long long)p.K);
  ALTO_REQUIRE(!p.a_is_2d || p.M % 32 == 0, "gemm: 2D scales for A need M (%lld) %% 32 == 0", (long long)p.M);
  ALTO_REQUIRE(!p.b_is_2d || p.N % 32 == 0, "gemm: 2D scales for B need N (%lld) %% 32 == 0", (long long)p.N);
  ALTO_REQUIRE(p.lda >= p.K / 2 && p.ldb >= p.K / 2 && p.lda % 16 == 0 && p.ldb % 16 == 0, "gemm: lda/ldb must be >= K/2 and multiples of 16 bytes");
  ALTO_REQUIRE(((reinterpret_cast<uintptr_t>(p.a) | reinterpret_cast<uintptr_t>(p.b)) & 15) == 0, "gemm: a and b must be 16-byte aligned");
  ALTO_REQUIRE(p.ldc >= p.N, "gemm: ldc < N");
  ALTO_REQUIRE(p.a_ss_r >= 0 && p.a_ss_k >= 0 && p.b_ss_r >= 0 && p.b_ss_k >= 0, "gemm: negative scale stride");
  ALTO_REQUIRE(p.c_dtype == ALTO_DT_BF16 || p.c_dtype == ALTO_DT_F32, "gemm: bad c_dtype %d", p.c_dtype);
  ALTO_REQUIRE((reinterpret_cast<uintptr_t>(p.c) & (p.c_dtype == ALTO_DT_F32 ? 3 : 1)) == 0, "gemm: c must be aligned to its element size");
  ALTO_REQUIRE(p.M < (1ll << 31) && p.N < (1ll << 31) && p.K < (1ll << 31), "gemm: size out of range");
  const OperandView A{p.a, p.lda, p.a_scales, p.a_ss_r, p.a_ss_k, p.a_is_2d}, B{p.b, p.ldb, p.b_scales, p.b_ss_r, p.b_ss_k, p.b_is_2d};
  g = GemmCall{{A, B, p.M, p.N, (int)(p.K / 32), p.c, p.ldc, p.out_scale}, p.K, p.c_dtype, false, Route::NONE};
  if (p.M == 0 || p.N == 0) return ALTO_MXFP4_OK;
  if (gemm_skinny_supported(A, B, p.M, p.N, p.K) && gemm_skinny_pays(p.M, p.N, p.K)) {
    g.route = Route::SKINNY;
    return ALTO_MXFP4_OK;
  }
  if (!(direct_pays(p.M, p.N, p.K, p.c_dtype) && (p.M + 63) / 64 <= 65535)) {
    const bool tiled = gemm_tiled_supported(A, B, p.M, p.N, p.K, p.c, p.c_dtype, p.ldc);
    int tile = gemm_mid_tile_size(p.M, p.N, p.c_dtype);
    if (tile == 256 && !tiled) tile = 128;   // (a long, narrow result or a short reduction)
    if (tile != 256 && gemm_mid_supported(A, B, p.M, p.N, p.K, p.c, p.ldc)) g.route = tile == 64 ? Route::MID64 : Route::MID128;
    else if (tiled) g.route = Route::TILED;
    // (fp32: the 128x128 tile's range reaches into that of the 256x128 tile; two products that share a launch stay on 128x128)
    g.narrow = g.route == Route::MID128 && tiled && ((p.M + 127) / 128) * ((p.N + 127) / 128) > 256 && gemm_narrow_pays(p.M, p.N);
    if (g.route != Route::NONE) return ALTO_MXFP4_OK;
  }
  ALTO_REQUIRE((p.M + 63) / 64 <= 65535, "gemm: M too large for the fallback kernel");
  g.route = Route::DIRECT;
  return ALTO_MXFP4_OK;
}

int plan_gemm_ps(const alto_mxfp4_product& p, GemmCall& g) {
  ALTO_REQUIRE(p.a && p.b && p.a_scales && p.b_scales && p.c, "gemm_ps: NULL pointer");
  ALTO_REQUIRE(p.M >= 0 && p.N >= 0 && p.K >= 0 && p.K % 32 == 0, "gemm_ps: K (%lld) must be a multiple of 32", (long long)p.K);
  ALTO_REQUIRE(p.lda >= p.K / 2 && p.ldb >= p.K / 2 && p.lda % 16 == 0 && p.ldb % 16 == 0, "gemm_ps: lda/ldb must be >= K/2 and multiples of 16 bytes");
  ALTO_REQUIRE(((reinterpret_cast<uintptr_t>(p.a) | reinterpret_cast<uintptr_t>(p.b) | reinterpret_cast<uintptr_t>(p.a_scales) | reinterpret_cast<uintptr_t>(p.b_scales)) & 15) == 0,
               "gemm_ps: a, b and their packed scales must be 16-byte aligned");
  ALTO_REQUIRE(p.ldc >= p.N, "gemm_ps: ldc < N");
  ALTO_REQUIRE(p.M < (1ll << 31) && p.N < (1ll << 31) && p.K < (1ll << 31), "gemm_ps: size out of range");
  const OperandView A{p.a, p.lda, p.a_scales, 16, p.M * 16, 0}, B{p.b, p.ldb, p.b_scales, 16, p.N * 16, 0};
  g = GemmCall{{A, B, p.M, p.N, (int)(p.K / 32), p.c, p.ldc, p.out_scale}, p.K, ALTO_DT_BF16, true, Route::NONE};
  if (p.M == 0 || p.N == 0) return ALTO_MXFP4_OK;
  const int64_t KB = (p.K / 32 + 15) / 16;
  // All three tile sizes read packed scales; the shapes are those that the 256x256 tile can serve (which of the three runs is a matter
  // of speed: same bits).  Fewer than 128 rows or 512 K take plain scales.
  const OperandView Ap{p.a, p.lda, p.a_scales, 1, 1, 0}, Bp{p.b, p.ldb, p.b_scales, 1, 1, 0};
  if (!(gemm_tiled_supported(Ap, Bp, p.M, p.N, p.K, p.c, ALTO_DT_BF16, p.ldc) && product_below(1ll << 31, KB, p.M, 16) && product_below(1ll << 31, KB, p.N, 16))) {
    set_error("gemm_ps: shape (%lld, %lld, %lld) is not served by the tile kernels; use alto_mxfp4_gemm with plain scales", (long long)p.M, (long long)p.N, (long long)p.K);
    return ALTO_MXFP4_ENOTIMPL;
  }
  const int tile = gemm_mid_tile_size(p.M, p.N, ALTO_DT_BF16);
  g.route = tile == 64 ? Route::MID64 : tile == 128 ? Route::MID128 : Route::TILED;
  return ALTO_MXFP4_OK;
}

int own_tile_size(const GemmCall& g) { return g.route == Route::MID64 ? 64 : g.route == Route::MID128 ? 128 : g.route == Route::TILED ? 256 : 0; }

// The tile of two packed products that share a launch, or 0: a launch each.  The bits are the same with every tile.
// Time of a tile size: what a launch costs, and then either the longest reduction, which one workgroup walks through, or
// all the work spread over the 256 compute units, whichever takes longer.  The constants are a least-squares fit to 346
// pairs of 512..16384 x 512..14336 x 512..14336, three tile sizes each (10 % rms); the tile it names takes 1.5 % longer than the
// best one.  A pair takes 0.84 of the time of two launches with a tile each (512 x 1024 x 1024 7.4 -> 5.1 us, 2048 x 4096 x 1024 22.0 -> 19.1,
// 2048 x 4096 x 4096 50.7 -> 41.6, 4096 x 4096 x 4096 72.8 -> 71.3, 8192 x 4096 x 14336 441 -> 441), of which half comes from the tiles: a rule
// by their number alone is 7 % or more behind, because a few tiles with a long reduction want them small.
// Beyond a factor of 16 between the reductions no tile suits both unless both ask for the same one (512 x 3840 x 13440, 128 and 256:
// 69 us apart, 79..90 together).
int shared_tile_size(const GemmCall& x, const GemmCall& y) {
  const double kx = (double)x.K, ky = (double)y.K;   // kx >= ky
  if (kx > 16 * ky) return x.route == y.route ? own_tile_size(x) : 0;
  const struct { int tile; double launch, step, share, ends; } sizes[] = {   // us; ns per K of a tile alone; ns per K and tile of a full chip; a tile's ends in K
      {64, 3.4, 1.75e-3, 1.02e-3, 700}, {128, 4.0, 3.4e-3, 2.42e-3, 950}, {256, 5.2, 5.2e-3, 7.15e-3, 950}};
  int best = 0;
  double least = 0;
  for (const auto& s : sizes) {
    auto tiles = [&](const GemmProblem& q) { return (double)((q.M + s.tile - 1) / s.tile) * (double)((q.N + s.tile - 1) / s.tile); };
    const double t = s.launch + std::max(s.step * kx, s.share / 256 * (tiles(x.q) * (kx + s.ends) + tiles(y.q) * (ky + s.ends)));
    if (best == 0 || t < least) best = s.tile, least = t;
  }
  return best;
}

// The tile of the launch that two products share, longer reduction first, or 0: a launch each.
int tile_of_two(const GemmCall& x, const GemmCall& y) {
  if (x.route == Route::NONE || y.route == Route::NONE || x.packed != y.packed || x.c_dtype != y.c_dtype) return 0;
  if (x.packed) return shared_tile_size(x, y);
  const int own = x.route == y.route ? own_tile_size(x) : 0;   // (plain scales: the two small tiles, where both ask for the same one)
  return own == 256 ? 0 : own;
}

int plan_gemm_two(const alto_mxfp4_product* first, const alto_mxfp4_product* second, GemmCall (&g)[2]) {
  ALTO_REQUIRE(first && second, "gemm_two: NULL product");
  for (int i = 0; i < 2; ++i) {
    const alto_mxfp4_product& p = i ? *second : *first;
    const int rc = p.packed ? plan_gemm_ps(p, g[i]) : plan_gemm(p, g[i]);
    if (rc != ALTO_MXFP4_OK) return rc;
  }
  return ALTO_MXFP4_OK;
}

int launch_gemm(const GemmCall& g, hipStream_t st) {
  const GemmProblem& q = g.q;
  switch (g.route) {
    case Route::NONE: return ALTO_MXFP4_OK;
    case Route::SKINNY: gemm_skinny_launch(q.A, q.B, q.M, q.N, g.K, q.c, g.c_dtype, q.ldc, q.out_scale, st); break;
    case Route::MID64: case Route::MID128:
      if (g.narrow) return gemm_tiled_launch(q.A, q.B, q.M, q.N, g.K, q.c, g.c_dtype, q.ldc, q.out_scale, st);
      gemm_mid_launch(g.route == Route::MID64 ? 64 : 128, q, nullptr, g.c_dtype, g.packed, st);
      break;
    case Route::TILED:
      if (g.packed) return gemm_tiled_launch_ps(q.A, q.B, q.M, q.N, g.K, q.c, q.ldc, q.out_scale, st);
      return gemm_tiled_launch(q.A, q.B, q.M, q.N, g.K, q.c, g.c_dtype, q.ldc, q.out_scale, st);
    case Route::DIRECT: {
      const dim3 grid((unsigned)((q.N + 63) / 64), (unsigned)((q.M + 63) / 64));
      if (g.c_dtype == ALTO_DT_BF16)
        hipLaunchKernelGGL(gemm_simple_kernel<__bf16>, grid, dim3(256), 0, st, q.A, q.B, q.M, q.N, q.G, (__bf16*)q.c, q.ldc, q.out_scale);
      else
        hipLaunchKernelGGL(gemm_simple_kernel<float>, grid, dim3(256), 0, st, q.A, q.B, q.M, q.N, q.G, (float*)q.c, q.ldc, q.out_scale);
      break;
    }
  }
  return check_launch("gemm");
}

}  // namespace
}  // namespace alto

extern "C" int alto_mxfp4_gemm(const uint8_t* a, int64_t lda, const uint8_t* a_scales, int64_t a_ss_r, int64_t a_ss_k, int a_is_2d,
                               const uint8_t* b, int64_t ldb, const uint8_t* b_scales, int64_t b_ss_r, int64_t b_ss_k, int b_is_2d,
                               int64_t M, int64_t N, int64_t K, void* c, int c_dtype, int64_t ldc, float out_scale, void* stream) {
  alto::GemmCall g;
  const int rc = alto::plan_gemm({a, a_scales, b, b_scales, lda, a_ss_r, a_ss_k, ldb, b_ss_r, b_ss_k, M, N, K, c, ldc, out_scale, a_is_2d, b_is_2d, c_dtype, 0}, g);
  return rc != ALTO_MXFP4_OK ? rc : alto::launch_gemm(g, (hipStream_t)stream);
}

extern "C" int alto_mxfp4_gemm_two(const alto_mxfp4_product* first, const alto_mxfp4_product* second, void* stream) {
  using namespace alto;
  GemmCall g[2];
  int rc = plan_gemm_two(first, second, g);
  if (rc != ALTO_MXFP4_OK) return rc;
  hipStream_t st = (hipStream_t)stream;
  const bool swap = g[1].K > g[0].K;   // the longer tiles first
  const GemmCall &x = g[swap], &y = g[!swap];
  const int tile = tile_of_two(x, y);
  if (tile == 256) return gemm_tiled_launch_two(x.q, y.q, st);
  if (tile != 0) {
    gemm_mid_launch(tile, x.q, &y.q, x.c_dtype, x.packed, st);
    return check_launch("gemm_two");
  }
  rc = launch_gemm(g[0], st);
  return rc != ALTO_MXFP4_OK ? rc : launch_gemm(g[1], st);
}

extern "C" int alto_mxfp4_gemm_two_tile(const alto_mxfp4_product* first, const alto_mxfp4_product* second) {
  using namespace alto;
  GemmCall g[2];
  const int rc = plan_gemm_two(first, second, g);
  if (rc != ALTO_MXFP4_OK) return rc;
  const bool swap = g[1].K > g[0].K;
  return tile_of_two(g[swap], g[!swap]);
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
  alto::GemmCall g;
  const int rc = alto::plan_gemm_ps({a, a_packed, b, b_packed, lda, 0, 0, ldb, 0, 0, M, N, K, c, ldc, out_scale, 0, 0, ALTO_DT_BF16, 1}, g);
  return rc != ALTO_MXFP4_OK ? rc : alto::launch_gemm(g, (hipStream_t)stream);
}
