// Tuned LDS-tiled MXFP4 GEMM (declarations).  See gemm_tiled.hip.
#pragma once
#include "gemm_simple.h"

namespace alto {
// One product C[M][N] = A . B^T over G groups of 32, as the tile kernels take it.
struct GemmProblem {
  OperandView A, B;
  int64_t M, N;
  int G;
  void* c;
  int64_t ldc;
  float out_scale;
};

// Two products in one launch: workgroups [0, before) are the tiles of g[0], the others those of g[1].
struct GemmPair {
  GemmProblem g[2];
  int tiles_m[2], tiles_n[2];
  int before;   // a multiple of 8: the XCDs come in the same order in both
};
inline GemmPair pair_of(const GemmProblem& first, const GemmProblem& second, int tm, int tn, unsigned& workgroups) {
  GemmPair p{{first, second}, {}, {}, 0};
  int64_t wgs[2];
  for (int i = 0; i < 2; ++i) {
    p.tiles_m[i] = (int)((p.g[i].M + tm - 1) / tm);
    p.tiles_n[i] = (int)((p.g[i].N + tn - 1) / tn);
    wgs[i] = ((int64_t)p.tiles_m[i] * p.tiles_n[i] + 7) / 8 * 8;
  }
  p.before = (int)wgs[0];
  workgroups = (unsigned)(wgs[0] + wgs[1]);
  return p;
}

bool gemm_tiled_supported(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, const void* c, int c_dtype, int64_t ldc);
// (the tiled launches return the status of the call; they choose between 256x256 and 256x128 tiles by the second rule)
bool gemm_narrow_pays(int64_t M, int64_t N);
int gemm_tiled_launch(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int c_dtype, int64_t ldc,
                      float out_scale, hipStream_t st);
// Packed scales (see pack_scales_kernel): the converter, and the tiled GEMM on operands that bring them (bf16 output).
void pack_scales_launch(const uint8_t* src, int64_t ss_r, int64_t ss_k, int is_2d, int64_t rows, int64_t G, uint8_t* dst, hipStream_t st);
int gemm_tiled_launch_ps(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int64_t ldc, float out_scale,
                         hipStream_t st);
// Two of them on packed scales in one launch, the tiles of `first` first.
int gemm_tiled_launch_two(const GemmProblem& first, const GemmProblem& second, hipStream_t st);
// Few rows of A (see gemm_skinny.hip).
bool gemm_skinny_supported(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K);
bool gemm_skinny_pays(int64_t M, int64_t N, int64_t K);
void gemm_skinny_launch(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int c_dtype, int64_t ldc, float out_scale,
                        hipStream_t st);
// 128x128 and 64x64 tiles (see gemm_mid.hip): which tile a shape takes (256, 128 or 64), and the launch of the two smaller ones.
bool gemm_mid_supported(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, const void* c, int64_t ldc);
int gemm_mid_tile_size(int64_t M, int64_t N, int c_dtype);
// second (or NULL): a second product of the same result and scale type in the same launch, behind the first one's tiles.
void gemm_mid_launch(int tile, const GemmProblem& first, const GemmProblem* second, int c_dtype, bool packed, hipStream_t st);
}  // namespace alto
