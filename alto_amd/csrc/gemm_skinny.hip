// MXFP4 GEMM with few rows of A (decode steps): C[M][N] = A[M][K] . B[N][K]^T for M <= 32 on gfx950 scaled MFMA.
//
// Such a product reads B once and does nothing else of size.  A workgroup owns 16 NT columns of C (16 NT rows of B) and all
// of M; its four waves deal the reduction out among themselves in pieces of 512 K and add their accumulators through LDS
// at the end, so that every compute unit has loads in flight from the start and no wave waits for another before the end.
// Nothing is staged: a lane of v_mfma_scale_f32_16x16x128_f8f6f4 holds one MX block (16 bytes) of one row, and which block
// of the 512-K piece the lane group q = lane / 16 holds at step j is free as long as A and B agree: it is block 4 q + j,
// so that the lane's four scale bytes are one dword, of which op_sel picks byte j.  B goes in as the first operand: a
// lane's four accumulator registers are then four neighbouring columns of one row of C.
// What bounds it: neighbouring lanes read different rows, so each load instruction touches 64 lines and the address unit
// takes about 64 clocks for it (K = 14336, N = 4096: 10 us for 29 MB of B and the same of A through the L2); 8 and 16 waves
// instead of four change nothing.  16 x 4096 x 4096: 14.5 us with one 32x32 tile per wave over all of K (the fallback
// kernel, 64 workgroups), 4.6 us here; 1 x 4096 x 4096 13.2 -> 3.8; 16 x 4096 x 14336 44.7 -> 10.0; 16 x 14336 x 4096 18.0 -> 8.3.
// From 33 rows on the 64x64 tiles are as good (64 x 4096 x 4096: 8.4 / 8.3).
#include "gemm_simple.h"
#include "gemm_tiled.h"

namespace alto {
namespace {

constexpr int SK_WAVES = 4;

// One operand as the lane sees it: codes through a descriptor whose range ends with the operand, scales by row.
struct SkinnyOperand {
  __amdgpu_buffer_rsrc_t codes;
  const uint8_t* srow;   // scales of this lane's row
  int off;               // byte offset of this lane's row in the descriptor
  int64_t ss_k;

  __device__ __forceinline__ void init(const OperandView& v, int64_t row0, int rows, int row, int kbytes) {
    const uint8_t* base = v.codes + row0 * v.ld;
    codes = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), 0, (int)((rows - 1) * v.ld + kbytes), 0x00020000);
    row = row < rows ? row : rows - 1;   // rows beyond the operand repeat its last one; their results are not stored
    off = row * (int)v.ld;
    const int64_t gr = row0 + row;
    srow = v.scales + (v.is_2d ? gr >> 5 : gr) * v.ss_r;
    ss_k = v.ss_k;
  }
  // block 4 q + j of piece p, zeros beyond K (an offset with bit 31 set is out of range and reads as zeros)
  __device__ __forceinline__ v8i_t block(int p, int q, int j, int G) const {
    const int g = 16 * p + 4 * q + j;
    const v4i_t v = __builtin_amdgcn_raw_buffer_load_b128(codes, g < G ? off + 16 * g : (int)0x80000000, 0, 0);
    return v8i_t{v[0], v[1], v[2], v[3], 0, 0, 0, 0};
  }
  // the scale bytes of blocks 4 q .. 4 q + 3 of piece p; blocks beyond K read as 127
  __device__ __forceinline__ int scale4(int p, int q, int G) const {
    const int g = 16 * p + 4 * q;
    if (ss_k == 1 && 16 * p + 16 <= G) {
      int v;
      __builtin_memcpy(&v, srow + g, 4);   // (any alignment)
      return v;
    }
    uint32_t v = 0x7F7F7F7Fu;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (g + j < G) v = (v & ~(0xFFu << (8 * j))) | ((uint32_t)srow[(int64_t)(g + j) * ss_k] << (8 * j));
    return (int)v;
  }
};

template <typename OutT, int MT, int NT>
__global__ __launch_bounds__(64 * SK_WAVES) void gemm_skinny_kernel(OperandView A, OperandView B, int M, int64_t N, int G, OutT* __restrict__ c, int64_t ldc,
                                                              float out_scale) {
  __shared__ v4f_t red[SK_WAVES][MT * NT][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int64_t n0 = (int64_t)blockIdx.x * (16 * NT);
  const int nrows = N - n0 < 16 * NT ? (int)(N - n0) : 16 * NT;
  SkinnyOperand b[NT], a[MT];
#pragma unroll
  for (int u = 0; u < NT; ++u) b[u].init(B, n0, nrows, 16 * u + r, G * 16);
#pragma unroll
  for (int t = 0; t < MT; ++t) a[t].init(A, 0, M, 16 * t + r, G * 16);
  v4f_t acc[MT][NT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int u = 0; u < NT; ++u) acc[t][u] = v4f_t{0.0f, 0.0f, 0.0f, 0.0f};

  const int P = (G + 15) / 16;
  for (int p = wave; p < P; p += SK_WAVES) {
    v8i_t bv[NT][4], av[MT][4];
    int sb[NT], sa[MT];
#pragma unroll
    for (int u = 0; u < NT; ++u) {
#pragma unroll
      for (int j = 0; j < 4; ++j) bv[u][j] = b[u].block(p, q, j, G);
      sb[u] = b[u].scale4(p, q, G);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
#pragma unroll
      for (int j = 0; j < 4; ++j) av[t][j] = a[t].block(p, q, j, G);
      sa[t] = a[t].scale4(p, q, G);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int u = 0; u < NT; ++u) {
        acc[t][u] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bv[u][0], av[t][0], acc[t][u], 4, 4, 0, sb[u], 0, sa[t]);
        acc[t][u] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bv[u][1], av[t][1], acc[t][u], 4, 4, 1, sb[u], 1, sa[t]);
        acc[t][u] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bv[u][2], av[t][2], acc[t][u], 4, 4, 2, sb[u], 2, sa[t]);
        acc[t][u] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bv[u][3], av[t][3], acc[t][u], 4, 4, 3, sb[u], 3, sa[t]);
      }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int u = 0; u < NT; ++u) red[wave][t * NT + u][lane] = acc[t][u];
  __syncthreads();
  // lane (r, q) of accumulator t * NT + u: row 16 t + r, columns n0 + 16 u + 4 q .. + 3
  for (int i = threadIdx.x; i < MT * NT * 64; i += 64 * SK_WAVES) {
    const int tu = i >> 6, l = i & 63;
    v4f_t s = red[0][tu][l];
#pragma unroll
    for (int w = 1; w < SK_WAVES; ++w) s += red[w][tu][l];
    const int m = 16 * (tu / NT) + (l & 15);
    const int64_t n = n0 + 16 * (tu % NT) + 4 * (l >> 4);
    if (m >= M) continue;
    OutT* dst = c + m * ldc + n;
#pragma unroll
    for (int v = 0; v < 4; ++v) s[v] *= out_scale;
    if (n + 4 <= N && ((reinterpret_cast<uintptr_t>(dst) & (4 * sizeof(OutT) - 1)) == 0)) {
      if constexpr (sizeof(OutT) == 2) *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3]));
      else *reinterpret_cast<v4f_t*>(dst) = s;
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (n + v < N) {
          if constexpr (sizeof(OutT) == 2) dst[v] = __builtin_bit_cast(OutT, (unsigned short)f32_to_bf16_bits(s[v]));
          else dst[v] = s[v];
        }
      }
    }
  }
}

template <typename OutT, int MT, int NT>
void launch_skinny(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int64_t ldc, float out_scale, hipStream_t st) {
  hipLaunchKernelGGL((gemm_skinny_kernel<OutT, MT, NT>), dim3((unsigned)((N + 16 * NT - 1) / (16 * NT))), dim3(64 * SK_WAVES), 0, st, A, B, (int)M, N,
                     (int)(K / 32), (OutT*)c, ldc, out_scale);
}

// Columns per workgroup: every workgroup reads all of A, so once there is more than one workgroup of 16 columns per compute
// unit they are made wider.  us at 16 / 32 / 64 columns, 16 rows: N = 4096, K = 4096 4.6 / 5.5 / 7.6; N = 5000, K = 2880
// 4.5 / 4.9 / 6.7; N = 8192, K = 8192 10.9 / 9.4 / 13.3; N = 14336, K = 4096 10.5 / 8.9 / 8.3; N = 14336, K = 14336 31.1 / 23.9 / 21.7.
template <typename OutT, int MT>
void dispatch_columns(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int64_t ldc, float out_scale, hipStream_t st) {
  const int64_t strips = (N + 15) / 16;
  if (strips <= 384) launch_skinny<OutT, MT, 1>(A, B, M, N, K, c, ldc, out_scale, st);
  else if (strips <= 640) launch_skinny<OutT, MT, 2>(A, B, M, N, K, c, ldc, out_scale, st);
  else launch_skinny<OutT, MT, 4>(A, B, M, N, K, c, ldc, out_scale, st);
}

template <typename OutT>
void dispatch_rows(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int64_t ldc, float out_scale, hipStream_t st) {
  if (M <= 16) dispatch_columns<OutT, 1>(A, B, M, N, K, c, ldc, out_scale, st);
  else dispatch_columns<OutT, 2>(A, B, M, N, K, c, ldc, out_scale, st);
}

}  // namespace

// Offsets inside 32 rows of A and 64 of B (four strips) are 32-bit.
bool gemm_skinny_supported(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K) {
  return M <= 32 && K > 0 && A.ld < (1ll << 25) && B.ld < (1ll << 25);
}

// Below 1024 K some of the four waves have no piece of the reduction and a partial piece loads its scales byte by byte, so wide
// results go to the kernels that deal out columns only: the direct kernel below 512, the 64x64 tiles from 512 on.  us,
// here / there, at 16 and 32 rows:
//   M x N \ K           320         416         512         544         640         768         992        1024
//   16 x 4096       3.2/3.4     3.2/3.7     2.7/3.5     2.8/4.1     3.1/4.0     3.3/4.1     3.2/4.4     3.0/4.1
//   16 x 8192       3.8/3.4     3.8/3.7     2.9/3.4     3.2/4.1     3.7/4.0     4.0/4.0     3.9/4.3     3.4/4.1
//   16 x 14336      4.9/3.4     4.9/3.8     3.4/3.6     3.9/4.3     4.8/4.2     5.4/4.2     5.1/4.5     4.2/4.2
//   32 x 4096       3.8/3.6     3.8/4.0     2.9/3.5     3.2/4.2     3.7/4.1     4.0/4.1     3.9/4.4     3.4/4.2
//   32 x 10240      4.6/3.7     4.6/4.0     3.8/3.6     4.0/4.3     4.7/4.2     5.5/4.2     5.0/4.5     4.9/4.3
//   32 x 14336      5.7/3.7     5.8/4.1     3.9/3.7     4.6/4.3     5.6/4.2     6.4/4.2     6.3/4.6     4.9/4.3
bool gemm_skinny_pays(int64_t M, int64_t N, int64_t K) {
  const int64_t strips = (N + 15) / 16;   // (384 and 640: where a workgroup's columns double)
  if (K >= 1024) return true;
  if (K < 512) return strips <= 384 && K >= (M <= 16 ? 320 : 416);
  if (K <= 544) return K == 512 || M <= 16 || strips <= 640;
  return strips <= (M <= 16 ? 640 : 384);
}

void gemm_skinny_launch(const OperandView& A, const OperandView& B, int64_t M, int64_t N, int64_t K, void* c, int c_dtype, int64_t ldc, float out_scale,
                        hipStream_t st) {
  if (c_dtype == ALTO_DT_BF16) dispatch_rows<__bf16>(A, B, M, N, K, c, ldc, out_scale, st);
  else dispatch_rows<float>(A, B, M, N, K, c, ldc, out_scale, st);
}

}  // namespace alto
