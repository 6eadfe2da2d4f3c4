// Fused quantize -> dequantize (gfx950): y = convert_from_mxfp4(convert_to_mxfp4(x)) in one pass over x, round to
// nearest even, blocks of 32 along the contiguous dim or 32x32.  Used where only the quantisation error is wanted
// (weight de-oscillation), so no codes or scales are written.
#include "common.h"

namespace alto {
namespace {

typedef unsigned short us2q_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pk_max_u16q(uint32_t a, uint32_t b) {
  us2q_t r = __builtin_elementwise_max(__builtin_bit_cast(us2q_t, a), __builtin_bit_cast(us2q_t, b));
  return __builtin_bit_cast(uint32_t, r);
}

// One workgroup (256 threads): 32 rows x 256 columns.  A lane holds 16 bytes (4 fp32 or 8 bf16 elements) of a row for NI
// rows, so a wave instruction reads and writes whole kilobytes in a row; 8 or 4 lanes share a block of 32 elements.
// Bound by memory.  The results go out as non-temporal stores: 14336 x 4096 fp32 (470 MB moved) took 95.8 us with two half
// kilobytes per wave instruction, 85.9 with whole ones and 69.4 with non-temporal stores on top (6.8 TB/s; a plain copy
// takes 87.5); bf16 44.5 -> 35.3.  Non-temporal loads lose (77 us).
template <typename T, bool B2D>
__global__ __launch_bounds__(256) void qdq_kernel(const T* __restrict__ x, int64_t ld_x, int64_t bs_x, T* __restrict__ y, int64_t ld_y,
                                                  int64_t bs_y, int M, int C, int uos) {
  typedef float f2_t __attribute__((ext_vector_type(2)));
  constexpr bool BF = sizeof(T) == 2;
  constexpr int VEC = 16 / sizeof(T);                       // elements of a lane
  constexpr int LPR = 256 / VEC, RPP = 256 / LPR, NI = 32 / RPP;   // lanes per row, rows per pass over the tile, passes
  __shared__ uint32_t blkmax[8];
  const int tid = threadIdx.x;
  const int col0 = blockIdx.x * 256, row0 = blockIdx.y * 32;
  const int64_t b = blockIdx.z;
  if (B2D) {
    if (tid < 8) blkmax[tid] = 0;
    __syncthreads();
  }
  const int chunk = tid % LPR, rsub = tid / LPR;
  const int c = col0 + chunk * VEC, blk = chunk * VEC / 32;
  uint4 w[NI];
  uint32_t amax[NI];
  bool valid[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = rsub + RPP * i;
    valid[i] = (row0 + r < M) && (c < C);
    w[i] = make_uint4(0, 0, 0, 0);
    if (valid[i]) w[i] = *reinterpret_cast<const uint4*>(x + b * bs_x + (int64_t)(row0 + r) * ld_x + c);
  }
  uint32_t all = 0;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    uint32_t a;
    if constexpr (BF) {
      a = pk_max_u16q(pk_max_u16q(w[i].x & 0x7FFF7FFFu, w[i].y & 0x7FFF7FFFu), pk_max_u16q(w[i].z & 0x7FFF7FFFu, w[i].w & 0x7FFF7FFFu));
      a = max(a & 0xFFFFu, a >> 16);
    } else {
      a = max(max(w[i].x & 0x7FFFFFFFu, w[i].y & 0x7FFFFFFFu), max(w[i].z & 0x7FFFFFFFu, w[i].w & 0x7FFFFFFFu));
    }
    amax[i] = a;
    all = max(all, a);
  }
  auto block_max = [](uint32_t a) {   // over the lanes that share a block
    a = max(a, dpp_u32<ALTO_DPP_QUAD_XOR1>(a));
    a = max(a, dpp_u32<ALTO_DPP_QUAD_XOR2>(a));
    if constexpr (!BF) a = max(a, dpp_u32<ALTO_DPP_HALF_MIRROR>(a));
    return a;
  };
  if constexpr (B2D) {   // the rows of this lane first, then the lanes, then one atomic per lane group and wave
    all = block_max(all);
    if (chunk % (32 / VEC) == 0) atomicMax(&blkmax[blk], all);
    __syncthreads();
    all = blkmax[blk];
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const uint32_t a = B2D ? all : block_max(amax[i]);
    if (!valid[i]) continue;
    uint32_t s;
    if (uos) s = e8m0_uos(BF ? u2f(a << 16) : u2f(a));
    else s = BF ? e8m0_from_bf16_bits(a) : e8m0_from_f32_bits(a);
    const float scale_f = u2f(s << 23);
    uint32_t codes = 0;
    if constexpr (BF) {
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, bf16_lo(w[i].x), bf16_hi(w[i].x), scale_f, 0);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, bf16_lo(w[i].y), bf16_hi(w[i].y), scale_f, 1);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, bf16_lo(w[i].z), bf16_hi(w[i].z), scale_f, 2);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, bf16_lo(w[i].w), bf16_hi(w[i].w), scale_f, 3);
    } else {
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, u2f(w[i].x), u2f(w[i].y), scale_f, 0);
      codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, u2f(w[i].z), u2f(w[i].w), scale_f, 1);
    }
    // decoded with scale 1 (exact), then multiplied: what a scale byte of 255 makes of a zero code stays as it is
    const f2_t p0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, 0) * scale_f, p1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, 1) * scale_f;
    T* dst = y + b * bs_y + (int64_t)(row0 + rsub + RPP * i) * ld_y + c;
    v4i_t o;
    if constexpr (BF) {
      const f2_t p2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, 2) * scale_f, p3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, 3) * scale_f;
      o = v4i_t{(int)pack_bf16x2(p0[0], p0[1]), (int)pack_bf16x2(p1[0], p1[1]), (int)pack_bf16x2(p2[0], p2[1]), (int)pack_bf16x2(p3[0], p3[1])};
    } else {
      o = v4i_t{(int)f2u(p0[0]), (int)f2u(p0[1]), (int)f2u(p1[0]), (int)f2u(p1[1])};
    }
    __builtin_nontemporal_store(o, reinterpret_cast<v4i_t*>(dst));
  }
}

}  // namespace
}  // namespace alto

extern "C" int alto_mxfp4_qdq(const void* x, int dtype, int64_t batch, int64_t M, int64_t C, int64_t ld_x, int64_t bs_x,
                              void* y, int64_t ld_y, int64_t bs_y, int is_2d, int use_uos, void* stream) {
  using namespace alto;
  ALTO_REQUIRE(x && y, "qdq: NULL pointer");
  ALTO_REQUIRE(dtype == ALTO_DT_BF16 || dtype == ALTO_DT_F32, "qdq: dtype %d is neither bf16 (0) nor f32 (1)", dtype);
  ALTO_REQUIRE(batch >= 0 && M >= 0 && C >= 0 && C % 32 == 0, "qdq: C (%lld) must be a multiple of 32", (long long)C);
  ALTO_REQUIRE(!is_2d || M % 32 == 0, "qdq: 2D blocks need M (%lld) %% 32 == 0", (long long)M);
  ALTO_REQUIRE(M < (1ll << 31) && C < (1ll << 31) && batch < 65536 && (M + 31) / 32 <= 65535, "qdq: size out of range");
  const int64_t vec = dtype == ALTO_DT_BF16 ? 8 : 4;
  ALTO_REQUIRE(ld_x >= C && ld_y >= C && ld_x % vec == 0 && ld_y % vec == 0 && bs_x % vec == 0 && bs_y % vec == 0,
               "qdq: row/batch strides must be >= C and multiples of %lld elements", (long long)vec);
  ALTO_REQUIRE(((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15) == 0, "qdq: x and y must be 16-byte aligned");
  if (batch == 0 || M == 0 || C == 0) return ALTO_MXFP4_OK;
  dim3 grid((unsigned)((C + 255) / 256), (unsigned)((M + 31) / 32), (unsigned)batch);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int uos = use_uos ? 1 : 0;
  if (dtype == ALTO_DT_BF16) {
    if (is_2d) hipLaunchKernelGGL((qdq_kernel<__bf16, true>), grid, dim3(256), 0, st, (const __bf16*)x, ld_x, bs_x, (__bf16*)y, ld_y, bs_y, (int)M, (int)C, uos);
    else hipLaunchKernelGGL((qdq_kernel<__bf16, false>), grid, dim3(256), 0, st, (const __bf16*)x, ld_x, bs_x, (__bf16*)y, ld_y, bs_y, (int)M, (int)C, uos);
  } else {
    if (is_2d) hipLaunchKernelGGL((qdq_kernel<float, true>), grid, dim3(256), 0, st, (const float*)x, ld_x, bs_x, (float*)y, ld_y, bs_y, (int)M, (int)C, uos);
    else hipLaunchKernelGGL((qdq_kernel<float, false>), grid, dim3(256), 0, st, (const float*)x, ld_x, bs_x, (float*)y, ld_y, bs_y, (int)M, (int)C, uos);
  }
  return check_launch("qdq");
}
