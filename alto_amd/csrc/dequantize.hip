// MXFP4 dequantizer and nibble transpose (gfx950).
#include <type_traits>

#include "common.h"

namespace alto {
namespace {

// 8 codes (one dword) of a block with scale sf, decoded to fp32.  The convert decodes with scale 1 (exact) and the scale is
// a multiplication of its own, so that the scale bytes 0 and 255 mean 0.0 and inf, as in value(code) * 2^(byte - 127) made from the bits.
__device__ __forceinline__ void decode8(uint32_t w, float sf, int static_clip, float (&v)[8]) {
  typedef float f2_t __attribute__((ext_vector_type(2)));
  const f2_t p0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 0), p1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 1);
  const f2_t p2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 2), p3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 3);
  v[0] = p0[0] * sf; v[1] = p0[1] * sf; v[2] = p1[0] * sf; v[3] = p1[1] * sf;
  v[4] = p2[0] * sf; v[5] = p2[1] * sf; v[6] = p3[0] * sf; v[7] = p3[1] * sf;
  if (static_clip) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = v[e] * (4.0f / 3.0f);
  }
}

// Dense output (unit column stride, rows of C elements, 16-byte aligned): codes, scales (1D) and output are then all linear
// in the index of the lane's chunk, so nothing is divided per thread except for 2D scales.  A lane stores one 16-byte chunk
// (8 bf16 or 4 fp32 elements), so that a wave instruction writes a whole kilobyte, and takes DEQ_CHUNKS of them a workgroup
// apart, with all their loads in flight.  Bound by memory.  4096 x 4096 to bf16 (42 MB moved) took 25.4 us with the general
// kernel below (two 64-bit divisions per thread, eight 2-byte stores), 7.9 with this one and ordinary stores, 6.4 with
// non-temporal ones; to fp32 15.9 with two half kilobytes per wave instruction, 12.3 with whole ones, 11.1 with
// non-temporal stores (8192 x 8192: 58 / 48 / 42.6).
// STREAM: non-temporal stores, for results of 8 MB and more.  A smaller one gains nothing by them (2 MB: 2.4 us either way) and
// its reader finds it in no cache: dequantize and multiply by [C, 64], us ordinary / non-temporal: 160 x 2880 17.8 / 20.1,
// 352 x 2912 17.9 / 20.7, 1024 x 2048 13.5 / 15.2, 2048 x 2048 (8 MB) 15.6 / 16.9 and 3.5 / 3.1 by itself, 2048 x 4096
// 26.0 / 24.9 and 5.2 / 3.9.
constexpr int DEQ_CHUNKS = 4;
constexpr int64_t DEQ_STREAM_BYTES = 8ll << 20;
template <typename OutT, bool B2D, bool STREAM>
__global__ __launch_bounds__(256) void dequant_dense_kernel(const uint8_t* __restrict__ codes, const uint8_t* __restrict__ scales, int64_t n,
                                                            uint32_t chunks_per_row, OutT* __restrict__ out, int static_clip) {
  constexpr bool BF = sizeof(OutT) == 2;
  constexpr int VEC = 16 / sizeof(OutT), CPB = 32 / VEC;   // elements of a chunk, chunks of a block
  const int64_t base = (int64_t)blockIdx.x * (256 * DEQ_CHUNKS) + threadIdx.x;
  uint32_t w[DEQ_CHUNKS], s[DEQ_CHUNKS];
#pragma unroll
  for (int i = 0; i < DEQ_CHUNKS; ++i) {
    const int64_t k = base + 256 * i;
    w[i] = s[i] = 0;
    if (k < n) {
      if constexpr (BF) w[i] = reinterpret_cast<const uint32_t*>(codes)[k];
      else w[i] = reinterpret_cast<const uint16_t*>(codes)[k];
      int64_t g = k / CPB;
      if constexpr (B2D) {   // (n < 2^32 is a condition of this instantiation)
        const uint32_t r = (uint32_t)k / chunks_per_row;
        g = (int64_t)(r >> 5) * (chunks_per_row / CPB) + ((uint32_t)k - r * chunks_per_row) / CPB;
      }
      s[i] = scales[g];
    }
  }
#pragma unroll
  for (int i = 0; i < DEQ_CHUNKS; ++i) {
    const int64_t k = base + 256 * i;
    if (k >= n) return;
    float v[8];
    decode8(w[i], u2f(s[i] << 23), static_clip, v);   // (fp32: the upper four are not used)
    v4i_t o;
    if constexpr (BF) o = v4i_t{(int)pack_bf16x2(v[0], v[1]), (int)pack_bf16x2(v[2], v[3]), (int)pack_bf16x2(v[4], v[5]), (int)pack_bf16x2(v[6], v[7])};
    else o = v4i_t{(int)f2u(v[0]), (int)f2u(v[1]), (int)f2u(v[2]), (int)f2u(v[3])};
    v4i_t* dst = reinterpret_cast<v4i_t*>(out + k * VEC);
    if constexpr (STREAM) __builtin_nontemporal_store(o, dst);
    else *dst = o;
  }
}

// Any output strides: one thread, 8 codes (one dword of packed data) of one row.
template <typename OutT>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* __restrict__ codes, const uint8_t* __restrict__ scales,
                                                      int64_t R, int64_t C, int is_2d, OutT* __restrict__ out,
                                                      int64_t osr, int64_t osc, int static_clip) {
  const int64_t chunks_per_row = C / 8;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= R * chunks_per_row) return;
  const int64_t r = idx / chunks_per_row;
  const int64_t c0 = (idx % chunks_per_row) * 8;
  const uint32_t w = *reinterpret_cast<const uint32_t*>(codes + r * (C / 2) + c0 / 2);
  const uint32_t s = scales[(is_2d ? r / 32 : r) * (C / 32) + c0 / 32];
  float v[8];
  decode8(w, u2f(s << 23), static_clip, v);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    OutT o;
    if constexpr (sizeof(OutT) == 2) {
      unsigned short hb = (unsigned short)f32_to_bf16_bits(v[e]);
      o = __builtin_bit_cast(OutT, hb);
    } else {
      o = v[e];
    }
    out[r * osr + (c0 + e) * osc] = o;
  }
}

// 64x64 code tile through LDS: in [R][C/2] (packed along C) -> out [C][R/2] (packed along R)
__global__ __launch_bounds__(256) void transpose_codes_kernel(const uint8_t* __restrict__ in, int64_t R, int64_t C, uint8_t* __restrict__ out) {
  __shared__ uint8_t t[64][65];  // unpacked codes
  const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 64;
  const int tid = threadIdx.x;
  // 64 rows x 32 bytes: thread reads one byte at a time (8 passes)
#pragma unroll
  for (int pass = 0; pass < 8; ++pass) {
    int lr = pass * 8 + tid / 32, lb = tid % 32;
    int64_t r = r0 + lr, cb = c0 / 2 + lb;
    uint8_t v = (r < R && cb < C / 2) ? in[r * (C / 2) + cb] : 0;
    t[lr][2 * lb] = v & 0xF;
    t[lr][2 * lb + 1] = v >> 4;
  }
  __syncthreads();
#pragma unroll
  for (int pass = 0; pass < 8; ++pass) {
    int lc = pass * 8 + tid / 32, lb = tid % 32;  // output row = column lc, output byte lb covers rows 2lb, 2lb+1
    int64_t c = c0 + lc, rb = r0 / 2 + lb;
    if (c < C && rb < R / 2) out[c * (R / 2) + rb] = t[2 * lb][lc] | (t[2 * lb + 1][lc] << 4);
  }
}

}  // namespace
}  // namespace alto

extern "C" int alto_mxfp4_dequantize(const uint8_t* codes, const uint8_t* scales, int64_t R, int64_t C, int is_2d,
                                     void* out, int out_dtype, int64_t out_stride_r, int64_t out_stride_c,
                                     int clip_mode, void* stream) {
  using namespace alto;
  ALTO_REQUIRE(codes && scales && out, "dequantize: NULL pointer");
  ALTO_REQUIRE(R >= 0 && C >= 0 && C % 32 == 0, "dequantize: C (%lld) must be a multiple of 32", (long long)C);
  ALTO_REQUIRE(!is_2d || R % 32 == 0, "dequantize: 2D blocks need R (%lld) %% 32 == 0", (long long)R);
  ALTO_REQUIRE(out_dtype == ALTO_DT_BF16 || out_dtype == ALTO_DT_F32, "dequantize: bad out_dtype %d", out_dtype);
  ALTO_REQUIRE((reinterpret_cast<uintptr_t>(codes) & 3) == 0, "dequantize: codes must be 4-byte aligned");
  ALTO_REQUIRE((reinterpret_cast<uintptr_t>(out) & (out_dtype == ALTO_DT_F32 ? 3 : 1)) == 0, "dequantize: out must be aligned to its element size");
  ALTO_REQUIRE(R < (1ll << 31) && C < (1ll << 31) && product_below(1ll << 39, R, C / 8), "dequantize: %lld x %lld exceeds the grid", (long long)R, (long long)C);
  if (R == 0 || C == 0) return ALTO_MXFP4_OK;
  const int64_t n = R * (C / 8);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int sc = clip_mode == ALTO_CLIP_STATIC;
  if (out_stride_c == 1 && (out_stride_r == C || R == 1) && (reinterpret_cast<uintptr_t>(out) & 15) == 0 && n < (1ll << 31)) {
    const int64_t nc = out_dtype == ALTO_DT_BF16 ? n : 2 * n;   // chunks of 16 bytes
    const uint32_t cpr = (uint32_t)(C / (out_dtype == ALTO_DT_BF16 ? 8 : 4));
    const dim3 grid((unsigned)((nc + 256 * DEQ_CHUNKS - 1) / (256 * DEQ_CHUNKS)));
    const bool stream_out = 16 * nc >= DEQ_STREAM_BYTES;
    auto go = [&](auto kern, auto* dst) { hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, codes, scales, nc, cpr, dst, sc); };
    auto pick = [&](auto* dst) {
      using T = std::remove_pointer_t<decltype(dst)>;
      if (is_2d) stream_out ? go(dequant_dense_kernel<T, true, true>, dst) : go(dequant_dense_kernel<T, true, false>, dst);
      else stream_out ? go(dequant_dense_kernel<T, false, true>, dst) : go(dequant_dense_kernel<T, false, false>, dst);
    };
    if (out_dtype == ALTO_DT_BF16) pick((__bf16*)out);
    else pick((float*)out);
    return check_launch("dequantize");
  }
  const dim3 grid((unsigned)((n + 255) / 256));
  if (out_dtype == ALTO_DT_BF16)
    hipLaunchKernelGGL(dequant_kernel<__bf16>, grid, dim3(256), 0, st, codes, scales, R, C, is_2d, (__bf16*)out, out_stride_r, out_stride_c, sc);
  else
    hipLaunchKernelGGL(dequant_kernel<float>, grid, dim3(256), 0, st, codes, scales, R, C, is_2d, (float*)out, out_stride_r, out_stride_c, sc);
  return check_launch("dequantize");
}

extern "C" int alto_mxfp4_transpose_codes(const uint8_t* in, int64_t R, int64_t C, uint8_t* out, void* stream) {
  using namespace alto;
  ALTO_REQUIRE(in && out, "transpose_codes: NULL pointer");
  ALTO_REQUIRE(R >= 0 && C >= 0 && R % 2 == 0 && C % 2 == 0, "transpose_codes: R and C must be even");
  ALTO_REQUIRE(R < (1ll << 31) && C < (1ll << 31), "transpose_codes: size out of range");
  if (R == 0 || C == 0) return ALTO_MXFP4_OK;
  dim3 grid((unsigned)((C + 63) / 64), (unsigned)((R + 63) / 64));
  ALTO_REQUIRE(grid.y <= 65535u, "transpose_codes: R too large");
  hipLaunchKernelGGL(transpose_codes_kernel, grid, dim3(256), 0, reinterpret_cast<hipStream_t>(stream), in, R, C, out);
  return check_launch("transpose_codes");
}
