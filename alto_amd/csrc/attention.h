// What the attention kernels (attention.hip) and their operand quantizer (attention_quantize.hip) share.
#pragma once
#include <type_traits>
#include <utility>

#include "common.h"

namespace alto {

struct AttnArgs {
  const uint8_t* q;  const uint8_t* qs;    // [B, Hq, Sq, D/2],  [B, Hq, Sq/32, D/32]; or NULL and, as bf16 values in the caller's layout,
  const __bf16* qx;  int64_t qx_sb, qx_sh, qx_ss;   // element (b, h, row, column) at these strides, unit stride along D
  const uint8_t* k;  const uint8_t* ks;    // [B, Hk, Sk, D/2],  [B, Hk, Sk/32, D/32]
  const uint8_t* vt; const uint8_t* vs;    // [B, Hk, Dv, Sk/2] packed along keys, [B, Hk, Sk/32, Dv/32]
  void* out; float* lse;                   // bf16 and fp32, element (b, h, row, column) at the strides below
  int64_t o_sb, o_sh, o_ss, l_sb, l_sh, l_ss;
  int Hq, Hk, Sq, Sk, Sk_used;             // Sk keys are allocated, the first Sk_used exist (packed sequences: Sq and Sk are token counts)
  int64_t k_bytes, v_bytes;                // extent of the code buffers
  float sm_scale;
  int causal;
  // optional additive terms on the scaled scores (triton_flash_attention_mxfp4.py:288-299), fp32:
  const float* bias;  int64_t bias_sb, bias_sh, bias_sm, bias_bytes;   // element (b, h, m, n) at b sb + h sh + m sm + n; NULL: none
  const float* alibi; int64_t alibi_sb, alibi_sh;                      // slope of (b, h) at b sb + h sh; NULL: none
};

// Sequences packed along the tokens (B = 1): sequence i owns query rows q0[i] .. + qn[i] and keys k0[i] .. + kn[i] (all
// multiples of 32) and the row blocks z0[i] .. z0[i+1] of the grid.  By value, in the kernel arguments: no copy to the
// device, nothing to keep alive.
constexpr int ATTN_MAX_SEQS = 64;
struct AttnSeqs {
  int n;
  int z0[ATTN_MAX_SEQS + 1], q0[ATTN_MAX_SEQS], qn[ATTN_MAX_SEQS], k0[ATTN_MAX_SEQS], kn[ATTN_MAX_SEQS];
};
struct AttnNoSeqs {};

// Uniform 4-byte aligned data through the scalar cache: as vector loads these sit in the same counter as the direct-to-LDS
// prefetch, and the wait for a block's scale bytes drains the prefetched block with them.  Whole causal calls, us, vector ->
// scalar: 4 x 4096 tokens x 32 heads x 64 258 -> 248, 2 x 3232 x 16 x 64 60.7 -> 59.2, 1 x 4096 x 32 x 128 110.4 -> 109.3,
// 4 x 2048 x 64 x 128 218 -> 216, packed sequences the same to 1.5 % faster; 4 x 1024 x 32 x 128 loses, 47.6 -> 48.4.
typedef const __attribute__((address_space(4))) uint32_t* scalar_u32;
__device__ __forceinline__ scalar_u32 scalar_ptr(const uint8_t* p) { return (scalar_u32)(uintptr_t)p; }

constexpr float ATTN_RCP_LN2 = 1.4426950408889634f;
constexpr float ATTN_LN2 = 0.6931471824645996f;

__device__ __forceinline__ v8i_t frag16(const uint8_t* p) {
  const uint4 w = *reinterpret_cast<const uint4*>(p);
  return v8i_t{(int)w.x, (int)w.y, (int)w.z, (int)w.w, 0, 0, 0, 0};
}
template <int N, typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) { static_for_impl<N>(static_cast<F&&>(f), std::make_integer_sequence<int, N>{}); }

typedef unsigned v2u_t __attribute__((ext_vector_type(2)));
typedef int v4i_8_t __attribute__((ext_vector_type(4), aligned(8)));   // 16 bytes at an 8-byte boundary
// v_permlane32_swap(a, b) returns {a of lanes 0..31 | b of lanes 0..31,  a of lanes 32..63 | b of lanes 32..63}
// (first | second half of the wave): a value and its copy come back as the low half's and the high half's values.
// fmaxf for values of which at most one is NaN, in one instruction: v_med3 with +infinity (opaque to the compiler, which would turn it
// back into a maximum and put a canonicalizing copy of either operand in front of it).
__device__ __forceinline__ float max_one(float x, float y) {
  float inf = __builtin_inff();
  asm("" : "+s"(inf));
  return __builtin_amdgcn_fmed3f(x, y, inf);
}
__device__ __forceinline__ float max_of_pair(v2u_t p) { return max_one(u2f(p[0]), u2f(p[1])); }

typedef unsigned short us2a_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk_max_u16a(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(us2a_t, a), __builtin_bit_cast(us2a_t, b)));
}

// absmax bits of 8 consecutive elements held in 4 (bf16) or 8 (fp32) dwords
template <typename T>
__device__ __forceinline__ uint32_t absmax8(const uint32_t* w) {
  if constexpr (sizeof(T) == 2) {
    const uint32_t a = pk_max_u16a(pk_max_u16a(w[0] & 0x7FFF7FFFu, w[1] & 0x7FFF7FFFu), pk_max_u16a(w[2] & 0x7FFF7FFFu, w[3] & 0x7FFF7FFFu));
    return max(a & 0xFFFFu, a >> 16);
  } else {
    uint32_t a = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) a = max(a, w[e] & 0x7FFFFFFFu);
    return a;
  }
}
template <typename T>
__device__ __forceinline__ uint32_t encode8(const uint32_t* w, float scale) {
  uint32_t o = 0;
  if constexpr (sizeof(T) == 2) {
    o = __builtin_amdgcn_cvt_scalef32_pk_fp4_bf16(o, __builtin_bit_cast(bf16x2_t, w[0]), scale, 0);
    o = __builtin_amdgcn_cvt_scalef32_pk_fp4_bf16(o, __builtin_bit_cast(bf16x2_t, w[1]), scale, 1);
    o = __builtin_amdgcn_cvt_scalef32_pk_fp4_bf16(o, __builtin_bit_cast(bf16x2_t, w[2]), scale, 2);
    o = __builtin_amdgcn_cvt_scalef32_pk_fp4_bf16(o, __builtin_bit_cast(bf16x2_t, w[3]), scale, 3);
  } else {
    o = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(o, u2f(w[0]), u2f(w[1]), scale, 0);
    o = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(o, u2f(w[2]), u2f(w[3]), scale, 1);
    o = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(o, u2f(w[4]), u2f(w[5]), scale, 2);
    o = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(o, u2f(w[6]), u2f(w[7]), scale, 3);
  }
  return o;
}


// Between a wave's LDS writes and its own lanes' reads of them.  The LDS keeps a wave's accesses in order, so this is no instruction;
// it keeps the compiler from moving either side past the other.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// A wave's 32 rows of Q, straight from bf16, as the score product takes them: lane (r = lane % 32, h = lane / 32) gets the codes of
// row r, columns 64 s + 32 h .. + 32, and the scale byte of that 32 x 32 block.  The loads are whole 128-byte lines (8 lanes a row,
// 8 rows an instruction; a lane that fetched its own 64 bytes cost 32 line lookups an instruction instead of 8); the codes change
// lanes through `scratch`, NK KB of LDS that only this wave uses, at consecutive addresses (two rows meet in a bank on the way out:
// 4 cycles a read).  Codes and scales are those of alto_mxfp4_attention_quantize.
template <int NK>
__device__ __forceinline__ void quantize_q(const __bf16* x, int64_t row_stride, int lane, uint8_t* scratch, v8i_t (&qf)[NK], int (&qsc)[NK]) {
  uint32_t w[NK][4][4];
#pragma unroll
  for (int s = 0; s < NK; ++s)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const v4i_t v = __builtin_nontemporal_load(reinterpret_cast<const v4i_t*>(x + (int64_t)(8 * i + (lane >> 3)) * row_stride + 64 * s + 8 * (lane & 7)));
      w[s][i][0] = v[0]; w[s][i][1] = v[1]; w[s][i][2] = v[2]; w[s][i][3] = v[3];
    }
#pragma unroll
  for (int s = 0; s < NK; ++s) {
    uint32_t m = max(max(absmax8<__bf16>(w[s][0]), absmax8<__bf16>(w[s][1])), max(absmax8<__bf16>(w[s][2]), absmax8<__bf16>(w[s][3])));
    m = max(m, dpp_u32<ALTO_DPP_QUAD_XOR1>(m));   // the block's rows and columns: the lanes that agree in bit 2
    m = max(m, dpp_u32<ALTO_DPP_QUAD_XOR2>(m));
    m = max(m, dpp_u32<ALTO_DPP_ROW_ROR8>(m));
    const v2u_t p16 = __builtin_amdgcn_permlane16_swap(m, m, false, false);
    m = max(p16[0], p16[1]);
    const v2u_t p32 = __builtin_amdgcn_permlane32_swap(m, m, false, false);
    m = max(p32[0], p32[1]);
    const uint32_t e = e8m0_from_bf16_bits(m);
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<uint32_t*>(scratch + 1024 * s + 256 * i + 4 * lane) = encode8<__bf16>(w[s][i], u2f(e << 23));
    qsc[s] = lane < 32 ? __builtin_amdgcn_readlane((int)e, 0) : __builtin_amdgcn_readlane((int)e, 4);
  }
  wave_lds_order();
#pragma unroll
  for (int s = 0; s < NK; ++s) qf[s] = frag16(scratch + 1024 * s + (lane & 31) * 32 + (lane >> 5) * 16);
}

// What workgroup row `z` of `nz` works on: its sequence and its block of rows, the last rows first with a causal mask.
struct AttnRows {
  int qn, kn, q_first, k_first, block;
};
template <typename SEQS>
__device__ __forceinline__ AttnRows attn_rows(const AttnArgs& a, const SEQS& seqs, int z, int nz) {
  AttnRows w{a.Sq, a.Sk_used, 0, 0, 0};
  if constexpr (std::is_same<SEQS, AttnSeqs>::value) {
    int lo = 0, hi = seqs.n - 1;   // the sequence this row block belongs to: the last one with z0[i] <= z
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (seqs.z0[mid] <= z) lo = mid; else hi = mid - 1;
    }
    w.qn = seqs.qn[lo]; w.kn = seqs.kn[lo]; w.q_first = seqs.q0[lo]; w.k_first = seqs.k0[lo];
    nz = seqs.z0[lo + 1] - seqs.z0[lo];
    z -= seqs.z0[lo];
  }
  w.block = a.causal ? nz - 1 - z : z;
  return w;
}
// Eight neighbouring workgroups go to the eight XCDs in turn: each gets a range of consecutive heads, so a key / value head comes
// into one L2 (two, where a range starts inside its query heads) and not into all of them: 195 -> 187 us for 4 x 2048 tokens,
// 64 / 8 heads of 128, causal.
__device__ __forceinline__ int attn_head(const AttnArgs& a) {
  return a.Hq % 8 == 0 ? (int)((blockIdx.x & 7) * (a.Hq >> 3) + (blockIdx.x >> 3)) : (int)blockIdx.x;
}

// Which key of a 32-key tile row i of the score product is: bits 2 and 3 of i change places, so that register v of half h holds key
// 16 (v / 8) + 8 h + v % 8.  A half's eight codes of a dword are then eight consecutive keys, and the operand of the product with V
// comes out of the half-wave swaps in key order (in the plain order, key 8 (v / 4) + 4 h + v % 4, it took four byte permutes more).
__device__ __forceinline__ int score_key(int i) { return (i & 0x13) | (i & 4) << 1 | (i & 8) >> 1; }

// Hides the scores of keys that a lane's row may not see: `seen` = how many keys from the lane's first one (8 h of the block) on
// it does.  (The empty assembly keeps each four comparisons next to their uses: all 32 results taken together spilled scalars that the
// loop over the blocks needs, and one at a time every use waits for its comparison.)
__device__ __forceinline__ void mask_scores(v16f_t (&S)[2], int seen) {
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int v = 0; v < 16; v += 4) {
      float x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = 32 * t + 16 * (v >> 3) + (v & 7) + i >= seen ? -__builtin_inff() : S[t][v + i];
      asm volatile("" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]));
#pragma unroll
      for (int i = 0; i < 4; ++i) S[t][v + i] = x[i];
    }
}

// Largest score of row r = lane % 32 in the tile h = lane / 32 (S: two tiles of 32 keys, a row's keys over the lanes r and r + 32), and
// in both tiles.  One swap hands either lane of a row the other one's part of its tile (a swap for each tile, as before, does the work
// for both tiles in both lanes).  ALONE (one wave a SIMD, nothing to fill a wait): the second swap does not wait for the first, for an
// instruction more.
template <bool ALONE>
__device__ __forceinline__ void row_maxima(const v16f_t (&S)[2], float& tile_max, float& row_max) {
  float x[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    x[t] = -__builtin_inff();   // (and never NaN)
#pragma unroll
    for (int v = 0; v < 16; ++v) x[t] = fmaxf(x[t], S[t][v]);
  }
  tile_max = max_of_pair(__builtin_amdgcn_permlane32_swap(f2u(x[0]), f2u(x[1]), false, false));
  const float mine = ALONE ? max_one(x[0], x[1]) : tile_max;
  row_max = max_of_pair(__builtin_amdgcn_permlane32_swap(f2u(mine), f2u(mine), false, false));
}

// Probabilities of a wave's 32 rows and 64 keys (S: scores of this lane's row, keys as score_key() deals them; tile_max: the row's
// largest score in the tile h, whose probability is the tile's largest: exp2 is monotonic; cs: factor into the base-2 domain; m_new:
// running maximum there): one E8M0 scale per (row, 32 keys), E2M1 codes (round to nearest even), as an operand of the product with V.
// Lane (r, h) multiplies tile h: it has that tile's scale, and gets the 16 codes of it that the other lane of the row holds.
__device__ __forceinline__ void quantize_probabilities(v16f_t (&S)[2], float tile_max, float cs, float m_new, v8i_t& pf, int& pscale) {
  const float am = __builtin_amdgcn_exp2f(__builtin_fmaf(tile_max, cs, -m_new));
  pscale = (int)e8m0_from_f32_bits(f2u(am));
  const v2u_t scale = __builtin_amdgcn_permlane32_swap((unsigned)pscale << 23, (unsigned)pscale << 23, false, false);   // of tile 0, of tile 1
  uint32_t c[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const float scale_f = u2f(scale[t]);
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      float p[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[t][8 * w + i], cs, -m_new));
      uint32_t o = f2u(p[0]);   // (every byte is replaced: starting from a register that ends here costs no move)
      o = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(o, p[0], p[1], scale_f, 0);
      o = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(o, p[2], p[3], scale_f, 1);
      o = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(o, p[4], p[5], scale_f, 2);
      o = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(o, p[6], p[7], scale_f, 3);
      c[t][w] = o;
    }
  }
  const v2u_t p0 = __builtin_amdgcn_permlane32_swap(c[0][0], c[1][0], false, false);   // keys 0..7 and 8..15 of the tile
  const v2u_t p1 = __builtin_amdgcn_permlane32_swap(c[0][1], c[1][1], false, false);   // keys 16..23 and 24..31
  pf = v8i_t{(int)p0[0], (int)p0[1], (int)p1[0], (int)p1[1], 0, 0, 0, 0};
}

// Row sums of the quantised probabilities, in one product of 16 x 16 x 128 (4 accumulator registers a lane instead of 16, and half the
// matrix time of a 32 x 32 x 64 product with a column of ones).  That product takes the operand of lane l for row l % 16 and keys
// 32 (l / 16) .. + 32, while the lane holds row l % 32 and the tile l / 32: for row i < 16 the key ranges 0 and 2 are its two tiles and 1
// and 3 those of row 16 + i.  Row n of the other operand is one where (n / 4) % 2 and the range agree in the lowest bit, so all
// registers of lane l get the sum of row l % 32.
__device__ __forceinline__ int row_sum_selector(int lane) { return ((lane >> 2) & 1) == ((lane >> 4) & 1) ? 0x22222222 : 0; }   // (E2M1 code 2 = 1.0)
__device__ __forceinline__ v4f_t add_row_sums(int selector, const v8i_t& pf, int pscale, v4f_t l) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(v8i_t{selector, selector, selector, selector, 0, 0, 0, 0}, pf, l, 4, 4, 0, 127, 0, pscale);
}

// Launch of the kernel whose four waves deal out the keys of 32 rows (attention_split.hip); `row_blocks` in units of 32 rows.
template <typename SEQS>
int launch_attn_split(const AttnArgs& a, const SEQS& seqs, int B, int row_blocks, int64_t D, int64_t Dv, hipStream_t st);

}  // namespace alto
