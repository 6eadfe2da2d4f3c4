// MXFP4 flash-attention forward for gfx950: S = Q K^T and O = P V both on v_mfma_scale_f32_32x32x64_f8f6f4, with the
// probabilities re-quantised to MXFP4 in registers and the row sums taken from the SAME quantised probabilities
// (the recurrence of alto/kernels/fp4/mxfp4/triton_flash_attention_mxfp4.py:168-400,640-890, key blocks of 64).
//
// One wave owns 32 query rows of one head.  The MFMA is issued as (first = rows that land in registers, second = rows that land in
// lanes).  S tiles keep the query row in the lane (lane % 32) and spread keys over the 16 accumulator registers, so the per-row softmax
// state (running max, rescale factor, sum) is one scalar per lane and the only cross-lane traffic is between the two lanes (l, l ^ 32)
// that share a row.  O tiles have the rows in the registers and the value columns in the lanes: a block whose running maximum rises in
// a few rows only rescales the registers of those rows, and a lane's columns are neighbours in memory.
//
// What bounds it: vector instructions (the matrix pipes are busy a fifth of the time).  Device time of changing inputs, us, against the
// kernel with O's rows in lanes, a maximum and a scale of either tile in both lanes of a row, row sums by a 32 x 32 x 64 product of ones
// and the plain key order, all with the same results bit for bit:
//   4 x 2048 tokens, 64 / 8 heads of 128: causal 177.6 -> 162.1, all keys 304 -> 281; 4096 tokens, 32 heads of 128, all keys 151.6 -> 141.7;
//   4 x 4096, 32 / 8 heads of 64: 428 -> 385, causal 230 -> 203; 2 x 2048, 32 / 8 heads of 192 / 256, causal: 61.0 -> 52.8, 63.3 -> 60.0.
// Of that, the maxima, scales, key order and mask (row_maxima() .. mask_scores() in attention.h) gave 5 % (D = 128) to 8 % (64), the
// rescale by rows 3 to 5 %, the smaller product for the sums 1 to 2 %.  The rescale factors take the way through the LDS: a product
// with a row of ones on the matrix pipe and ds_bpermute were 2 to 4 % slower; groups of four rows instead of eight are 1 % faster with
// long sequences of D = 128, 3 % slower with D = 64 and 1 % slower with 1024 tokens.  Four workgroups a compute unit do not fit D = 128
// (12 registers spilled: 178), five are no faster with D = 64.
#include <algorithm>
#include <memory>
#include <new>

#include "attention.h"

namespace alto {

#ifndef ATTN_WG_PER_CU
#define ATTN_WG_PER_CU 3
#endif
// NK = D / 64 (MFMA K steps of Q K^T), ND = Dv / 32 (output tiles).
// The four waves of a workgroup own 128 consecutive query rows of one head and walk the key blocks together: a block's
// K codes (64 rows x D/2 bytes) and V codes (Dv rows x 32 bytes) are fetched once per workgroup, two blocks ahead, with
// direct-to-LDS loads (16 bytes per lane, 1 KB per wave instruction, no registers in between) into a three-slot ring;
// one barrier per block.  (Fetching the pieces per wave straight from global memory made the vector-memory path the
// bound: 8 KB per wave and block in scattered 16-byte accesses.  One block ahead through registers left the waves
// waiting for the load at the end of every block: the kernel ran at 38 % VALU issue with the matrix pipes at 11 %.)
constexpr int ATTN_RING = 3;
template <int NK, int ND>
struct AttnTile {
  static constexpr int D = NK * 64, DV = ND * 32;
  static constexpr int K_BYTES = 64 * (D / 2), V_BYTES = DV * 32;       // one block of K codes, of V codes
  static constexpr int SLOT = K_BYTES + V_BYTES;
  static constexpr int FACTORS = ATTN_RING * SLOT, QUERY = FACTORS + 4 * 128;   // behind the ring: 32 row factors a wave, then Q's codes on their way through the lanes
};

// The body of the kernel as a function of its own because of the `__restrict__` on the outputs: inlining then marks the
// direct-to-LDS loads as not aliasing them, and only with that mark does the compiler's wait insertion keep those loads
// in flight across the LDS reads that follow (unmarked, it puts an `s_waitcnt vmcnt(0)` before the next LDS read).
// BIASED: the scores get a.bias and / or the ALiBi term -slope |row + Sk - Sq - key| added after the scaling and the mask,
// before the running maximum (:288-308); a separate instantiation, the plain one carries none of it.
// QBF: Q comes as bf16 values and every wave quantizes its own rows (no other wave reads them), which saves writing the codes
// and reading them back and leaves the operand quantizer K and V only.  4 x 2048 tokens, 64 / 8 heads of 128, causal (134 of the
// 168 MB are Q), changing inputs, us: quantizer and this kernel on codes 38.8 and 169.5, 201 together; with QBF 8.8 and 181, 187
// together (another box: 38.6 and 162.7, 193.5; 8.8 and 171.8, 181).  How the kernel with QBF got there: every lane fetching the 64
// bytes it multiplies 201, whole lines (quantize_q) 197, at raised wave priority 195 (the two other workgroups of the compute unit hide the
// wait, the priority lets the arithmetic behind it through), Q read non-temporally 2 less; of use to the kernel on codes as well:
// the heads dealt to the XCDs in ranges 195 -> 187, the results stored as whole rows 187 -> 181 (then through the LDS).
// SEQS: AttnSeqs, or AttnNoSeqs for B sequences of one length.
// ALONE: for launches that leave a SIMD about one wave (see launch_plan): what a wave waits for costs its time, and instructions cost none.  The
// rescale takes all rows without a branch (four branches of which none is taken, in nearly every block of the first thousand keys,
// cost 90 clocks a block), V's codes are read ahead of it, and the second swap of row_maxima() does not wait for the first.
template <int NK, int ND, bool BIASED, bool QBF, bool ALONE, typename SEQS>
__device__ __forceinline__ void attn_fwd_body(const AttnArgs& a, const SEQS& seqs, __bf16* __restrict__ out, float* __restrict__ lse_out, uint8_t* ring) {
  constexpr int D = NK * 64, DV = ND * 32;
  constexpr int K_BYTES = AttnTile<NK, ND>::K_BYTES, V_BYTES = AttnTile<NK, ND>::V_BYTES, SLOT = AttnTile<NK, ND>::SLOT;
  constexpr int K_PIECES = K_BYTES / 16, V_PIECES = V_BYTES / 16;
  constexpr int PIECES = K_PIECES + V_PIECES;             // 16-byte pieces of one block, K first; both multiples of 64
  constexpr int DMA_MAX = (PIECES + 255) / 256;           // loads per wave and block: DMA_MAX, or one less for the last waves

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  // grid (heads, batch, row blocks): with a causal mask every head's longest rows are dispatched before anybody's shorter
  // ones, so the launch ends with the cheapest workgroups (packed sequences: the host passes them longest first)
  const AttnRows w = attn_rows(a, seqs, (int)blockIdx.z, (int)gridDim.z);
  const int qn = w.qn, kn = w.kn, q_first = w.q_first, k_first = w.k_first;
  const int qblk = w.block;
  const int q0 = (qblk * 4 + wave) * 32;
  const bool live = q0 < qn;                      // a wave past the last row still helps with loads and barriers
  const int hq = attn_head(a), b = blockIdx.y;
  const int hk = hq / (a.Hq / a.Hk);
  // rows of the operand buffers where this (sequence, head) starts
  const int64_t q_base = ((int64_t)b * a.Hq + hq) * a.Sq + q_first, bhk = (int64_t)b * a.Hk + hk, k_base = bhk * a.Sk + k_first;
  const int qrow = live ? q0 + r : 0;
  const int shift = kn - qn;                           // causal mask is aligned to the bottom-right corner

  // ---- Q pieces: row qrow, K step ks, half h -> 16 bytes; one scale byte per (32-row block, 32-column block)
  v8i_t qf[NK];
  int qsc[NK];
  if constexpr (!QBF) {
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      qf[s] = frag16(a.q + (q_base + qrow) * (D / 2) + s * 32 + h * 16);
      qsc[s] = a.qs[(q_base / 32 + qrow / 32) * (D / 32) + 2 * s + h];
    }
  }

  v16f_t acc_o[ND];
  v4f_t acc_l = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc_o[d][v] = 0.0f;
  float m_i = -__builtin_inff();                   // running row max of S * sm_scale * log2(e)
  const float c2 = a.sm_scale * ATTN_RCP_LN2;
  const float cs = BIASED ? 1.0f : c2;   // what is left to multiply once the scores are in the base-2 domain
  // bias rows of this (batch, head): a descriptor over the rest of the tensor (no range when there is no bias: loads give 0)
  const __amdgpu_buffer_rsrc_t rsrc_bias = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>((BIASED && a.bias) ? a.bias + b * a.bias_sb + hq * a.bias_sh : nullptr), 0,
      (BIASED && a.bias) ? (int)(a.bias_bytes - (b * a.bias_sb + hq * a.bias_sh) * 4) : 0, 0x00020000);
  const float slope2 = (BIASED && a.alibi) ? a.alibi[b * a.alibi_sb + hq * a.alibi_sh] * ATTN_RCP_LN2 : 0.0f;

  const int selector = row_sum_selector(lane);
  float* const factors = reinterpret_cast<float*>(ring + AttnTile<NK, ND>::FACTORS + wave * 128);   // of this wave's rows, on their way to the registers

  // blocks this wave needs, and the most any wave of the workgroup needs (the last wave's rows reach furthest)
  const int all_blk = (kn + 63) / 64;
  int nblk = all_blk, wg_blk = all_blk;
  if (a.causal) {
    const int lim = (q0 + 32 + shift + 63) / 64;
    nblk = lim < all_blk ? lim : all_blk;
    int q_end = qblk * 128 + 128;
    q_end = q_end < qn ? q_end : qn;
    const int wlim = (q_end + shift + 63) / 64;
    wg_blk = wlim < all_blk ? wlim : all_blk;
  }
  if (!live) nblk = 0;

  // ---- cooperative fetch of one block: wave instruction j moves pieces [256 j + 64 wave, + 64) of the block, K pieces
  // first (contiguous in memory), then V pieces (piece p = 16 bytes of row p / 2, half p % 2); the piece index is also the
  // position in the slot.  A last block that reaches past its sequence holds whatever codes follow in the buffer (zeros
  // beyond its end): those keys are masked, so their probabilities are exact zeros (and their V scales are replaced below).
  typedef __attribute__((address_space(3))) uint8_t lds_u8;
  auto extent = [](int64_t want, int64_t left) { return (int)(want < left ? want : left); };   // (want < 2^31: checked on the host)
  const int64_t k_off = k_base * (D / 2), v_off = bhk * DV * (int64_t)(a.Sk / 2) + k_first / 2;
  const __amdgpu_buffer_rsrc_t rsrc_k = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.k + k_off), 0, extent((int64_t)all_blk * 64 * (D / 2), a.k_bytes - k_off), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_v = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.vt + v_off), 0, extent((int64_t)DV * (a.Sk / 2) + 32, a.v_bytes - v_off), 0x00020000);
  // Where a piece sits inside its row of the slot: the LDS serves a 16-byte read of 16 lanes per pass from 64 banks
  // (256 bytes), and the 16 lanes of a fragment read ask for the same piece of 16 consecutive rows.  With PR pieces per
  // row, 16 / PR rows share a 256-byte line; piece c of row `row` goes to position c ^ ((row / (16 / PR)) % PR), which
  // spreads those 16 reads over all banks.  (Rows of 96 bytes, D = 192, keep the plain order.)  The loads put the pieces
  // there: lane i of a load fills position p0 + i and fetches the piece that belongs there.
  constexpr int KPR = D / 32, KSW = (KPR == 2 || KPR == 4 || KPR == 8) ? 16 / KPR : 0;   // pieces per K row; rows per swizzle step
  const int n_dma = (PIECES - 64 * wave + 255) / 256;   // this wave's loads per block (wave-uniform)
  auto dma = [&](int kb, int slot) {
    lds_u8* base = (lds_u8*)ring + slot * SLOT;
#pragma unroll
    for (int j = 0; j < DMA_MAX; ++j) {
      const int p0 = 256 * j + 64 * wave;   // wave-uniform
      if (PIECES % 256 != 0 && p0 >= PIECES) continue;
      if (p0 < K_PIECES) {
        const int p = p0 + lane, row = p / KPR;
        const int c = KSW ? (p % KPR) ^ ((row / (KSW ? KSW : 1)) % KPR) : p % KPR;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_k, (__attribute__((address_space(3))) void*)(base + p0 * 16), 16, (row * KPR + c) * 16,
                                                 __builtin_amdgcn_readfirstlane(kb * K_BYTES), 0, 0);
      } else {
        const int p = p0 - K_PIECES + lane, row = p >> 1, column = ND * (row & 31) + (row >> 5);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_v, (__attribute__((address_space(3))) void*)(base + p0 * 16), 16,
                                                 column * (a.Sk / 2) + (((p & 1) ^ ((row >> 3) & 1)) * 16), __builtin_amdgcn_readfirstlane(kb * 32), 0, 0);
      }
    }
  };
  const int kr = score_key(r);                                      // this lane's key of a tile
  const int k_swz = KSW ? ((kr / (KSW ? KSW : 1)) % KPR) * 16 : 0;  // XOR on the byte offset of a piece inside its K row
  const int v_swz = ((r >> 3) & 1) * 16;                            // and inside its 32-byte V row
  auto wait_dma = [&](bool one_block_in_flight) {   // this wave's loads are done, except the youngest block's if asked
    if (!one_block_in_flight) __builtin_amdgcn_s_waitcnt(0x0070 | 0x0F00 | 0);                      // vmcnt(0)
    else if (n_dma == DMA_MAX) __builtin_amdgcn_s_waitcnt(0x0070 | 0x0F00 | (DMA_MAX & 15));        // vmcnt(DMA_MAX)
    else __builtin_amdgcn_s_waitcnt(0x0070 | 0x0F00 | ((DMA_MAX - 1) & 15));
  };
  // Scale bytes of a block: 2 D/32 bytes of K (key tile t, 32-column block j at byte t D/32 + j) and 2 Dv/32 bytes of V
  // (key tile t, column block d at byte t Dv/32 + d) sit at wave-uniform addresses: whole dwords by scalar loads, one block
  // ahead; the MFMA picks a byte of a dword with op_sel, the lane half h shifts its byte into place.  The address is a
  // multiple of 4 except for head dims of 64 and 192, whose 32-row bands have 2 or 6 bytes: a sequence or head that starts
  // at an odd band is then read from the dword below and shifted down by two bytes.
  constexpr int KS_DW = 2 * (D / 32) / 4, VS_DW = (2 * (DV / 32) + 3) / 4;
  constexpr bool K_ODD = (D / 32) % 4 != 0, V_ODD = (DV / 32) % 4 != 0;
  uint32_t ksw[KS_DW], vsw[VS_DW], ksw_next[KS_DW], vsw_next[VS_DW];
  auto fetch = [](const uint8_t* p, auto oddc, auto& w) {
    constexpr int N = sizeof(w) / 4;
    if constexpr (decltype(oddc)::value) {
      const uint32_t odd = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)p & 2u);
      const scalar_u32 q = scalar_ptr(p - odd);
      uint32_t t[N + 1];
#pragma unroll
      for (int i = 0; i < N; ++i) t[i] = q[i];
      t[N] = q[odd ? N : 0];   // (never past the dword that holds the last byte)
#pragma unroll
      for (int i = 0; i < N; ++i) w[i] = (uint32_t)((((uint64_t)t[i + 1] << 32) | t[i]) >> (8 * odd));
    } else {
      const scalar_u32 q = scalar_ptr(p);
#pragma unroll
      for (int i = 0; i < N; ++i) w[i] = q[i];
    }
  };
  auto fetch_scales = [&](int kb, uint32_t (&kw)[KS_DW], uint32_t (&vw)[VS_DW]) {
    const int64_t band = k_base / 32 + kb * 2;
    fetch(a.ks + band * (D / 32), std::bool_constant<K_ODD>{}, kw);
    fetch(a.vs + band * (DV / 32), std::bool_constant<V_ODD>{}, vw);
  };
  if (wg_blk > 0) {
    fetch_scales(0, ksw_next, vsw_next);
    dma(0, 0);
    if (wg_blk > 1) dma(1, 1);
  }
  if constexpr (QBF) {   // behind the first blocks' loads, which then travel with it
    __builtin_amdgcn_s_setprio(3);
    quantize_q<NK>(a.qx + b * a.qx_sb + hq * a.qx_sh + (int64_t)(q_first + (live ? q0 : 0)) * a.qx_ss, a.qx_ss, lane, ring + AttnTile<NK, ND>::QUERY + wave * (NK * 1024), qf, qsc);
    __builtin_amdgcn_s_setprio(0);
  }
  // (the bare barrier instruction: `__syncthreads()` would first wait for every outstanding load, the prefetched block's
  // included; the ring is written by the direct-to-LDS loads only, and wait_dma has waited for this wave's part)
  wait_dma(wg_blk > 1);
  asm volatile("s_barrier" ::: "memory");

  // The block that ends with its first 32 keys, if there is one: the V scale bytes of the other 32 belong to what follows in the
  // buffer, or were never written.  The codes of those probabilities are zeros, but a zero code times the E8M0 NaN (0xFF) is
  // NaN: such bytes become 127.  (Chosen here and compared per block it costs nothing to 1 %; as a comparison of keys beside the
  // mask it cost up to 5 %: six packed sequences of 544 tokens x 16 heads x 128, not causal, 27.2 us without, 27.5 / 28.5.)
  const int half_blk = (kn & 32) != 0 ? kn >> 6 : -1;
  int slot = 0;   // of block kb
  for (int kb = 0; kb < wg_blk; ++kb) {
    const int key0 = kb * 64;
    const uint8_t* tile = ring + slot * SLOT;
#pragma unroll
    for (int i = 0; i < KS_DW; ++i) ksw[i] = ksw_next[i];
#pragma unroll
    for (int i = 0; i < VS_DW; ++i) vsw[i] = vsw_next[i];
    if (kb == half_blk) vsw[VS_DW - 1] = DV == 128 ? 0x7F7F7F7Fu : (vsw[0] & 0xFFFFu) | 0x7F7F0000u;
    // the next block's scale bytes, then the codes of the block after it (into the slot the previous block used: every wave
    // left it at the last barrier); both travel during this block's arithmetic
    if (kb + 1 < wg_blk) fetch_scales(kb + 1, ksw_next, vsw_next);
    if (kb + 2 < wg_blk) dma(kb + 2, slot == 0 ? ATTN_RING - 1 : slot - 1);
    if (kb < nblk) {
      v4f_t bb[BIASED ? 2 : 1][BIASED ? 4 : 1];   // bias of this lane's 32 scores: keys key0 + 32 t + 16 (g / 2) + 8 h + 4 (g % 2) + (0..3)
      if constexpr (BIASED) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const v4i_t w = __builtin_amdgcn_raw_buffer_load_b128(rsrc_bias, (int)((qrow * a.bias_sm + key0 + 32 * t + 16 * (g >> 1) + 8 * h + 4 * (g & 1)) * 4), 0, 0);
            bb[t][g] = __builtin_bit_cast(v4f_t, w);
          }
      }
      // ---- S = Q K^T for two 32-key tiles; K scale of (tile t, step s, half h) = byte t D/32 + 2 s + h
      v16f_t S[2];
      int ksh[KS_DW];
#pragma unroll
      for (int i = 0; i < KS_DW; ++i) ksh[i] = (int)(ksw[i] >> (8 * h));
      static_for<2>([&](auto tc) {
        constexpr int t = decltype(tc)::value;
#pragma unroll
        for (int v = 0; v < 16; ++v) S[t][v] = 0.0f;
        static_for<NK>([&](auto sc) {
          constexpr int s = decltype(sc)::value;
          constexpr int byte = t * (D / 32) + 2 * s;
          const v8i_t kf = frag16(tile + (32 * t + kr) * (D / 2) + ((32 * s + 16 * h) ^ k_swz));
          S[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(kf, qf[s], S[t], 4, 4, byte % 4, ksh[byte / 4], 0, qsc[s]);
        });
      });
      if constexpr (BIASED) {   // scores into the base-2 domain with their additive terms
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int key = key0 + 32 * t + 16 * (v >> 3) + 8 * h + (v & 7);
            float x = __builtin_fmaf(bb[t][v >> 2][v & 3], ATTN_RCP_LN2, S[t][v] * c2);
            x = __builtin_fmaf(-slope2, __builtin_fabsf((float)(qrow + shift - key)), x);
            S[t][v] = x;
          }
      }
      // ---- mask (only blocks the diagonal crosses or that reach past the last key), running max kept in the base-2 domain: m = max(S) * sm_scale * log2(e)
      if ((a.causal && key0 + 63 > q0 + shift) || key0 + 64 > kn) {
        asm volatile("" ::: "memory");   // keep this a branch: most blocks skip it
        mask_scores(S, (a.causal && qrow + shift + 1 < kn ? qrow + shift + 1 : kn) - key0 - 8 * h);
      }
      float tile_max, mx;
      row_maxima<ALONE>(S, tile_max, mx);
      float m_new = max_one(m_i, mx * cs);
      // a bias may hide every key a row has seen so far (-inf): such a row keeps m = -inf and takes exp2(-inf - 0) = 0
      // everywhere instead of exp2(-inf + inf)
      const float m_sub = (BIASED && m_new == -__builtin_inff()) ? 0.0f : m_new;
      const float alpha = __builtin_amdgcn_exp2f(m_i - m_sub);
      m_i = m_new;
      m_new = m_sub;

      v8i_t pf;
      int pscale;
      quantize_probabilities(S, tile_max, cs, m_new, pf, pscale);

      // ---- row sums of the quantised probabilities (a column of ones) and O += P V
      v8i_t vf[ALONE ? ND : 1];
      auto read_v = [&](int d) { return frag16(tile + K_BYTES + (32 * d + r) * 32 + ((16 * h) ^ v_swz)); };
      if constexpr (ALONE) {
#pragma unroll
        for (int d = 0; d < ND; ++d) vf[d] = read_v(d);
      }
      const uint32_t changed = (uint32_t)__builtin_amdgcn_ballot_w64(alpha != 1.0f);   // (both lanes of a row have its alpha)
      if (changed != 0) {
        acc_l[0] *= alpha;   // all registers hold the row sum; only [0] is read
        factors[r] = alpha;
        wave_lds_order();
        v4f_t f[4];   // (all read before the first branch: read in the branches they cost 4 % with D = 128)
#pragma unroll
        for (int g = 0; g < 4; ++g) f[g] = *reinterpret_cast<const v4f_t*>(factors + 8 * g + 4 * h);
        static_for<4>([&](auto gc) {
          constexpr int g = decltype(gc)::value;   // registers 4 g .. + 4 of the two halves: rows 8 g .. + 8
          if (ALONE || changed & (0xFFu << (8 * g))) {
            if constexpr (!ALONE) asm volatile("" ::: "memory");   // keep this a branch
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int d = 0; d < ND; ++d) acc_o[d][4 * g + i] *= f[g][i];
          }
        });
      }
      acc_l = add_row_sums(selector, pf, pscale, acc_l);
      // V scale of (key tile h, this lane's columns ND r .. + ND) = byte h Dv/32 + r / (32 / ND)
      const int vsh = DV == 128 ? (int)((h ? vsw[VS_DW - 1] : vsw[0]) >> (8 * (r >> 3))) : (int)(vsw[0] >> (16 * h + 8 * (r >> 4)));
      static_for<ND>([&](auto dc) {
        constexpr int d = decltype(dc)::value;
        acc_o[d] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(pf, ALONE ? vf[ALONE ? d : 0] : read_v(d), acc_o[d], 4, 4, 0, pscale, 0, vsh);
      });
    }
    wait_dma(kb + 2 < wg_blk);   // block kb + 1 has landed (this wave's part; the barrier collects the others')
    asm volatile("s_barrier" ::: "memory");
    slot = slot == ATTN_RING - 1 ? 0 : slot + 1;
  }
  if (!live) return;

  // ---- O = acc / l, bf16; log-sum-exp.  A lane holds ND consecutive columns of 16 rows: a store instruction writes two whole rows.
  const float l = acc_l[0];
  factors[r] = 1.0f / l;
  wave_lds_order();
  __bf16* o_lane = out + b * a.o_sb + hq * a.o_sh + (int64_t)(q_first + q0 + 4 * h) * a.o_ss + ND * r;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const v4f_t rl = *reinterpret_cast<const v4f_t*>(factors + 8 * g + 4 * h);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      __bf16* o = o_lane + (8 * g + i) * a.o_ss;
      const int v = 4 * g + i;
      const uint32_t w = pack_bf16x2(acc_o[0][v] * rl[i], acc_o[1][v] * rl[i]);
      if constexpr (ND == 4) *reinterpret_cast<uint2*>(o) = make_uint2(w, pack_bf16x2(acc_o[2][v] * rl[i], acc_o[3][v] * rl[i]));
      else *reinterpret_cast<uint32_t*>(o) = w;
    }
  }
  if (h == 0) lse_out[b * a.l_sb + hq * a.l_sh + (q_first + qrow) * a.l_ss] = (m_i + log2f(l)) * ATTN_LN2;
}

template <int NK, int ND, bool BIASED, bool QBF, bool ALONE, typename SEQS>
__global__ __launch_bounds__(256, BIASED ? 2 : ATTN_WG_PER_CU) void attn_fwd_kernel(AttnArgs a, SEQS seqs) {
  __shared__ __attribute__((aligned(16))) uint8_t ring[AttnTile<NK, ND>::QUERY + (QBF ? 4 * NK * 1024 : 0)];
  attn_fwd_body<NK, ND, BIASED, QBF, ALONE>(a, seqs, reinterpret_cast<__bf16*>(a.out), a.lse, ring);
}

template <int NK, int ND, typename SEQS>
static int launch_attn(const AttnArgs& a, const SEQS& seqs, int B, int row_blocks, bool alone, hipStream_t st) {
  dim3 grid((unsigned)a.Hq, (unsigned)B, (unsigned)row_blocks);
  if (a.bias || a.alibi) {
    hipLaunchKernelGGL((attn_fwd_kernel<NK, ND, true, false, false, SEQS>), grid, dim3(256), 0, st, a, seqs);
    return check_launch("attention_fwd");
  }
  if constexpr (NK <= 2) {
    if (alone) {
      if (a.qx) hipLaunchKernelGGL((attn_fwd_kernel<NK, ND, false, true, true, SEQS>), grid, dim3(256), 0, st, a, seqs);
      else hipLaunchKernelGGL((attn_fwd_kernel<NK, ND, false, false, true, SEQS>), grid, dim3(256), 0, st, a, seqs);
      return check_launch("attention_fwd");
    }
  }
  if (a.qx) hipLaunchKernelGGL((attn_fwd_kernel<NK, ND, false, true, false, SEQS>), grid, dim3(256), 0, st, a, seqs);
  else hipLaunchKernelGGL((attn_fwd_kernel<NK, ND, false, false, false, SEQS>), grid, dim3(256), 0, st, a, seqs);
  return check_launch("attention_fwd");
}

// What a call is launched as: the rows of one workgroup, and for 128 of them whether a SIMD has its waves ALONE.
struct LaunchPlan {
  int rows;
  bool alone;
};

// Rows of one workgroup: 32 where its waves deal out the keys (attention_split.hip), 128 where every wave walks them all.
//
// The split kernel takes about 1.6 times the instructions per row and key and a quarter of the time for one row's keys, so it pays while
// the launch is as long as its longest rows, i.e. while its workgroups, each counted as its share of the longest one (6 blocks of keys
// on top for what does not depend on their number), are about as many as are resident at a time: 4 per compute unit with D = 64, 3 with
// 128, 2 above.  How many of these slots may be taken: equal workgroups (all keys) are bound to the round, a causal mask's fill up
// another's end, more so the more blocks there are; up to 8 blocks the start of a workgroup counts for more; the 128 rows of D = 192 wait
// for bank conflicts.  Device time, us, 128 rows / 32 rows, share of the slots in brackets:
//   D = 128, causal: 8 heads x 4096 tokens 60.7 / 34.2 (.73), 14 x 4096 63.9 / 58.1 (1.27), 31 x 2048 36.6 / 38.9 (1.51), 39 x 1024
//   21.1 / 18.6 (1.05), 56 x 1024 22.3 / 25.1 (1.51), 81 x 256 9.0 / 7.8 (.70), 122 x 256 9.5 / 11.0 (1.05);
//   all keys: 6 x 4096 60.7 / 45.3 (1.0), 13 x 2048 33.9 / 34.5 (1.08), 30 x 1024 20.5 / 21.8 (1.25), 101 x 256 9.0 / 10.5 (1.05);
//   D = 192, causal: 8 x 4096 71.7 / 37.5 (1.09), 20 x 2048 42.3 / 32.7 (1.46), 70 x 256 9.8 / 10.3 (.90);
//   D = 256, all keys: 4 x 4096 69.5 / 54.0 (1.0), 10 x 2048 39.3 / 44.6 (1.25), 67 x 256 9.9 / 12.4 (1.05).
// Over 238 shapes at .7 to 1.9 of the slots, the mean loss against the better kernel of each is 1.3 % (D = 192: 4 %).
// Sequences of different lengths, all keys: the workgroups of the short ones fill the ends of the others' as a causal mask's do, from 16
// blocks on (2016 tokens in two sequences, 16 heads of 128: 33.5 / 25.2 (1.14), 36.0 / 32.6 (1.19), 39.9 / 35.5 (1.30); 3360 in seven, 16 of 64:
// 30.5 / 28.3 (1.17), 27.6 / 26.7 (1.19), with 14 blocks 22.2 / 23.6 (1.31); 4096 in three, 8 of 128: 37.3 / 37.9 (1.23); 2976 in six, 20 of 64:
// 27.9 / 27.5 (1.32), 30.5 / 29.6 (1.37), with 11 blocks 21.1 / 23.9 (1.58)).
// Packed sequences of one length are equal workgroups like a batch's: D = 128 keeps to the batch's line while the 128 rows have a compute unit
// for each workgroup (two of 1024: 13 heads 26.5 / 28.0 (1.08), 16 heads 28.2 / 29.9 (1.33); three of 1536, 7 heads 35.3 / 37.1 (1.31)) and goes on
// once they do not (two of 1280, 13 heads 36.2 / 33.9 (1.35); three of 1344, 8 heads 38.5 / 34.7 (1.31)); D = 64 goes on from 20 blocks
// (three of 1024, 14 heads 27.4 / 28.1 (1.31); two of 1536, 14 heads 35.8 / 35.0 (1.31); two of 2048, 11 heads 43.4 / 42.7 (1.38)).
// Packed sequences are weighed all together, also where there are more than one launch holds (64): such a call keeps to 128 rows
// sooner than each of its launches by itself would have to.
//
// ALONE: all keys, heads of 64 and 128, up to one 128-row workgroup a unit; two with heads of 64, and a few more with sequences of different
// lengths, whose long ones end alone.  us without / with (and the kernel with O's rows in lanes, which had no groups to branch over):
//   D = 128: 14 heads x 2048 tokens (224 workgroups) 40.0 / 39.7 (39.4), 16 x 2048 (256) 41.1 / 40.7 (39.7), 4 x 8 x 1024 (256) 27.4 / 26.8 (26.8), two packed
//   of 1024, 16 heads 27.4 / 26.7 (26.5); beyond: 9 x 4096 (288) .947 / .986 of the old time, 12 x 4096 (384) .939 / .975;
//   eight of 4064 tokens, 12 heads (408) 35.2 / 34.3 (34.4), 16 heads (544) 35.5 / 34.8 (34.9), 20 heads (680) .934 / .951 of the old time;
//   D = 64: 40 x 1024 (320) 24.9 / 24.2 (24.6), 64 x 1024 (512) 27.2 / 26.7 (26.9), 16 x 4096 (512) 77.3 / 77.0 (78.3), eight of 4064, 16 heads (544) 28.7 / 28.0
//   (27.8); beyond: 20 x 4096 (640) .918 / .948, 96 x 1024 (768) .957 / .967 of the old time.
// A causal mask fills up the units with other workgroups (all at .90 to .98 of the old time without), and D = 192 and 256 gain nothing.
static LaunchPlan launch_plan(const AttnArgs& a, int64_t B, int64_t D, int n_seqs, const int32_t* cu_q, const int32_t* cu_k) {
  if (a.bias || a.alibi || a.Sq / 32 > 65535) return {128, false};
  double work = 0.0;
  int64_t longest = 0, rows_128 = 0;   // rows_128: workgroups of 128 rows
  bool equal = true;
  for (int i = 0; i < (n_seqs ? n_seqs : 1); ++i) {
    const int64_t bands = (n_seqs ? cu_q[i + 1] - cu_q[i] : a.Sq) / 32, n = ((n_seqs ? cu_k[i + 1] - cu_k[i] : a.Sk_used) + 63) / 64;
    work += (double)bands * (double)(n + 6) - (a.causal ? 0.25 * (double)bands * (double)(bands - 1) : 0.0);   // (a causal band ends half a block before the next)
    longest = n > longest ? n : longest;
    rows_128 += (bands + 3) / 4;
    if (n_seqs) equal = equal && cu_q[i + 1] - cu_q[i] == cu_q[1] - cu_q[0] && cu_k[i + 1] - cu_k[i] == cu_k[1] - cu_k[0];
  }
  const int per_cu = D == 64 ? 4 : (D == 128 ? 3 : 2);
  const bool wide = n_seqs > 1 && !a.causal && longest >= 16 && D <= 128 && (!equal || (D == 64 ? longest >= 20 : B * a.Hq * rows_128 > 256));
  const double share = longest <= 8 ? 0.95 : (D == 192 || wide ? 1.4 : (a.causal ? (longest >= 48 ? 1.3 : 1.125) : (D == 64 ? 1.125 : 1.02)));
  if ((double)B * a.Hq * work <= 256.0 * share * per_cu * (double)(longest + 6)) return {32, false};
  return {128, !a.causal && D <= 128 && B * a.Hq * rows_128 <= (!equal ? 576 : (D == 64 ? 512 : 256))};
}

template <typename SEQS>
static int launch_attn_dims(const AttnArgs& a, const SEQS& seqs, int B, int row_blocks, const LaunchPlan& plan, int64_t D, int64_t Dv, hipStream_t st) {
  if (plan.rows == 32) return launch_attn_split(a, seqs, B, row_blocks, D, Dv, st);
  switch (D + (Dv == 128 ? 1 : 0)) {
    case 64: return launch_attn<1, 2>(a, seqs, B, row_blocks, plan.alone, st);
    case 65: return launch_attn<1, 4>(a, seqs, B, row_blocks, plan.alone, st);
    case 128: return launch_attn<2, 2>(a, seqs, B, row_blocks, plan.alone, st);
    case 129: return launch_attn<2, 4>(a, seqs, B, row_blocks, plan.alone, st);
    case 192: return launch_attn<3, 2>(a, seqs, B, row_blocks, plan.alone, st);
    case 193: return launch_attn<3, 4>(a, seqs, B, row_blocks, plan.alone, st);
    case 256: return launch_attn<4, 2>(a, seqs, B, row_blocks, plan.alone, st);
    case 257: return launch_attn<4, 4>(a, seqs, B, row_blocks, plan.alone, st);
  }
  return ALTO_MXFP4_EINVAL;
}

}  // namespace alto

extern "C" int alto_mxfp4_attention_fwd_ex(const void* q_codes, const void* q_scales, const void* k_codes, const void* k_scales,
                                           const void* vt_codes, const void* v_scales, void* out, float* lse, int64_t B, int64_t Hq,
                                           int64_t Hk, int64_t Sq, int64_t Sk, int64_t Sk_used, int64_t D, int64_t Dv, float sm_scale,
                                           int causal, const float* bias, int64_t bias_sb, int64_t bias_sh, int64_t bias_sm,
                                           const float* alibi_slopes, int64_t alibi_sb, int64_t alibi_sh, void* stream) {
  using namespace alto;
  ALTO_REQUIRE(!alibi_slopes || (alibi_sb >= 0 && alibi_sh >= 0), "attention_fwd: negative alibi strides");
  ALTO_REQUIRE(q_codes && q_scales && k_codes && k_scales && vt_codes && v_scales && out && lse, "attention_fwd: null pointer");
  ALTO_REQUIRE(B > 0 && Hq > 0 && Hk > 0 && Hq % Hk == 0, "attention_fwd: Hq=%lld must be a positive multiple of Hk=%lld", (long long)Hq, (long long)Hk);
  ALTO_REQUIRE(Sq > 0 && Sq % 32 == 0, "attention_fwd: Sq=%lld must be a positive multiple of 32", (long long)Sq);
  ALTO_REQUIRE(Sk > 0 && Sk % 64 == 0, "attention_fwd: Sk=%lld must be a positive multiple of 64", (long long)Sk);
  ALTO_REQUIRE(D == 64 || D == 128 || D == 192 || D == 256, "attention_fwd: head dim D=%lld must be 64, 128, 192 or 256", (long long)D);
  ALTO_REQUIRE(Dv == 64 || Dv == 128, "attention_fwd: value dim Dv=%lld must be 64 or 128", (long long)Dv);
  ALTO_REQUIRE(Sk_used > 0 && Sk_used <= Sk && Sk - Sk_used < 64 && Sk_used % 32 == 0,
               "attention_fwd: Sk_used=%lld must be a multiple of 32 in (Sk - 64, Sk]", (long long)Sk_used);
  ALTO_REQUIRE(!causal || Sq <= Sk_used, "attention_fwd: causal attention needs Sq <= Sk (got %lld > %lld)", (long long)Sq, (long long)Sk_used);
  ALTO_REQUIRE(B <= 65535 && (Sq + 127) / 128 <= 65535, "attention_fwd: B and Sq / 128 must fit a grid dimension");
  ALTO_REQUIRE(Hq < (1ll << 31) && Sk < (1ll << 31) && product_below(1ll << 40, B * Sq, Hq, D > Dv ? D : Dv), "attention_fwd: tensor too large");
  int64_t bias_bytes = 0;
  if (bias) {   // (B, Hq, Sq and Sk_used are in range here)
    ALTO_REQUIRE(bias_sb >= 0 && bias_sh >= 0 && bias_sm >= Sk_used && bias_sm % 4 == 0 && (uintptr_t)bias % 16 == 0,
                 "attention_fwd: bias rows must be 16-byte aligned with unit stride along the keys (row stride %lld)", (long long)bias_sm);
    ALTO_REQUIRE(product_below(1ll << 29, Sq, bias_sm) && product_below(1ll << 30, B - 1, bias_sb) && product_below(1ll << 30, Hq - 1, bias_sh),
                 "attention_fwd: bias tensor too large");
    bias_bytes = ((B - 1) * bias_sb + (Hq - 1) * bias_sh + (Sq - 1) * bias_sm + Sk_used) * 4;
    ALTO_REQUIRE(bias_bytes < (1ll << 32), "attention_fwd: bias tensor too large");
  }
  ALTO_REQUIRE(((uintptr_t)q_codes | (uintptr_t)k_codes | (uintptr_t)vt_codes) % 16 == 0 && (uintptr_t)out % 8 == 0,
               "attention_fwd: code pointers must be 16-byte aligned, out 8-byte aligned");
  ALTO_REQUIRE(((uintptr_t)k_scales | (uintptr_t)v_scales | (uintptr_t)lse | (uintptr_t)alibi_slopes) % 4 == 0,
               "attention_fwd: K and V scale pointers, lse and the alibi slopes must be 4-byte aligned");
  AttnArgs a{(const uint8_t*)q_codes, (const uint8_t*)q_scales, nullptr, 0, 0, 0, (const uint8_t*)k_codes, (const uint8_t*)k_scales,
             (const uint8_t*)vt_codes, (const uint8_t*)v_scales, out, lse, Hq * Sq * Dv, Sq * Dv, Dv, Hq * Sq, Sq, 1, (int)Hq, (int)Hk, (int)Sq, (int)Sk,
             (int)Sk_used, B * Hk * Sk * (D / 2), B * Hk * Dv * (Sk / 2), sm_scale, causal ? 1 : 0,
             bias, bias_sb, bias_sh, bias_sm, bias_bytes, alibi_slopes, alibi_sb, alibi_sh};
  const LaunchPlan plan = launch_plan(a, B, D, 0, nullptr, nullptr);
  return launch_attn_dims(a, AttnNoSeqs{}, (int)B, (int)((Sq + plan.rows - 1) / plan.rows), plan, D, Dv, (hipStream_t)stream);
}

namespace alto {
// Q as the strided entries get it: quantized codes and scales, or bf16 values at element strides
struct QueryOperand {
  const void* codes;
  const void* scales;
  const void* values;
  int64_t sb, sh, ss;
};

static int check_boundaries(int64_t B, int64_t Sq, int64_t Sk, int n_seqs, const int32_t* cu_q, const int32_t* cu_k, int causal) {
  ALTO_REQUIRE(n_seqs > 0 && cu_q && cu_k && B == 1, "attention_fwd: packed sequences need their boundaries and B = 1");
  ALTO_REQUIRE(cu_q[0] == 0 && cu_k[0] == 0 && cu_q[n_seqs] == Sq && cu_k[n_seqs] == Sk, "attention_fwd: the sequence boundaries must run from 0 to the token counts");
  for (int i = 0; i < n_seqs; ++i) {
    ALTO_REQUIRE(cu_q[i + 1] > cu_q[i] && cu_k[i + 1] > cu_k[i] && cu_q[i + 1] % 32 == 0 && cu_k[i + 1] % 32 == 0,
                 "attention_fwd: sequence boundaries must be increasing multiples of 32 tokens");
    ALTO_REQUIRE(!causal || cu_q[i + 1] - cu_q[i] <= cu_k[i + 1] - cu_k[i], "attention_fwd: causal attention needs Sq <= Sk (got %d > %d)", cu_q[i + 1] - cu_q[i],
                 cu_k[i + 1] - cu_k[i]);
  }
  return ALTO_MXFP4_OK;
}

static int attention_fwd_strided(const QueryOperand& q, const void* k_codes, const void* k_scales, const void* vt_codes, const void* v_scales, void* out,
                                 float* lse, int64_t B, int64_t Hq, int64_t Hk, int64_t Sq, int64_t Sk, int64_t D, int64_t Dv, int64_t o_sb, int64_t o_sh,
                                 int64_t o_ss, int64_t l_sb, int64_t l_sh, int64_t l_ss, int n_seqs, const int32_t* cu_q, const int32_t* cu_k, float sm_scale,
                                 int causal, const float* alibi_slopes, int64_t alibi_sb, int64_t alibi_sh, hipStream_t st) {
  ALTO_REQUIRE(B > 0 && Hq > 0 && Hk > 0 && Hq % Hk == 0, "attention_fwd: Hq=%lld must be a positive multiple of Hk=%lld", (long long)Hq, (long long)Hk);
  ALTO_REQUIRE(Sq > 0 && Sq % 32 == 0 && Sk > 0 && Sk % 32 == 0, "attention_fwd: Sq=%lld and Sk=%lld must be positive multiples of 32", (long long)Sq, (long long)Sk);
  ALTO_REQUIRE(D == 64 || D == 128 || D == 192 || D == 256, "attention_fwd: head dim D=%lld must be 64, 128, 192 or 256", (long long)D);
  ALTO_REQUIRE(Dv == 64 || Dv == 128, "attention_fwd: value dim Dv=%lld must be 64 or 128", (long long)Dv);
  ALTO_REQUIRE(B <= 65535 && Sq < (1ll << 31) && Sk < (1ll << 31) && Hq < (1ll << 31), "attention_fwd: size out of range");
  ALTO_REQUIRE(product_below(1ll << 40, B * Sq, Hq, D > Dv ? D : Dv) && product_below(1ll << 40, B * Sk, Hk, D > Dv ? D : Dv) && product_below(1ll << 31, Sk, D) &&
                   product_below(1ll << 31, Sk, Dv), "attention_fwd: tensor too large");
  ALTO_REQUIRE(o_sb >= 0 && o_sh >= 0 && o_ss >= 0 && l_sb >= 0 && l_sh >= 0 && l_ss >= 0 && (o_sb | o_sh | o_ss) % 4 == 0,
               "attention_fwd: output strides must be non-negative, those of out multiples of 4 elements");
  ALTO_REQUIRE((o_sb | o_sh | o_ss | l_sb | l_sh | l_ss) < (1ll << 40), "attention_fwd: output stride out of range");
  ALTO_REQUIRE(((uintptr_t)q.codes | (uintptr_t)q.values | (uintptr_t)k_codes | (uintptr_t)vt_codes) % 16 == 0 && (uintptr_t)out % 8 == 0,
               "attention_fwd: operand pointers must be 16-byte aligned, out 8-byte aligned");
  ALTO_REQUIRE(((uintptr_t)k_scales | (uintptr_t)v_scales | (uintptr_t)lse | (uintptr_t)alibi_slopes) % 4 == 0,
               "attention_fwd: K and V scale pointers, lse and the alibi slopes must be 4-byte aligned");
  AttnArgs a{(const uint8_t*)q.codes, (const uint8_t*)q.scales, (const __bf16*)q.values, q.sb, q.sh, q.ss, (const uint8_t*)k_codes, (const uint8_t*)k_scales,
             (const uint8_t*)vt_codes, (const uint8_t*)v_scales, out, lse, o_sb, o_sh, o_ss, l_sb, l_sh, l_ss, (int)Hq, (int)Hk, (int)Sq, (int)Sk,
             (int)Sk, B * Hk * Sk * (D / 2), B * Hk * Dv * (Sk / 2), sm_scale, causal ? 1 : 0, nullptr, 0, 0, 0, 0, alibi_slopes, alibi_sb, alibi_sh};
  if (n_seqs == 0) {
    ALTO_REQUIRE(!causal || Sq <= Sk, "attention_fwd: causal attention needs Sq <= Sk (got %lld > %lld)", (long long)Sq, (long long)Sk);
    ALTO_REQUIRE((Sq + 127) / 128 <= 65535, "attention_fwd: Sq / 128 must fit a grid dimension");
    const LaunchPlan plan = launch_plan(a, B, D, 0, nullptr, nullptr);
    return launch_attn_dims(a, AttnNoSeqs{}, (int)B, (int)((Sq + plan.rows - 1) / plan.rows), plan, D, Dv, st);
  }
  if (const int rc = check_boundaries(B, Sq, Sk, n_seqs, cu_q, cu_k, causal)) return rc;
  // longest sequences first, up to ATTN_MAX_SEQS of them and 65535 row blocks per launch
  std::unique_ptr<int[]> order(new (std::nothrow) int[(size_t)n_seqs]);   // (no exception may leave a C entry)
  if (!order) {
    set_error("attention_fwd: no host memory for the order of %d sequences", n_seqs);
    return ALTO_MXFP4_ELAUNCH;
  }
  for (int i = 0; i < n_seqs; ++i) order[(size_t)i] = i;
  std::sort(order.get(), order.get() + n_seqs, [&](int x, int y) {
    const int kx = cu_k[x + 1] - cu_k[x], ky = cu_k[y + 1] - cu_k[y];
    return kx != ky ? kx > ky : x < y;
  });
  const LaunchPlan plan = launch_plan(a, 1, D, n_seqs, cu_q, cu_k);
  const int rows = plan.rows;
  for (int at = 0; at < n_seqs;) {
    AttnSeqs t;
    t.n = 0;
    t.z0[0] = 0;
    for (; at < n_seqs && t.n < ATTN_MAX_SEQS; ++at) {
      const int s = order[(size_t)at], qn = cu_q[s + 1] - cu_q[s], blocks = (qn + rows - 1) / rows;
      ALTO_REQUIRE(blocks <= 65535, "attention_fwd: Sq / 128 must fit a grid dimension");
      if (t.z0[t.n] + blocks > 65535) break;
      t.q0[t.n] = cu_q[s]; t.qn[t.n] = qn; t.k0[t.n] = cu_k[s]; t.kn[t.n] = cu_k[s + 1] - cu_k[s];
      t.z0[t.n + 1] = t.z0[t.n] + blocks;
      ++t.n;
    }
    const int rc = launch_attn_dims(a, t, 1, t.z0[t.n], plan, D, Dv, st);
    if (rc != ALTO_MXFP4_OK) return rc;
  }
  return ALTO_MXFP4_OK;
}
}  // namespace alto

extern "C" int alto_mxfp4_attention_fwd_strided(const void* q_codes, const void* q_scales, const void* k_codes, const void* k_scales,
                                                const void* vt_codes, const void* v_scales, void* out, float* lse, int64_t B, int64_t Hq,
                                                int64_t Hk, int64_t Sq, int64_t Sk, int64_t D, int64_t Dv, int64_t o_sb, int64_t o_sh, int64_t o_ss,
                                                int64_t l_sb, int64_t l_sh, int64_t l_ss, int n_seqs, const int32_t* cu_q, const int32_t* cu_k,
                                                float sm_scale, int causal, const float* alibi_slopes, int64_t alibi_sb, int64_t alibi_sh, void* stream) {
  ALTO_REQUIRE(q_codes && q_scales && k_codes && k_scales && vt_codes && v_scales && out && lse, "attention_fwd: null pointer");
  ALTO_REQUIRE(!alibi_slopes || (alibi_sb >= 0 && alibi_sh >= 0), "attention_fwd: negative alibi strides");
  return alto::attention_fwd_strided({q_codes, q_scales, nullptr, 0, 0, 0}, k_codes, k_scales, vt_codes, v_scales, out, lse, B, Hq, Hk, Sq, Sk, D, Dv, o_sb, o_sh, o_ss,
                                     l_sb, l_sh, l_ss, n_seqs, cu_q, cu_k, sm_scale, causal, alibi_slopes, alibi_sb, alibi_sh, (hipStream_t)stream);
}

extern "C" int alto_mxfp4_attention_fwd_bf16q(const void* q, int64_t q_sb, int64_t q_sh, int64_t q_ss, const void* k_codes, const void* k_scales,
                                              const void* vt_codes, const void* v_scales, void* out, float* lse, int64_t B, int64_t Hq, int64_t Hk,
                                              int64_t Sq, int64_t Sk, int64_t D, int64_t Dv, int64_t o_sb, int64_t o_sh, int64_t o_ss, int64_t l_sb,
                                              int64_t l_sh, int64_t l_ss, int n_seqs, const int32_t* cu_q, const int32_t* cu_k, float sm_scale, int causal,
                                              void* stream) {
  ALTO_REQUIRE(q && k_codes && k_scales && vt_codes && v_scales && out && lse, "attention_fwd: null pointer");
  for (int64_t s : {q_sb, q_sh, q_ss})
    ALTO_REQUIRE(s >= 0 && s < (1ll << 44) && s % 8 == 0, "attention_fwd: strides of q must be non-negative multiples of 8 elements");
  return alto::attention_fwd_strided({nullptr, nullptr, q, q_sb, q_sh, q_ss}, k_codes, k_scales, vt_codes, v_scales, out, lse, B, Hq, Hk, Sq, Sk, D, Dv, o_sb, o_sh, o_ss,
                                     l_sb, l_sh, l_ss, n_seqs, cu_q, cu_k, sm_scale, causal, nullptr, 0, 0, (hipStream_t)stream);
}

extern "C" int alto_mxfp4_attention_rows_per_workgroup(int64_t B, int64_t Hq, int64_t Sq, int64_t Sk, int64_t D, int n_seqs, const int32_t* cu_q, const int32_t* cu_k,
                                                       int causal) {
  using namespace alto;
  ALTO_REQUIRE(B > 0 && Hq > 0 && Sq > 0 && Sk > 0, "attention_rows_per_workgroup: sizes must be positive");
  ALTO_REQUIRE(B < (1ll << 31) && Hq < (1ll << 31) && Sq < (1ll << 31) && Sk < (1ll << 31), "attention_rows_per_workgroup: size out of range");
  if (n_seqs != 0)
    if (const int rc = check_boundaries(B, Sq, Sk, n_seqs, cu_q, cu_k, causal)) return rc;
  AttnArgs a{};
  a.Hq = (int)Hq; a.Sq = (int)Sq; a.Sk_used = (int)Sk; a.causal = causal ? 1 : 0;
  return launch_plan(a, B, D, n_seqs, cu_q, cu_k).rows;
}

extern "C" int alto_mxfp4_attention_fwd(const void* q_codes, const void* q_scales, const void* k_codes, const void* k_scales,
                                        const void* vt_codes, const void* v_scales, void* out, float* lse, int64_t B, int64_t Hq,
                                        int64_t Hk, int64_t Sq, int64_t Sk, int64_t Sk_used, int64_t D, int64_t Dv, float sm_scale,
                                        int causal, void* stream) {
  return alto_mxfp4_attention_fwd_ex(q_codes, q_scales, k_codes, k_scales, vt_codes, v_scales, out, lse, B, Hq, Hk, Sq, Sk, Sk_used, D, Dv, sm_scale,
                                     causal, nullptr, 0, 0, 0, nullptr, 0, 0, stream);
}
