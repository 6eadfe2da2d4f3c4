// MXFP4 flash-attention forward for launches that cannot fill the chip with one wave per 32 rows (attention.hip): the four waves
// of a workgroup share 32 query rows of one head and deal the key blocks out.
//
// What a probability code is depends on the running row maximum, i.e. on all earlier blocks, and the sums over the blocks have an
// order, so the keys cannot simply be cut in four.  In round n, wave w takes block 4 n + w:
//   A(n)  scores of the block, their row maxima to the LDS;
//   B(n)  running maxima of the round's four blocks (four values a row), probability codes of the block and its rescale factors to
//         the LDS: 1.5 KB;
//   C(n)  wave d walks the round's four blocks in order and multiplies the codes with its 32 columns of V.
// Each probability, each rescale and each accumulator sees the same operations in the same order as in attention.hip: the results
// are the same bit for bit, whichever of the two runs.  C(n) runs beside B(n + 1) (independent instructions in one stretch of
// code, one barrier a round between A and the two), so the chain through the accumulators hides behind the softmax, which is most
// of the work and runs on four SIMDs.  K and V pieces go from global memory straight to registers (a workgroup's waves read
// different pieces), a round ahead.  A wave without a block in the last round computes on the last block again and contributes
// -inf as its maximum; nobody reads its codes.
#include "attention.h"

namespace alto {
namespace {

// (LDS writes of this wave done, then the barrier; loads stay in flight, unlike behind __syncthreads())
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int NK, int ND>
struct SplitLds {   // codes, scale bytes and rescale factors of two rounds; row maxima of two rounds
  static constexpr int CODES = 0, AUX = 8 * 1024, MAXIMA = AUX + 8 * 512, BYTES = MAXIMA + 8 * 128;
  // Q's codes and scales lie in the slots of round 0, which B(0) writes behind a barrier; the result rows replace the last codes
  static_assert(NK <= 4 && 32 * ND * 32 * 2 <= MAXIMA, "");
};

template <int NK, int ND, bool QBF, typename SEQS>
__device__ __forceinline__ void attn_split_body(const AttnArgs& a, const SEQS& seqs, __bf16* __restrict__ out, float* __restrict__ lse_out, uint8_t* lds) {
  using L = SplitLds<NK, ND>;
  constexpr int D = NK * 64, DV = ND * 32, K_BYTES = 64 * (D / 2), KS_DW = D / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  const AttnRows w = attn_rows(a, seqs, (int)blockIdx.z, (int)gridDim.z);
  const int kn = w.kn, q0 = w.block * 32, shift = kn - w.qn, qrow = q0 + r;
  const int hq = attn_head(a), b = blockIdx.y, hk = hq / (a.Hq / a.Hk);
  const int64_t q_base = ((int64_t)b * a.Hq + hq) * a.Sq + w.q_first, bhk = (int64_t)b * a.Hk + hk, k_base = bhk * a.Sk + w.k_first;
  const int all_blk = (kn + 63) / 64;
  int nblk = all_blk;
  if (a.causal) {
    const int lim = (q0 + 32 + shift + 63) / 64;
    nblk = lim < all_blk ? lim : all_blk;
  }
  // Parts of C: role d < ND has the output columns 32 d .. + 32, role SUMS the row sums.  Dealt differently from workgroup to
  // workgroup, since wave w of each is on the same SIMD.
  constexpr int SUMS = ND == 2 ? 2 : 0;
  const unsigned id = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  const int role = (wave + (int)(id + (id >> 8))) & 3;
  const int half_blk = (kn & 32) != 0 ? kn >> 6 : -1;   // the block whose second half does not exist

  // ---- K pieces of this wave's blocks (as attention.hip's fragments) and the 2 D/32 scale bytes of each (2-byte aligned).  A last
  // block that reaches past its sequence reads what follows in the buffer (zeros beyond its end); those keys are masked.
  auto extent = [](int64_t want, int64_t left) { return (int)(want < left ? want : left); };
  const int64_t k_off = k_base * (D / 2), v_off = bhk * DV * (int64_t)(a.Sk / 2) + w.k_first / 2;
  const __amdgpu_buffer_rsrc_t rsrc_k = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.k + k_off), 0, extent((int64_t)all_blk * K_BYTES, a.k_bytes - k_off), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_v = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.vt + v_off), 0, extent((int64_t)DV * (a.Sk / 2) + 32, a.v_bytes - v_off), 0x00020000);
  struct __attribute__((packed, aligned(2))) KScales { uint32_t w[KS_DW]; };
  v4i_t kf[2][NK];
  KScales ksc;
  auto load_k = [&](int kb) {
    kb = kb < nblk ? kb : nblk - 1;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int s = 0; s < NK; ++s) kf[t][s] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_k, (32 * t + score_key(r)) * (D / 2) + 32 * s + 16 * h, kb * K_BYTES, 0);
    ksc = *reinterpret_cast<const KScales*>(a.ks + (k_base / 32 + kb * 2) * (D / 32));
  };
  load_k(wave);

  // ---- Q pieces, as in attention.hip; from bf16, wave s quantizes step s for all
  v8i_t qf[NK];
  int qsc[NK];
  if constexpr (QBF) {
    if (wave < NK) {
      v8i_t f[1];
      int e[1];
      quantize_q<1>(a.qx + b * a.qx_sb + hq * a.qx_sh + (int64_t)(w.q_first + q0) * a.qx_ss + 64 * wave, a.qx_ss, lane, lds + wave * 1024, f, e);
      reinterpret_cast<int*>(lds + L::AUX)[wave * 64 + lane] = e[0];
    }
    lds_barrier();
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      qf[s] = frag16(lds + s * 1024 + r * 32 + h * 16);
      qsc[s] = reinterpret_cast<const int*>(lds + L::AUX)[s * 64 + lane];
    }
  } else {
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      qf[s] = frag16(a.q + (q_base + qrow) * (D / 2) + s * 32 + h * 16);
      qsc[s] = a.qs[(q_base / 32 + qrow / 32) * (D / 32) + 2 * s + h];
    }
  }

  v16f_t acc_o;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc_o[v] = 0.0f;
  v4f_t acc_l = {0.0f, 0.0f, 0.0f, 0.0f};
  float m_i = -__builtin_inff();
  const float cs = a.sm_scale * ATTN_RCP_LN2;
  const int selector = row_sum_selector(lane);

  // ---- V pieces of this wave's columns: row 32 role + r of V^T; scale byte of (key tile h, column block role)
  v4i_t vf[4];
  int vsc[4];
  auto load_v = [&](int first) {
    const int d = role < ND ? role : 0;   // (with 64 columns, two waves have none)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kb = first + i < nblk ? first + i : nblk - 1;
      vf[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_v, (32 * d + r) * (a.Sk / 2) + 16 * h, kb * 32, 0);
      const uint8_t* band = a.vs + (k_base / 32 + kb * 2) * ND;
      vsc[i] = band[(unsigned)(h * ND + d)];
    }
  };
  v16f_t S[2];
  float tile_max;
  auto phase_a = [&](int first, int buf) {
    const int kb = first + wave, key0 = kb * 64;
    int ksh[KS_DW];
#pragma unroll
    for (int i = 0; i < KS_DW; ++i) ksh[i] = (int)(ksc.w[i] >> (8 * h));
    static_for<2>([&](auto tc) {
      constexpr int t = decltype(tc)::value;
#pragma unroll
      for (int v = 0; v < 16; ++v) S[t][v] = 0.0f;
      static_for<NK>([&](auto sc) {
        constexpr int s = decltype(sc)::value, byte = t * (D / 32) + 2 * s;
        const v4i_t f = kf[t][s];
        S[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(v8i_t{f[0], f[1], f[2], f[3], 0, 0, 0, 0}, qf[s], S[t], 4, 4, byte % 4, ksh[byte / 4], 0, qsc[s]);
      });
    });
    load_k(kb + 4);
    if ((a.causal && key0 + 63 > q0 + shift) || key0 + 64 > kn) {
      asm volatile("" ::: "memory");   // keep this a branch: most blocks skip it
      mask_scores(S, (a.causal && qrow + shift + 1 < kn ? qrow + shift + 1 : kn) - key0 - 8 * h);
    }
    float mx;
    row_maxima<false>(S, tile_max, mx);
    mx = kb < nblk ? mx * cs : -__builtin_inff();
    reinterpret_cast<float*>(lds + L::MAXIMA)[(4 * buf + wave) * 32 + r] = mx;   // (both lanes of a row hold it)
  };
  auto phase_b = [&](int buf) {
    float m_old = 0.0f, m_new = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float m = fmaxf(m_i, reinterpret_cast<const float*>(lds + L::MAXIMA)[(4 * buf + i) * 32 + r]);
      m_old = i == wave ? m_i : m_old;
      m_new = i == wave ? m : m_new;
      m_i = m;
    }
    const float alpha = __builtin_amdgcn_exp2f(m_old - m_new);
    v8i_t pf;
    int pscale;
    quantize_probabilities(S, tile_max, cs, m_new, pf, pscale);
    const int slot = (4 * buf + wave) * 64 + lane;
    reinterpret_cast<v4i_t*>(lds + L::CODES)[slot] = v4i_t{pf[0], pf[1], pf[2], pf[3]};
    reinterpret_cast<uint2*>(lds + L::AUX)[slot] = make_uint2(f2u(alpha), (uint32_t)pscale);
  };
  // C: O += P V, then the row sums, in the order of the blocks.  (The codes are read ahead of B's arithmetic, which gains 1 to 3 %, where
  // their 24 registers do not cost a workgroup per compute unit: with D = 64 that loses 8 to 12 %.)
  uint2 aux[4];
  v4i_t codes[4];
  auto read_codes = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      aux[i] = reinterpret_cast<const uint2*>(lds + L::AUX)[(4 * buf + i) * 64 + lane];
      codes[i] = reinterpret_cast<const v4i_t*>(lds + L::CODES)[(4 * buf + i) * 64 + lane];
    }
  };
  auto phase_c = [&](int first, auto tailc) {
    constexpr bool TAIL = decltype(tailc)::value;
    if (ND == 4 || role < ND) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (!TAIL || first + i < nblk) {
          const float alpha = u2f(aux[i].x);
#pragma unroll
          for (int v = 0; v < 16; ++v) acc_o[v] *= alpha;
          const int vs = TAIL && first + i == half_blk && h != 0 ? 127 : vsc[i];   // (a scale byte nobody wrote may be the E8M0 NaN)
          acc_o = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(v8i_t{vf[i][0], vf[i][1], vf[i][2], vf[i][3], 0, 0, 0, 0},
                                                                  v8i_t{codes[i][0], codes[i][1], codes[i][2], codes[i][3], 0, 0, 0, 0}, acc_o, 4, 4, 0, vs, 0, (int)aux[i].y);
        }
    }
    if (role == SUMS) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (!TAIL || first + i < nblk) {
          acc_l[0] *= u2f(aux[i].x);   // all registers hold the row sum; only [0] is read
          acc_l = add_row_sums(selector, v8i_t{codes[i][0], codes[i][1], codes[i][2], codes[i][3], 0, 0, 0, 0}, (int)aux[i].y, acc_l);
        }
    }
  };

  // round -1 adds nothing: codes of zero, factors of one
  {
    const int slot = (4 + wave) * 64 + lane;
    reinterpret_cast<v4i_t*>(lds + L::CODES)[slot] = v4i_t{0, 0, 0, 0};
    reinterpret_cast<uint2*>(lds + L::AUX)[slot] = make_uint2(f2u(1.0f), 127u);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      vf[i] = v4i_t{0, 0, 0, 0};
      vsc[i] = 127;
    }
  }
  int first = 0, buf = 0;
  for (;; first += 4, buf ^= 1) {
    phase_a(first, buf);
    lds_barrier();
    if constexpr (NK > 1) read_codes(buf ^ 1);
    phase_b(buf);
    if constexpr (NK == 1) read_codes(buf ^ 1);
    phase_c(0, std::false_type{});
    load_v(first);
    if (first + 4 >= nblk) break;
  }
  lds_barrier();
  read_codes(buf);
  phase_c(first, std::true_type{});

  // ---- O = acc / l, bf16, stored as whole rows (as in attention.hip); log-sum-exp
  constexpr int PR = DV / 8;
  if (role == SUMS) {
    if (h == 0) lse_out[b * a.l_sb + hq * a.l_sh + (w.q_first + qrow) * a.l_ss] = (m_i + log2f(acc_l[0])) * ATTN_LN2;
    reinterpret_cast<float*>(lds + L::MAXIMA)[r] = acc_l[0];
  }
  lds_barrier();   // (everybody has read the last codes as well)
  const float rl = 1.0f / reinterpret_cast<const float*>(lds + L::MAXIMA)[r];
  if (role < ND) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      uint2 o;
      o.x = pack_bf16x2(acc_o[4 * g + 0] * rl, acc_o[4 * g + 1] * rl);
      o.y = pack_bf16x2(acc_o[4 * g + 2] * rl, acc_o[4 * g + 3] * rl);
      *reinterpret_cast<uint2*>(lds + r * (DV * 2) + (((4 * role + g) ^ ((r / (16 / PR)) % PR)) * 16 + 8 * h)) = o;
    }
  }
  lds_barrier();
  __bf16* o_first = out + b * a.o_sb + hq * a.o_sh + (int64_t)(w.q_first + q0) * a.o_ss;
#pragma unroll
  for (int i = 0; i < PR / 8; ++i) {
    const int p = 256 * i + tid, row = p / PR, c = p % PR;
    const v4i_t o = *reinterpret_cast<const v4i_t*>(lds + row * (DV * 2) + (c ^ ((row / (16 / PR)) % PR)) * 16);
    *reinterpret_cast<v4i_8_t*>(o_first + row * a.o_ss + 8 * c) = o;
  }
}

template <int NK, int ND, bool QBF, typename SEQS>
__global__ __launch_bounds__(256, NK > 2 ? 2 : 3) void attn_split_kernel(AttnArgs a, SEQS seqs) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[SplitLds<NK, ND>::BYTES];
  attn_split_body<NK, ND, QBF>(a, seqs, reinterpret_cast<__bf16*>(a.out), a.lse, lds);
}

template <int NK, int ND, typename SEQS>
int launch(const AttnArgs& a, const SEQS& seqs, int B, int row_blocks, hipStream_t st) {
  const dim3 grid((unsigned)a.Hq, (unsigned)B, (unsigned)row_blocks);
  if (a.qx) hipLaunchKernelGGL((attn_split_kernel<NK, ND, true, SEQS>), grid, dim3(256), 0, st, a, seqs);
  else hipLaunchKernelGGL((attn_split_kernel<NK, ND, false, SEQS>), grid, dim3(256), 0, st, a, seqs);
  return check_launch("attention_fwd");
}

}  // namespace

template <typename SEQS>
int launch_attn_split(const AttnArgs& a, const SEQS& seqs, int B, int row_blocks, int64_t D, int64_t Dv, hipStream_t st) {
  switch (D + (Dv == 128 ? 1 : 0)) {
    case 64: return launch<1, 2>(a, seqs, B, row_blocks, st);
    case 65: return launch<1, 4>(a, seqs, B, row_blocks, st);
    case 128: return launch<2, 2>(a, seqs, B, row_blocks, st);
    case 129: return launch<2, 4>(a, seqs, B, row_blocks, st);
    case 192: return launch<3, 2>(a, seqs, B, row_blocks, st);
    case 193: return launch<3, 4>(a, seqs, B, row_blocks, st);
    case 256: return launch<4, 2>(a, seqs, B, row_blocks, st);
    case 257: return launch<4, 4>(a, seqs, B, row_blocks, st);
  }
  return ALTO_MXFP4_EINVAL;
}
template int launch_attn_split<AttnSeqs>(const AttnArgs&, const AttnSeqs&, int, int, int64_t, int64_t, hipStream_t);
template int launch_attn_split<AttnNoSeqs>(const AttnArgs&, const AttnNoSeqs&, int, int, int64_t, int64_t, hipStream_t);

}  // namespace alto
