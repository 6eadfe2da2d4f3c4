// Operand quantizer of the attention forward (gfx950): K and V, and Q where the attention kernel does not quantize it itself
// (fp32 inputs), in one launch, straight from the caller's layout.
//
// Each operand is [B][heads][S][D] seen through element strides of the batch, head and row dims (unit stride along D), so
// the [B, S, heads, D] tensors of a model and tokens packed as [T, heads, D] are read where they lie.  Every 32 x 32 block
// gets one E8M0 scale and E2M1 codes (round to nearest even; the values of alto_mxfp4_quantize with is_2d):
//   Q, K  codes packed along D     [B][H][S][D/2],  scales [B][H][S/32][D/32]
//   V     codes packed along the keys [B][H][D][S/2], scales [B][H][S/32][D/32]
//
// What bounds it is HBM: one read of the operands and a quarter of that written (4 x 2048 tokens x (64 + 8 + 8) heads x 128 in
// bf16: 41 us for 210 MB, 5.1 TB/s, the rate of a plain copy).  A wave owns 32 rows x COLS columns, so a
// block's absmax is a reduction inside the wave (registers, quad DPP, lane shuffles: no LDS, no barrier for Q and K), and
// four waves take four consecutive row bands of one head, which gives V 64-byte pieces of its transposed rows to store.
// COLS = 128 whenever the head dims allow: a row piece is then a whole 256-byte segment of bf16 and a wave's code stores
// are contiguous.  The general quantizer this replaces here wants one batch stride, so [B, S, heads, D] inputs were copied
// first (three copies, 101 us, and 47 us for four more launches), and its 256-column tile leaves half of the lanes idle at
// D = 128.  That forward went from 315 to 217 us with it; since the attention kernel reads a bf16 Q itself, K and V alone take 9 of
// those 41 us.
#include "attention.h"

namespace alto {
namespace {

struct AttnOperand {
  const void* x;
  int64_t sb, sh, ss;       // element strides of batch, head, row
  uint8_t* codes;
  uint8_t* scales;
  int H, S, D;
  int groups;               // ceil(S / 128): groups of four bands
  int head_major;           // workgroup order: 1 walks the groups of a head first (heads far apart in memory), 0 the heads of a group
  int64_t wgs;              // workgroups of this operand
};
struct AttnQuantArgs {
  AttnOperand q, k, v;
};

// STREAM: non-temporal loads.
template <typename T, int COLS, bool STREAM>
__global__ __launch_bounds__(256) void attn_quant_kernel(const AttnQuantArgs a) {
  constexpr int DW = sizeof(T) == 2 ? 4 : 8;       // dwords of 8 elements
  constexpr int LPR = COLS / 8;                    // lanes per row
  constexpr int RPI = 64 / LPR, NI = 32 / RPI;     // rows per load instruction, instructions per band
  constexpr int PITCH = 32 * COLS + 32;            // bytes of one band's codes in LDS (V), one per byte; the pad spreads the banks
  __shared__ __align__(16) uint8_t vcodes[4 * PITCH];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int64_t wg = blockIdx.x;
  int which = 0;
  if (wg >= a.q.wgs) { wg -= a.q.wgs; which = 1; if (wg >= a.k.wgs) { wg -= a.k.wgs; which = 2; } }
  const AttnOperand& p = which == 0 ? a.q : (which == 1 ? a.k : a.v);
  const int chunks = p.D / COLS;
  const int chunk = (int)(wg % chunks);
  wg /= chunks;
  int group, head;
  int64_t b;
  if (p.head_major) {
    group = (int)(wg % p.groups); wg /= p.groups;
    head = (int)(wg % p.H); b = wg / p.H;
  } else {
    head = (int)(wg % p.H); wg /= p.H;
    group = (int)(wg % p.groups); b = wg / p.groups;
  }
  const int band = group * 4 + wave;               // S % 32 == 0: a band is all inside or all outside
  const bool live = band * 32 < p.S;
  const int col = chunk * COLS + (lane % LPR) * 8, row0 = band * 32 + lane / LPR;
  const int64_t bh = b * p.H + head;
  uint32_t w[NI][DW];
  if (live) {
    const T* x = reinterpret_cast<const T*>(p.x) + b * p.sb + head * p.sh + col;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const v4i_t* src = reinterpret_cast<const v4i_t*>(x + (int64_t)(row0 + i * RPI) * p.ss);
#pragma unroll
      for (int e = 0; e < DW / 4; ++e) {
        const v4i_t v = STREAM ? __builtin_nontemporal_load(src + e) : src[e];
        w[i][4 * e + 0] = v[0]; w[i][4 * e + 1] = v[1]; w[i][4 * e + 2] = v[2]; w[i][4 * e + 3] = v[3];
      }
    }
    // the block's 32 rows x 32 columns sit in the lanes that agree in (lane % LPR) / 4
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < NI; ++i) m = max(m, absmax8<T>(w[i]));
    m = max(m, dpp_u32<ALTO_DPP_QUAD_XOR1>(m));
    m = max(m, dpp_u32<ALTO_DPP_QUAD_XOR2>(m));
#pragma unroll
    for (int d = LPR; d < 64; d <<= 1) m = max(m, (uint32_t)__shfl_xor((int)m, d, 64));
    const uint32_t s = sizeof(T) == 2 ? e8m0_from_bf16_bits(m) : e8m0_from_f32_bits(m);
    const float scale = u2f(s << 23);
    if (lane < LPR && (lane & 3) == 0) p.scales[(bh * (p.S / 32) + band) * (p.D / 32) + (col >> 5)] = (uint8_t)s;
    if (which < 2) {
      uint8_t* dst = p.codes + (bh * p.S + row0) * (p.D / 2) + (col >> 1);
#pragma unroll
      for (int i = 0; i < NI; ++i) *reinterpret_cast<uint32_t*>(dst + (int64_t)i * RPI * (p.D / 2)) = encode8<T>(w[i], scale);
    } else {
#pragma unroll
      for (int i = 0; i < NI; ++i) {   // one code per byte, in column order
        const uint32_t o = encode8<T>(w[i], scale), ev = o & 0x0F0F0F0Fu, od = (o >> 4) & 0x0F0F0F0Fu;
        uint2 two;
        two.x = __builtin_amdgcn_perm(od, ev, 0x05010400u);
        two.y = __builtin_amdgcn_perm(od, ev, 0x07030602u);
        *reinterpret_cast<uint2*>(&vcodes[wave * PITCH + (lane / LPR + i * RPI) * COLS + (lane % LPR) * 8]) = two;
      }
    }
  }
  if (which < 2) return;   // (whole workgroup)
  __syncthreads();
  // V: 16-byte piece (32 keys) of column c and band g; four lanes store the four bands' pieces of one column, 64 bytes
#pragma unroll
  for (int c0 = 0; c0 < COLS; c0 += 64) {
    const int c = c0 + (tid >> 2), g = tid & 3;
    if ((group * 4 + g) * 32 < p.S) {
      const uint8_t* src = &vcodes[g * PITCH + c];
      uint32_t out[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t o = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) o |= (uint32_t)src[(8 * j + e) * COLS] << (4 * e);
        out[j] = o;
      }
      *reinterpret_cast<uint4*>(p.codes + (bh * p.D + chunk * COLS + c) * (int64_t)(p.S / 2) + (group * 4 + g) * 16) = make_uint4(out[0], out[1], out[2], out[3]);
    }
  }
}

}  // namespace
}  // namespace alto

namespace alto {
// q == NULL: K and V only
static int quantize_operands(const void* q, const void* k, const void* v, int dtype, int64_t B, int64_t Hq, int64_t Hk, int64_t Sq, int64_t Sk, int64_t D,
                             int64_t Dv, int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t k_sb, int64_t k_sh, int64_t k_ss, int64_t v_sb, int64_t v_sh,
                             int64_t v_ss, uint8_t* q_codes, uint8_t* q_scales, uint8_t* k_codes, uint8_t* k_scales, uint8_t* vt_codes, uint8_t* v_scales,
                             hipStream_t st) {
  ALTO_REQUIRE(dtype == ALTO_DT_BF16 || dtype == ALTO_DT_F32, "attention_quantize: dtype %d is neither bf16 (0) nor f32 (1)", dtype);
  ALTO_REQUIRE(B > 0 && Hq > 0 && Hk > 0, "attention_quantize: empty batch or no heads");
  ALTO_REQUIRE(Sq > 0 && Sq % 32 == 0 && Sk > 0 && Sk % 32 == 0, "attention_quantize: Sq=%lld and Sk=%lld must be positive multiples of 32", (long long)Sq, (long long)Sk);
  ALTO_REQUIRE(D > 0 && D % 64 == 0 && D <= 4096 && Dv > 0 && Dv % 64 == 0 && Dv <= 4096, "attention_quantize: head dim D=%lld, value dim Dv=%lld must be multiples of 64", (long long)D, (long long)Dv);
  ALTO_REQUIRE(Sq < (1ll << 31) && Sk < (1ll << 31) && Hq < (1ll << 31) && Hk < (1ll << 31) && B < (1ll << 31) && product_below(1ll << 40, B, Hq, Sq) &&
                   product_below(1ll << 40, B, Hk, Sk) && product_below(1ll << 44, B * Hq, Sq, D) && product_below(1ll << 44, B * Hk, Sk, D > Dv ? D : Dv),
               "attention_quantize: tensor too large");
  const int64_t vec = dtype == ALTO_DT_BF16 ? 8 : 4;
  for (int64_t st : {q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss})
    ALTO_REQUIRE(st >= 0 && st < (1ll << 44) && st % vec == 0, "attention_quantize: strides must be non-negative multiples of %lld elements", (long long)vec);
  ALTO_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)vt_codes) & 15) == 0 && (((uintptr_t)q_codes | (uintptr_t)k_codes) & 3) == 0,
               "attention_quantize: inputs and vt_codes must be 16-byte aligned, q_codes and k_codes 4-byte aligned");
  const int cols = (D % 128 == 0 && Dv % 128 == 0) ? 128 : 64;
  AttnQuantArgs a{};
  auto fill = [&](AttnOperand& o, const void* x, int64_t sb, int64_t sh, int64_t ss, uint8_t* codes, uint8_t* scales, int64_t H, int64_t S, int64_t d) {
    const int64_t groups = (S + 127) / 128;
    o = AttnOperand{x, sb, sh, ss, codes, scales, (int)H, (int)S, (int)d, (int)groups, sh > ss ? 1 : 0, 0};
    return product_below(1ll << 31, B * H, groups, d / cols) ? (o.wgs = B * H * groups * (d / cols)) : -1;
  };
  const int64_t nq = q ? fill(a.q, q, q_sb, q_sh, q_ss, q_codes, q_scales, Hq, Sq, D) : (a.q.wgs = 0), nk = fill(a.k, k, k_sb, k_sh, k_ss, k_codes, k_scales, Hk, Sk, D),
                nv = fill(a.v, v, v_sb, v_sh, v_ss, vt_codes, v_scales, Hk, Sk, Dv);
  ALTO_REQUIRE(nq >= 0 && nk > 0 && nv > 0 && nq + nk + nv < (1ll << 31), "attention_quantize: too many workgroups");
  const dim3 grid((unsigned)(nq + nk + nv));
  // bf16 operands of 128 MB and more are read past the caches, which then keep the codes for the attention kernel (whole calls,
  // causal, changing inputs, without -> with, us: 160 MB 222 -> 216, 320 MB 443 -> 430).  Smaller ones may be in a cache already
  // (96 MB the same).  fp32 operands lose: two load instructions use half of each line, and the second finds it in no cache
  // (this kernel at 192 MB 45 -> 51, at 640 MB 141 -> 157; whole calls 131 -> 137 and 490 -> 502).
  const bool stream_in = dtype == ALTO_DT_BF16 && ((q ? B * Hq * Sq * D : 0) + B * Hk * Sk * (D + Dv)) * 2 >= (128ll << 20);
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, a); };
  if (dtype == ALTO_DT_BF16) {
    if (cols == 128) stream_in ? go(attn_quant_kernel<__bf16, 128, true>) : go(attn_quant_kernel<__bf16, 128, false>);
    else stream_in ? go(attn_quant_kernel<__bf16, 64, true>) : go(attn_quant_kernel<__bf16, 64, false>);
  } else {
    cols == 128 ? go(attn_quant_kernel<float, 128, false>) : go(attn_quant_kernel<float, 64, false>);
  }
  return check_launch("attention_quantize");
}
}  // namespace alto

extern "C" int alto_mxfp4_attention_quantize(const void* q, const void* k, const void* v, int dtype, int64_t B, int64_t Hq, int64_t Hk, int64_t Sq,
                                             int64_t Sk, int64_t D, int64_t Dv, int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t k_sb, int64_t k_sh,
                                             int64_t k_ss, int64_t v_sb, int64_t v_sh, int64_t v_ss, uint8_t* q_codes, uint8_t* q_scales,
                                             uint8_t* k_codes, uint8_t* k_scales, uint8_t* vt_codes, uint8_t* v_scales, void* stream) {
  ALTO_REQUIRE(q && k && v && q_codes && q_scales && k_codes && k_scales && vt_codes && v_scales, "attention_quantize: null pointer");
  return alto::quantize_operands(q, k, v, dtype, B, Hq, Hk, Sq, Sk, D, Dv, q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, q_codes, q_scales, k_codes, k_scales,
                                 vt_codes, v_scales, (hipStream_t)stream);
}

extern "C" int alto_mxfp4_attention_quantize_kv(const void* k, const void* v, int dtype, int64_t B, int64_t Hk, int64_t Sk, int64_t D, int64_t Dv,
                                                int64_t k_sb, int64_t k_sh, int64_t k_ss, int64_t v_sb, int64_t v_sh, int64_t v_ss, uint8_t* k_codes,
                                                uint8_t* k_scales, uint8_t* vt_codes, uint8_t* v_scales, void* stream) {
  ALTO_REQUIRE(k && v && k_codes && k_scales && vt_codes && v_scales, "attention_quantize: null pointer");
  return alto::quantize_operands(nullptr, k, v, dtype, B, Hk, Hk, Sk, Sk, D, Dv, 0, 0, 0, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, nullptr, nullptr, k_codes, k_scales, vt_codes,
                                 v_scales, (hipStream_t)stream);
}
