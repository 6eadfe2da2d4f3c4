// MXFP4 GEMM tiles of 128x128 and 64x64 for gfx950: the same data path as the 256x256 tile (gemm_tile.h) cut for problems
// that do not have enough 256x256 tiles to give every compute unit one.
//
// A workgroup of 4 waves (2 x 2) owns the tile; a wave owns TMW x TNW MFMA tiles of 32x32 (v_mfma_scale_f32_32x32x64).
//   global --buffer_load_dwordx4 ... lds--> LDS ring of NST stages of 256 K (whole 128-byte lines of TM + TN rows, pieces
//   XOR-swizzled by (row / 2) % 8 as in gemm_tile.h) --ds_read_b128--> MFMA operands, four K steps of 64 per stage.
// 128x128 with two stages takes 64 KB, 64x64 with three takes 48 KB, so two or three workgroups share a compute unit and
// one computes while another waits for its stage: no interleaving by hand as in the large tile.
// Scales do not pass through LDS: the eight bytes that a lane needs for a 512-K block are one 8-byte load (packed form: rows
// 16 bytes apart, 64 lanes read 512 bytes in a row) or one 16-byte load and four byte permutes (plain rows).
// Operand order, K order and rounding are those of the 256x256 tile: the results are the same bit for bit.
#pragma once
#include "gemm_tile.h"

namespace alto {

template <int TMW_, int TNW_, int NST_>
struct MidTile {
  static constexpr int WM = 2, WN = 2, TMW = TMW_, TNW = TNW_, NST = NST_;
  static constexpr int NWAVE = WM * WN, THREADS = 64 * NWAVE;
  static constexpr int TM = 32 * WM * TMW, TN = 32 * WN * TNW;
  static constexpr int STAGE = (TM + TN) * 128;
  static constexpr int LOADS = (TM + TN) / 8 / NWAVE, LOADS_A = TM / 8 / NWAVE;   // load instructions per wave and stage
  static constexpr int CH = TN / 8;                                                 // 16-byte chunks of a bf16 tile row
  static constexpr int LDS = NST * STAGE > TM * TN * 2 ? NST * STAGE : TM * TN * 2;
  static_assert(TM / 8 % NWAVE == 0 && TN / 8 % NWAVE == 0 && NWAVE % 2 == 0, "whole load instructions per operand");
};
using Mid128 = MidTile<2, 2, 2>;
using Mid64 = MidTile<1, 1, 3>;

// Scale bytes of one operand row for the lane's half h: dword ms, byte j = scale of group 16 kb + 8 ms + 2 j + h.
struct MidScales {
  const uint8_t* row;
  int64_t ss_k;
  template <bool PS>
  __device__ __forceinline__ void init(const OperandView& v, int64_t r, int h) {
    ss_k = v.ss_k;
    row = v.scales + (v.is_2d ? r >> 5 : r) * v.ss_r + (PS ? 8 * h : 0);   // (packed: ss_r = 16, ss_k = bytes per 512-K block)
  }
  template <bool PS>
  __device__ __forceinline__ void load(int kb, int G, int h, uint32_t (&raw)[4]) const {
    if constexpr (PS) {
      const uint2 v = *reinterpret_cast<const uint2*>(row + kb * ss_k);
      raw[0] = v.x;
      raw[1] = v.y;
    } else {
      if (G >= 16) {   // one 16-byte load (any alignment) that never leaves the row; pick shifts what a clamped start moved
        const int g0 = 16 * kb < G - 16 ? 16 * kb : G - 16;
        __builtin_memcpy(raw, row + g0, 16);
      } else {         // a row shorter than one load: byte by byte, 127 beyond K
        uint8_t b[16];
#pragma unroll
        for (int g = 0; g < 16; ++g) b[g] = row[g < G ? g : G - 1];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          raw[d] = 0;
#pragma unroll
          for (int j = 0; j < 4; ++j) raw[d] |= (uint32_t)(4 * d + j < G ? b[4 * d + j] : 127) << (8 * j);
        }
      }
    }
  }
  template <bool PS>
  __device__ __forceinline__ static void pick(int kb, int G, uint32_t (&raw)[4], int h, int (&s)[2]) {
    if constexpr (PS) {
      s[0] = (int)raw[0];
      s[1] = (int)raw[1];
    } else {
      const int sh = 16 * kb - (G - 16);   // > 0: the block reaches sh bytes past its row and was loaded from sh bytes before its start
      if (G >= 16 && sh > 0) {
        unsigned __int128 v = ((unsigned __int128)(((uint64_t)raw[3] << 32) | raw[2]) << 64) | (((uint64_t)raw[1] << 32) | raw[0]);
        const unsigned __int128 ones = ((unsigned __int128)0x7F7F7F7F7F7F7F7Full << 64) | 0x7F7F7F7F7F7F7F7Full;
        v = (v >> (8 * sh)) | (ones << (128 - 8 * sh));
        raw[0] = (uint32_t)v;
        raw[1] = (uint32_t)(v >> 32);
        raw[2] = (uint32_t)(v >> 64);
        raw[3] = (uint32_t)(v >> 96);
      }
      const uint32_t sel = 0x06040200u + (h ? 0x01010101u : 0u);
      s[0] = (int)__builtin_amdgcn_perm(raw[1], raw[0], sel);
      s[1] = (int)__builtin_amdgcn_perm(raw[3], raw[2], sel);
    }
  }
};

// One tile of C: rows [m0, m0 + TM) within [m_lo, m_hi), columns [n0, n0 + TN) below n_hi (N a multiple of 8, rows of C
// 16-byte aligned).  Every thread of the workgroup must call it.  TileArgs::s_k0, k_lead and ps_* are not used: whole reductions.
template <typename OutT, typename T, bool PS>
__device__ __forceinline__ void gemm_mid_tile(const TileArgs& ta, OutT* __restrict__ c, int64_t ldc, uint8_t* smem) {
  typedef __attribute__((address_space(3))) uint8_t lds_u8;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wm = wave / T::WN, wn = wave % T::WN, r = lane & 31, h = lane >> 5;
  const int G = ta.G, kbytes = G * 16;
  const int NS = (G + 7) / 8, KB = (G + 15) / 16;

  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(ta.A.codes), 0, (int)ta.a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(ta.B.codes), 0, (int)ta.b_bytes, 0x00020000);
  // load instruction i of a wave: chunk NWAVE i + wave = 8 rows x 128 bytes, A rows first; slot l % 8 of row l / 8 takes
  // piece (l % 8) ^ ((row / 2) % 8)
  const int gpiece = (lane & 7) ^ ((4 * (wave & 1) + (lane >> 4)) & 7);
  uint32_t off[T::LOADS];
#pragma unroll
  for (int i = 0; i < T::LOADS; ++i) {
    const bool is_a = i < T::LOADS_A;
    int row = 8 * (T::NWAVE * (is_a ? i : i - T::LOADS_A) + wave) + (lane >> 3) + (int)(is_a ? ta.m0 : ta.n0);
    const int last = (int)(is_a ? ta.m_hi : ta.n_hi) - 1, first = is_a ? (int)ta.m_lo : 0;
    row = row < last ? row : last;
    row = row > first ? row : first;
    off[i] = (uint32_t)row * (uint32_t)(is_a ? ta.A.ld : ta.B.ld) + gpiece * 16;
  }
  auto gload = [&](int s, int slot) {
    const int koff = __builtin_amdgcn_readfirstlane(s * 128);
    const uint32_t oob = koff + gpiece * 16 < kbytes ? 0u : 0x80000000u;   // beyond K: out of range, zeros land in LDS
#pragma unroll
    for (int i = 0; i < T::LOADS; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(i < T::LOADS_A ? rsrc_a : rsrc_b,
                                               (__attribute__((address_space(3))) void*)((lds_u8*)smem + slot * T::STAGE + (T::NWAVE * i + wave) * 1024), 16,
                                               (int)(off[i] | oob), koff, 0, 0);
  };

  MidScales sca[T::TMW], scb[T::TNW];
#pragma unroll
  for (int t = 0; t < T::TMW; ++t) {
    int64_t row = ta.m0 + 32 * (wm * T::TMW + t) + r;
    row = row < ta.m_hi ? row : ta.m_hi - 1;
    row = row < ta.m_lo ? ta.m_lo : row;
    sca[t].template init<PS>(ta.A, row, h);
  }
#pragma unroll
  for (int u = 0; u < T::TNW; ++u) {
    int64_t row = ta.n0 + 32 * (wn * T::TNW + u) + r;
    row = row < ta.n_hi ? row : ta.n_hi - 1;
    scb[u].template init<PS>(ta.B, row, h);
  }
  uint32_t ra[T::TMW][4], rb[T::TNW][4];   // scale bytes of the next block, as loaded
  auto sload = [&](int kb) {
#pragma unroll
    for (int t = 0; t < T::TMW; ++t) sca[t].template load<PS>(kb, G, h, ra[t]);
#pragma unroll
    for (int u = 0; u < T::TNW; ++u) scb[u].template load<PS>(kb, G, h, rb[u]);
  };

  v16f_t acc[T::TMW][T::TNW];
#pragma unroll
  for (int t = 0; t < T::TMW; ++t)
#pragma unroll
    for (int u = 0; u < T::TNW; ++u)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[t][u][v] = 0.0f;

  const uint32_t c0 = (uint32_t)(h ^ ((r >> 1) & 7)) << 4;
  const uint32_t a_off = (uint32_t)(32 * T::TMW * wm + r) * 128 + c0, b_off = (uint32_t)(T::TM + 32 * T::TNW * wn + r) * 128 + c0;
  int sa[T::TMW][2], sb[T::TNW][2];
  auto compute = [&](auto msc, int slot) {
    constexpr int MS = decltype(msc)::value;
    const uint8_t* base = smem + slot * T::STAGE;
    auto step = [&](auto jc) {
      constexpr int J = decltype(jc)::value;
      v8i_t fa[T::TMW], fb[T::TNW];
#pragma unroll
      for (int t = 0; t < T::TMW; ++t) {
        const uint4 v = *reinterpret_cast<const uint4*>(base + ((a_off ^ (J * 32)) + t * 4096));
        fa[t] = v8i_t{(int)v.x, (int)v.y, (int)v.z, (int)v.w, 0, 0, 0, 0};
      }
#pragma unroll
      for (int u = 0; u < T::TNW; ++u) {
        const uint4 v = *reinterpret_cast<const uint4*>(base + ((b_off ^ (J * 32)) + u * 4096));
        fb[u] = v8i_t{(int)v.x, (int)v.y, (int)v.z, (int)v.w, 0, 0, 0, 0};
      }
#pragma unroll
      for (int t = 0; t < T::TMW; ++t)
#pragma unroll
        for (int u = 0; u < T::TNW; ++u)
          acc[t][u] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb[u], fa[t], acc[t][u], 4, 4, J, sb[u][MS], J, sa[t][MS]);
    };
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
    step(std::integral_constant<int, 2>{});
    step(std::integral_constant<int, 3>{});
  };
  // stage s: its loads have landed for every wave (and every wave is done with stage s - 1, whose slot the loads of stage
  // s + NST - 1 may then overwrite)
  int slot = 0;
  auto arrive = [&](int s) {
    // (the loads of NST - 2 later stages stay in flight; younger scale loads only make the wait stricter)
    if constexpr (T::NST == 2) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((T::NST - 2) * T::LOADS) : "memory");
  };
  auto next_slot = [&](int k) { const int v = slot + k; return v >= T::NST ? v - T::NST : v; };

  sload(0);
#pragma unroll
  for (int s = 0; s < T::NST - 1; ++s) gload(s, s);   // (stages beyond K load zeros)
  for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
    for (int t = 0; t < T::TMW; ++t) MidScales::pick<PS>(kb, G, ra[t], h, sa[t]);
#pragma unroll
    for (int u = 0; u < T::TNW; ++u) MidScales::pick<PS>(kb, G, rb[u], h, sb[u]);
    arrive(2 * kb);
    if (kb + 1 < KB) sload(kb + 1);
    gload(2 * kb + T::NST - 1, next_slot(T::NST - 1));
    compute(std::integral_constant<int, 0>{}, slot);
    slot = next_slot(1);
    if (2 * kb + 1 < NS) {
      arrive(2 * kb + 1);
        gload(2 * kb + T::NST, next_slot(T::NST - 1));
      compute(std::integral_constant<int, 1>{}, slot);
      slot = next_slot(1);
    }
  }

  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // the loads beyond K have landed, nobody reads operands any more
  if constexpr (sizeof(OutT) == 2) {
    // bf16: the tile is assembled in LDS as rows of CH 16-byte chunks (chunk index XORed with the row) and stored row-wise
    constexpr int CH = T::CH;
#pragma unroll
    for (int t = 0; t < T::TMW; ++t)
#pragma unroll
      for (int u = 0; u < T::TNW; ++u)
#pragma unroll
        for (int vq = 0; vq < 4; ++vq) {
          const int row = 32 * (wm * T::TMW + t) + r, ch = 4 * (wn * T::TNW + u) + vq;
          uint2 o;
          o.x = pack_bf16x2(acc[t][u][4 * vq + 0] * ta.out_scale, acc[t][u][4 * vq + 1] * ta.out_scale);
          o.y = pack_bf16x2(acc[t][u][4 * vq + 2] * ta.out_scale, acc[t][u][4 * vq + 3] * ta.out_scale);
          *reinterpret_cast<uint2*>(smem + row * (CH * 16) + ((ch ^ (r & (CH - 1))) << 4) + 8 * h) = o;
        }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < T::TM * CH / T::THREADS; ++it) {
      const int idx = it * T::THREADS + tid, row = idx / CH, ch = idx % CH;
      const uint4 v = *reinterpret_cast<const uint4*>(smem + row * (CH * 16) + ((ch ^ (row & (CH - 1))) << 4));
      const int64_t m = ta.m0 + row, n = ta.n0 + 8 * ch;
      if (m >= ta.m_lo && m < ta.m_hi && n + 8 <= ta.n_hi) *reinterpret_cast<uint4*>(c + m * ldc + n) = v;
    }
  } else {
#pragma unroll
    for (int t = 0; t < T::TMW; ++t) {
      const int64_t m = ta.m0 + 32 * (wm * T::TMW + t) + r;
      const bool mok = m >= ta.m_lo && m < ta.m_hi;
#pragma unroll
      for (int u = 0; u < T::TNW; ++u)
#pragma unroll
        for (int vq = 0; vq < 4; ++vq) {
          const int64_t n = ta.n0 + 32 * (wn * T::TNW + u) + 8 * vq + 4 * h;
          if (mok && n + 4 <= ta.n_hi)
            *reinterpret_cast<float4*>(c + m * ldc + n) = make_float4(acc[t][u][4 * vq + 0] * ta.out_scale, acc[t][u][4 * vq + 1] * ta.out_scale,
                                                                        acc[t][u][4 * vq + 2] * ta.out_scale, acc[t][u][4 * vq + 3] * ta.out_scale);
        }
    }
  }
}

}  // namespace alto
