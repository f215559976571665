// Decode of the legacy, IQ and fp4 codecs into matrix-core operands, shared by the kernels of kq_codes.hip and
// kq_mid.hip.  A weight of these codecs is (block scale) x (small code); the code, exact in f16, is the B operand of
// v_mfma_f32_32x32x16_f16, and the block scale multiplies the f32 sum of its 16 or 32 weights afterwards.
#pragma once

#include "kq_mma.h"

namespace kqcodes {

using namespace kqmma;

typedef u32x4 u32x4_a1 __attribute__((aligned(1)));  // the hardware serves unaligned vector loads
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int CK_STEP = 256;  // weights of K per step

// ------------------------------------------------------------------ codec traits
template <int C>
struct CodeGeom {
  static constexpr int WPB = kq_geom(C).wpb, BPB = kq_geom(C).bpb;
  static constexpr int BLOCKS = CK_STEP / WPB;      // blocks per step and row
  static constexpr int BYTES = BLOCKS * BPB;        // wire bytes per step and row
  static constexpr int PIECES = (BYTES + 15) / 16;  // 16-byte pieces (the last may read past the step)
  static constexpr int LROW = (PIECES | 1) * 16;    // LDS row stride: an odd number of pieces
  // scale granularity: one MFMA (16 weights) or two (32 weights) per scale
  static constexpr int SB = (C == KQ_NVFP4 || C == KQ_IQ2_XS || C == KQ_IQ2_S || C == KQ_IQ1_M) ? 16 : 32;
  static constexpr bool HAS_MIN = C == KQ_Q4_1 || C == KQ_Q5_1;
  // f16 codebook in LDS: entries of 8 weights (16 bytes) or 4 weights (8 bytes)
  static constexpr int GRID_N = C == KQ_IQ2_XXS ? 256 : C == KQ_IQ2_XS ? 512 : C == KQ_IQ2_S ? 1024
                               : (C == KQ_IQ1_S || C == KQ_IQ1_M) ? 2048 : C == KQ_IQ3_XXS ? 256 : C == KQ_IQ3_S ? 512 : 0;
  static constexpr int GRID_W = (C == KQ_IQ3_XXS || C == KQ_IQ3_S) ? 4 : 8;
  static constexpr int GRID_OFF = C == KQ_IQ2_XXS ? KQ_GRID_IQ2XXS : C == KQ_IQ2_XS ? KQ_GRID_IQ2XS
                                 : C == KQ_IQ2_S ? KQ_GRID_IQ2S : (C == KQ_IQ1_S || C == KQ_IQ1_M) ? KQ_GRID_IQ1S
                                 : C == KQ_IQ3_XXS ? KQ_GRID_IQ3XXS : KQ_GRID_IQ3S;
  static constexpr bool GRID_SIGNED = C == KQ_IQ1_S || C == KQ_IQ1_M;  // int8 entries
  // 32-weight blocks whose byte j holds weights j and j + 16 as indices of a 16-value table (iq4_nl, iq4_xs, mxfp4): the
  // table in LDS maps a byte to the f16 pair of its two values, and the activations of a block are staged as
  // x[j], x[j + 16] interleaved, so four table reads are the B operand of an MFMA with no further arithmetic
  static constexpr bool PAIR_LUT = C == KQ_IQ4_NL || C == KQ_IQ4_XS || C == KQ_MXFP4;
  // pair table: 256 entries of 4 bytes.  The grouped kernel keeps one copy per LDS bank (entry b copy c at
  // 128 b + 4 c, lane l reads copy l % 32: the 64 data-dependent reads of an instruction never meet in a bank),
  // + 1 KiB for the plain table the copies are made from; the per-entry kernel, whose launches are too short to
  // earn the 32 KiB build back, keeps the plain table.
  static constexpr int GRID_BYTES = PAIR_LUT ? 1024 : GRID_N * GRID_W * 2;
  static constexpr int GROUPED_GRID_BYTES = PAIR_LUT ? 32768 + 1024 : GRID_BYTES;
  // 256-entry table spreading 8 bits over the 8 halves of a B operand: sign bits (bit 15) for the
  // signed codebooks, the fifth code bit (bit 4) for q5_0 / q5_1
  static constexpr bool SIGNS = C == KQ_IQ2_XXS || C == KQ_IQ2_XS || C == KQ_IQ2_S || C == KQ_IQ3_XXS || C == KQ_IQ3_S;
  static constexpr bool FIFTH = C == KQ_Q5_0 || C == KQ_Q5_1;
  static constexpr int SPREAD_BYTES = (SIGNS || FIFTH) ? 4096 : 0;
  static constexpr int SPREAD_BIT = SIGNS ? 15 : 4;
};

// ------------------------------------------------------------------ small helpers
__device__ __forceinline__ uint32_t pk_sub(uint32_t v, float bias) {
  const f16x2 b = {(_Float16)bias, (_Float16)bias};
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, v) - b);
}
// bytes (c0 c1 c2 c3) of `b`, each below 256 -> f16 pairs (c0, c2) and (c1, c3), less `bias`:
// 0x6400 | c is the f16 1024 + c (one byte permute makes a pair), and the subtraction is exact
__device__ __forceinline__ void bytes_to_f16(uint32_t b, float bias, uint32_t& e, uint32_t& o) {
  const uint32_t k = opaque_vgpr(0x64646464u);
  e = pk_sub(__builtin_amdgcn_perm(k, b, 0x04020400u), 1024.f + bias);
  o = pk_sub(__builtin_amdgcn_perm(k, b, 0x04030401u), 1024.f + bias);
}
// two dwords of 8 bytes -> B operand in the fragment order k0 k2 k1 k3 k4 k6 k5 k7
__device__ __forceinline__ f16x8 bytes8_to_frag(uint32_t lo, uint32_t hi, float bias) {
  u32x4 r;
  uint32_t e, o;
  bytes_to_f16(lo, bias, e, o);
  r[0] = e;
  r[1] = o;
  bytes_to_f16(hi, bias, e, o);
  r[2] = e;
  r[3] = o;
  return __builtin_bit_cast(f16x8, r);
}
// 16-entry byte table lookup on the four nibble-valued bytes of n: two 8-entry byte permutes and a
// per-byte select on bit 3 (the select mask is a third permute)
__device__ __forceinline__ uint32_t lut16(uint32_t n, uint32_t t0, uint32_t t1, uint32_t t2, uint32_t t3) {
  const uint32_t sel = n & 0x07070707u;
  const uint32_t lo = __builtin_amdgcn_perm(t1, t0, sel);
  const uint32_t hi = __builtin_amdgcn_perm(t3, t2, sel);
  // selector bytes 0x0c / 0x0d read as 0x00 / 0xff: 0xff in every byte whose bit 3 is set
  const uint32_t mask = __builtin_amdgcn_perm(n, n, ((n >> 3) & 0x01010101u) | 0x0c0c0c0cu);
  return (hi & mask) | (lo & ~mask);
}
// One lane's eight consecutive activations h[0..7] (8-group `pc` of a row) to the row's staging area: in the fragment
// order k0 k2 k1 k3 inside the group, or (PAIR) with x[j], x[j + 16] interleaved over each 32: lanes pc and pc ^ 2 of a
// quad hold x[8 a ..] and x[16 + 8 a ..] and write one half each of the 16 interleaved values.
template <bool PAIR>
__device__ __forceinline__ void stage_group(uint8_t* row_lds, int pc, const _Float16* h) {
  if constexpr (!PAIR) {
    const f16x8 v8 = {h[0], h[2], h[1], h[3], h[4], h[6], h[5], h[7]};
    *reinterpret_cast<f16x8*>(row_lds + 16 * pc) = v8;
  } else {
    uint32_t own[4], par[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      own[e] = (uint32_t)__builtin_bit_cast(uint16_t, h[2 * e]) | ((uint32_t)__builtin_bit_cast(uint16_t, h[2 * e + 1]) << 16);
      par[e] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)own[e], 0x4E, 0xf, 0xf, true);  // quad_perm [2,3,0,1]
    }
    const bool high = (pc & 2) != 0;
    const uint32_t a0 = high ? par[2] : own[0], a1 = high ? par[3] : own[1];
    const uint32_t b0 = high ? own[2] : par[0], b1 = high ? own[3] : par[1];
    const u32x4 o = {(a0 & 0xffffu) | (b0 << 16), (a0 >> 16) | (b0 & 0xffff0000u), (a1 & 0xffffu) | (b1 << 16),
                     (a1 >> 16) | (b1 & 0xffff0000u)};
    *reinterpret_cast<u32x4*>(row_lds + 64 * (pc >> 2) + 32 * (pc & 1) + (high ? 16 : 0)) = o;
  }
}
__device__ __forceinline__ float f16bits(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }

// 128-bit value >> 8 k bits (k >= 1 bytes)
__device__ __forceinline__ u32x4 shr_bytes(u32x4 v, uint32_t k) {
  if (k >= 16) return u32x4{0, 0, 0, 0};
  uint64_t lo = (uint64_t)v[0] | ((uint64_t)v[1] << 32), hi = (uint64_t)v[2] | ((uint64_t)v[3] << 32);
  if (k & 8) {
    lo = hi;
    hi = 0;
  }
  const uint32_t sh = 8 * (k & 7);
  if (sh) {
    lo = (lo >> sh) | (hi << (64 - sh));
    hi >>= sh;
  }
  return u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

// The wire bytes of one (row, step) in registers: the lane fetches them from LDS with 16-byte reads
// (row stride an odd number of 16-byte pieces: conflict-free) and every field is then picked at a
// compile-time byte offset, so that the decode issues no narrow, bank-conflicting LDS reads.
template <int NDW>
struct RowRegs {
  uint32_t d[NDW];
  template <int OFF>
  __device__ __forceinline__ uint32_t u32() const {
    static_assert(OFF >= 0 && OFF / 4 < NDW, "offset outside the row");
    if constexpr (OFF % 4 == 0)
      return d[OFF / 4];
    else
      return __builtin_amdgcn_alignbyte(d[OFF / 4 + 1 < NDW ? OFF / 4 + 1 : OFF / 4], d[OFF / 4], OFF % 4);
  }
  template <int OFF>
  __device__ __forceinline__ uint32_t u16() const {
    if constexpr (OFF % 4 <= 2)
      return (d[OFF / 4] >> (8 * (OFF % 4))) & 0xffffu;
    else
      return u32<OFF>() & 0xffffu;
  }
  template <int OFF>
  __device__ __forceinline__ uint32_t u8() const {
    return (d[OFF / 4] >> (8 * (OFF % 4))) & 0xffu;
  }
};
__device__ __forceinline__ uint32_t pick(int kg, uint32_t a, uint32_t b) { return kg ? b : a; }

struct Tables {
  const uint8_t* grid;    // f16 codebook (LDS)
  const uint8_t* spread;  // 256 x 16-byte bit-spread table (LDS)
  int pair_shift;         // log2 of the byte distance between pair-table entries (2, or 7 with a copy per bank)
};

// The B operand of MFMA J (weights 16 J + 8 kg .. + 7 of the step) of the row whose step bytes are in
// `row`.  J is a compile-time constant.
template <int C, int J, class R>
__device__ __forceinline__ f16x8 codes(const R& row, int kg, const Tables& t) {
  using G = CodeGeom<C>;
  if constexpr (C == KQ_Q8_0) {
    constexpr int off = (J / 2) * 34 + 2 + 16 * (J & 1);
    const uint32_t lo = pick(kg, row.template u32<off>(), row.template u32<off + 8>());
    const uint32_t hi = pick(kg, row.template u32<off + 4>(), row.template u32<off + 12>());
    return bytes8_to_frag(lo ^ 0x80808080u, hi ^ 0x80808080u, 128.f);
  } else if constexpr (C == KQ_Q4_0 || C == KQ_Q4_1 || C == KQ_Q5_0 || C == KQ_Q5_1 || C == KQ_IQ4_NL ||
                       C == KQ_IQ4_XS || C == KQ_MXFP4) {
    // 32 weights: 0..15 = low nibbles of q[0..15], 16..31 = high nibbles
    constexpr int QOFF = C == KQ_Q4_0 || C == KQ_IQ4_NL ? 2 : C == KQ_Q4_1 ? 4 : C == KQ_Q5_0 ? 6 : C == KQ_Q5_1 ? 8 : 1;
    constexpr int boff = (J / 2) * G::BPB, off = C == KQ_IQ4_XS ? 8 + 16 * (J / 2) : boff + QOFF;
    if constexpr (G::PAIR_LUT) {
      // staged positions 16 J + 8 kg .. + 7 = bytes 8 (J % 2) + 4 kg .. + 3 of block J / 2, both nibbles of each
      const uint32_t w = pick(kg, row.template u32<off + 8 * (J & 1)>(), row.template u32<off + 8 * (J & 1) + 4>());
      u32x4 r;
#pragma unroll
      for (int e = 0; e < 4; e++)
        r[e] = *reinterpret_cast<const uint32_t*>(t.grid + (((w >> (8 * e)) & 0xffu) << t.pair_shift));
      return __builtin_bit_cast(f16x8, r);
    }
    uint32_t lo = pick(kg, row.template u32<off>(), row.template u32<off + 8>());
    uint32_t hi = pick(kg, row.template u32<off + 4>(), row.template u32<off + 12>());
    if constexpr (J & 1) {
      lo >>= 4;
      hi >>= 4;
    }
    lo &= 0x0f0f0f0fu;
    hi &= 0x0f0f0f0fu;
    if constexpr (C == KQ_Q5_0 || C == KQ_Q5_1) {
      // fifth bits of weights 16 (J & 1) + 8 kg .. + 7: one byte of qh, spread to bit 4 of every half
      constexpr int hoff = boff + (C == KQ_Q5_0 ? 2 : 4) + 2 * (J & 1);
      const uint32_t hb = pick(kg, row.template u8<hoff>(), row.template u8<hoff + 1>());
      const u32x4 sp = *reinterpret_cast<const u32x4*>(t.spread + 16 * hb);
      u32x4 r = __builtin_bit_cast(u32x4, bytes8_to_frag(lo, hi, -1024.f));  // keep the 1024 + q form
      r |= sp;
      const float bias = C == KQ_Q5_0 ? 1024.f + 16.f : 1024.f;
      r[0] = pk_sub(r[0], bias);
      r[1] = pk_sub(r[1], bias);
      r[2] = pk_sub(r[2], bias);
      r[3] = pk_sub(r[3], bias);
      return __builtin_bit_cast(f16x8, r);
    } else {
      return bytes8_to_frag(lo, hi, C == KQ_Q4_0 ? 8.f : 0.f);
    }
  } else if constexpr (C == KQ_NVFP4) {
    // 64-weight blocks, 16-weight groups: weights 0..7 = low nibbles of q[0..7], 8..15 = high nibbles
    constexpr int off = (J / 4) * 36 + 4 + 8 * (J & 3);
    const int sh = 4 * kg;
    const uint32_t lo = (row.template u32<off>() >> sh) & 0x0f0f0f0fu;
    const uint32_t hi = (row.template u32<off + 4>() >> sh) & 0x0f0f0f0fu;
    return bytes8_to_frag(lut16(lo, 0x83828180u, 0x8c888684u, 0x7d7e7f80u, 0x74787a7cu),
                          lut16(hi, 0x83828180u, 0x8c888684u, 0x7d7e7f80u, 0x74787a7cu), 128.f);
  } else {
    // codebook codecs: 8-weight group l = 2 (J & 1) + kg of 32-weight sub-block ib = J / 2
    constexpr int ib = J / 2, l0 = 2 * (J & 1);
    const int l = l0 + kg;
    u32x4 r;
    uint32_t sbits = 0;
    if constexpr (C == KQ_IQ2_XXS) {
      const uint32_t aux = row.template u32<2 + 8 * ib + 4>();
      const uint32_t gi = pick(kg, row.template u8<2 + 8 * ib + l0>(), row.template u8<2 + 8 * ib + l0 + 1>());
      r = *reinterpret_cast<const u32x4*>(t.grid + 16 * gi);
      sbits = (aux >> (7 * l)) & 127u;
      sbits |= (uint32_t)(__builtin_popcount(sbits) & 1) << 7;
    } else if constexpr (C == KQ_IQ2_XS) {
      const uint32_t q = pick(kg, row.template u16<2 + 8 * ib + 2 * l0>(), row.template u16<2 + 8 * ib + 2 * l0 + 2>());
      r = *reinterpret_cast<const u32x4*>(t.grid + 16 * (q & 511u));
      sbits = q >> 9;
      sbits |= (uint32_t)(__builtin_popcount(sbits) & 1) << 7;
    } else if constexpr (C == KQ_IQ2_S) {
      const uint32_t qb = pick(kg, row.template u8<2 + 4 * ib + l0>(), row.template u8<2 + 4 * ib + l0 + 1>());
      const uint32_t gi = qb | ((row.template u8<66 + ib>() << (8 - 2 * l)) & 0x300u);
      r = *reinterpret_cast<const u32x4*>(t.grid + 16 * gi);
      sbits = pick(kg, row.template u8<34 + 4 * ib + l0>(), row.template u8<34 + 4 * ib + l0 + 1>());
    } else if constexpr (C == KQ_IQ3_XXS) {
      const uint32_t aux = row.template u32<66 + 4 * ib>();
      const uint32_t qq = pick(kg, row.template u16<2 + 8 * ib + 2 * l0>(), row.template u16<2 + 8 * ib + 2 * l0 + 2>());
      const u32x2 g1 = *reinterpret_cast<const u32x2*>(t.grid + 8 * (qq & 0xffu));
      const u32x2 g2 = *reinterpret_cast<const u32x2*>(t.grid + 8 * (qq >> 8));
      r = u32x4{g1[0], g1[1], g2[0], g2[1]};
      sbits = (aux >> (7 * l)) & 127u;
      sbits |= (uint32_t)(__builtin_popcount(sbits) & 1) << 7;
    } else if constexpr (C == KQ_IQ3_S) {
      const uint32_t h = row.template u8<66 + ib>();
      const uint32_t qq = pick(kg, row.template u16<2 + 8 * ib + 2 * l0>(), row.template u16<2 + 8 * ib + 2 * l0 + 2>());
      const uint32_t i1 = (qq & 0xffu) | ((h << (8 - 2 * l)) & 256u);
      const uint32_t i2 = (qq >> 8) | ((h << (7 - 2 * l)) & 256u);
      const u32x2 g1 = *reinterpret_cast<const u32x2*>(t.grid + 8 * i1);
      const u32x2 g2 = *reinterpret_cast<const u32x2*>(t.grid + 8 * i2);
      r = u32x4{g1[0], g1[1], g2[0], g2[1]};
      sbits = pick(kg, row.template u8<74 + 4 * ib + l0>(), row.template u8<74 + 4 * ib + l0 + 1>());
    } else if constexpr (C == KQ_IQ1_S) {
      const uint32_t qh = row.template u16<34 + 2 * ib>();
      const uint32_t qb = pick(kg, row.template u8<2 + 4 * ib + l0>(), row.template u8<2 + 4 * ib + l0 + 1>());
      r = *reinterpret_cast<const u32x4*>(t.grid + 16 * (qb | (((qh >> (3 * l)) & 7u) << 8)));
      const float delta = (qh & 0x8000u) ? 0.125f : -0.125f;  // subtracted below
      r[0] = pk_sub(r[0], delta);
      r[1] = pk_sub(r[1], delta);
      r[2] = pk_sub(r[2], delta);
      r[3] = pk_sub(r[3], delta);
    } else {  // KQ_IQ1_M
      const uint32_t hb = row.template u8<32 + 2 * ib + (J & 1)>();
      const uint32_t nib = kg ? (hb >> 4) : (hb & 15u);
      const uint32_t qb = pick(kg, row.template u8<4 * ib + l0>(), row.template u8<4 * ib + l0 + 1>());
      r = *reinterpret_cast<const u32x4*>(t.grid + 16 * (qb | ((nib & 7u) << 8)));
      const float delta = (nib & 8u) ? 0.125f : -0.125f;  // subtracted below
      r[0] = pk_sub(r[0], delta);
      r[1] = pk_sub(r[1], delta);
      r[2] = pk_sub(r[2], delta);
      r[3] = pk_sub(r[3], delta);
    }
    if constexpr (G::SIGNS) {
      const u32x4 sp = *reinterpret_cast<const u32x4*>(t.spread + 16 * sbits);
      r ^= sp;
    }
    return __builtin_bit_cast(f16x8, r);
  }
}

// f32 scale of scale block SBI of the step (SBI counts G::SB-weight blocks); mn = block minimum (q4_1 / q5_1)
template <int C, int SBI, class R>
__device__ __forceinline__ float block_scale(const R& row, float& mn) {
  constexpr int BPB = CodeGeom<C>::BPB;
  mn = 0.f;
  if constexpr (C == KQ_Q8_0 || C == KQ_Q4_0 || C == KQ_Q5_0 || C == KQ_IQ4_NL) {
    return f16bits(row.template u16<SBI * BPB>());
  } else if constexpr (C == KQ_Q4_1 || C == KQ_Q5_1) {
    const uint32_t dm = row.template u32<SBI * BPB>();
    mn = f16bits(dm >> 16);
    return f16bits(dm & 0xffffu);
  } else if constexpr (C == KQ_MXFP4) {
    return kq::e8m0_half(row.template u8<SBI * 17>());
  } else if constexpr (C == KQ_NVFP4) {
    return kq::ue4m3_half(row.template u8<(SBI / 4) * 36 + (SBI & 3)>());
  } else if constexpr (C == KQ_IQ4_XS) {
    const float d = f16bits(row.template u16<0>());
    const uint32_t sh = row.template u16<2>();
    const int ls = (int)((row.template u8<4 + (SBI >> 1)>() >> (4 * (SBI & 1))) & 15u) | (int)(((sh >> (2 * SBI)) & 3u) << 4);
    return d * (float)(ls - 32);
  } else if constexpr (C == KQ_IQ2_XXS) {
    const float d = f16bits(row.template u16<0>());
    const uint32_t aux = row.template u32<2 + 8 * SBI + 4>();
    return d * (0.5f + (float)(aux >> 28)) * 0.25f;
  } else if constexpr (C == KQ_IQ2_XS || C == KQ_IQ2_S) {  // 16-weight blocks
    const float d = f16bits(row.template u16<0>());
    const uint32_t scb = row.template u8<(C == KQ_IQ2_XS ? 66 : 74) + (SBI >> 1)>();
    return d * (0.5f + (float)((SBI & 1) ? (scb >> 4) : (scb & 15u))) * 0.25f;
  } else if constexpr (C == KQ_IQ3_XXS) {
    const float d = f16bits(row.template u16<0>());
    const uint32_t aux = row.template u32<66 + 4 * SBI>();
    return d * (0.5f + (float)(aux >> 28)) * 0.5f;
  } else if constexpr (C == KQ_IQ3_S) {
    const float d = f16bits(row.template u16<0>());
    const uint32_t sb = row.template u8<106 + (SBI >> 1)>();
    return d * (float)(1 + 2 * (int)((SBI & 1) ? (sb >> 4) : (sb & 15u)));
  } else if constexpr (C == KQ_IQ1_S) {
    const float d = f16bits(row.template u16<0>());
    const uint32_t qh = row.template u16<34 + 2 * SBI>();
    return d * (float)(2 * (int)((qh >> 12) & 7u) + 1);
  } else {  // KQ_IQ1_M, 16-weight blocks
    const uint32_t s0 = row.template u16<48>(), s1 = row.template u16<50>(), s2 = row.template u16<52>(),
                   s3 = row.template u16<54>();
    const float d = f16bits((s0 >> 12) | ((s1 >> 8) & 0x00f0u) | ((s2 >> 4) & 0x0f00u) | (s3 & 0xf000u));
    constexpr int ib = SBI >> 1;
    const uint32_t scw = ib < 2 ? s0 : ib < 4 ? s1 : ib < 6 ? s2 : s3;
    const int sc3 = (scw >> (6 * (ib & 1) + 3 * (SBI & 1))) & 7;
    return d * (float)(2 * sc3 + 1);
  }
}

// Decode tables of a workgroup of NT threads (callers put a barrier behind): the f16 codebook at grid_lds, the bit
// spreading at spread_lds.  BANKED: the pair table as one copy per LDS bank (see GROUPED_GRID_BYTES); contains a
// barrier of its own.
template <int C, int NT, bool BANKED>
__device__ __forceinline__ void build_tables(uint8_t* grid_lds, uint8_t* spread_lds, const uint8_t* grids, int tid) {
  using G = CodeGeom<C>;
  if constexpr (G::GRID_N > 0) {
    const uint8_t* src = grids + G::GRID_OFF;
    if constexpr (G::GRID_W == 8) {
      for (int e = tid; e < G::GRID_N; e += NT) {
        const u32x2 v = *reinterpret_cast<const u32x2*>(src + 8 * e);
        f16x8 f;
        if constexpr (G::GRID_SIGNED)
          f = bytes8_to_frag(v[0] ^ 0x80808080u, v[1] ^ 0x80808080u, 128.f);
        else
          f = bytes8_to_frag(v[0], v[1], 0.f);
        *reinterpret_cast<f16x8*>(grid_lds + 16 * e) = f;
      }
    } else {
      for (int e = tid; e < G::GRID_N; e += NT) {
        const uint32_t v = *reinterpret_cast<const uint32_t*>(src + 4 * e);
        uint32_t ev, od;
        bytes_to_f16(v, 0.f, ev, od);
        *reinterpret_cast<u32x2*>(grid_lds + 8 * e) = u32x2{ev, od};
      }
    }
  }
  if constexpr (G::PAIR_LUT) {
    // BANKED: one entry per thread into a plain table, then eight lanes write the 128 bytes of an entry's copies: a
    // wave store covers consecutive LDS
    uint32_t* plain = reinterpret_cast<uint32_t*>(BANKED ? grid_lds + 32768 : grid_lds);
    if (tid < 256) {
      const f16x2 e = C == KQ_MXFP4 ? f16x2{(_Float16)kq::kv_mxfp4(tid & 15), (_Float16)kq::kv_mxfp4(tid >> 4)}
                                    : f16x2{(_Float16)kq::kv_iq4nl(tid & 15), (_Float16)kq::kv_iq4nl(tid >> 4)};
      plain[tid] = __builtin_bit_cast(uint32_t, e);
    }
    if constexpr (BANKED) {
      lds_barrier();
      for (int i = tid; i < 256 * 8; i += NT) {
        const uint32_t ev = plain[i >> 3];
        *reinterpret_cast<u32x4*>(grid_lds + 16 * i) = u32x4{ev, ev, ev, ev};
      }
    }
  }
  if constexpr (G::SPREAD_BYTES > 0) {
    if (tid < 256) {
      const uint32_t b = tid;
      auto bit = [&](int i) { return (b >> i) & 1u; };
      constexpr int P = G::SPREAD_BIT;
      *reinterpret_cast<u32x4*>(spread_lds + 16 * tid) =
          u32x4{(bit(0) << P) | (bit(2) << (P + 16)), (bit(1) << P) | (bit(3) << (P + 16)),
                (bit(4) << P) | (bit(6) << (P + 16)), (bit(5) << P) | (bit(7) << (P + 16))};
    }
  }
}

}  // namespace kqcodes
