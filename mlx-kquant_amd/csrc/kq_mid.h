// What the matmuls of 9 rows and more on any codec share (kq_mid.hip, kq_tile.hip): the wire geometry of a 256-weight step in
// LDS, a row of it in registers, and the step of a block that holds a row of wide range.
#pragma once

#include "kq_codes.h"
#include "kq_decode.h"
#include "kq_dma.h"
#include "kq_kfrag.h"

namespace kqmid {

using namespace kqcodes;
using namespace kqdma;
using kqmma::u32x4;

template <int C>
constexpr bool k_quant() { return C <= KQ_Q6_K; }
template <int C>
constexpr bool fp4() { return C == KQ_MXFP4 || C == KQ_NVFP4; }

// Wire geometry of a step (256 weights of a row) in LDS: piece p < PIECES - 1 holds bytes 16 p .., the last one the step's
// last 16 bytes.  Rows are an odd number of pieces apart (a dummy piece where needed): conflict-free row-per-lane reads.
template <int C>
struct MidGeom {
  static constexpr int WPB = kq_geom(C).wpb, BPB = kq_geom(C).bpb;
  static constexpr int BYTES = CK_STEP / WPB * BPB;
  static constexpr int PIECES = (BYTES + 15) / 16, LP = PIECES | 1, LROW = 16 * LP;
  static constexpr int LOADS = (32 * LP + 63) / 64;
  // activation order (store_frags) and sum fragments per step
  static constexpr int ORD = C == KQ_Q4_K || C == KQ_Q5_K || C == KQ_Q6_K                       ? 0
                             : C == KQ_IQ4_NL || C == KQ_IQ4_XS || C == KQ_MXFP4 ? 2
                             : C == KQ_NVFP4                                     ? 3
                                                                                 : 1;
  static constexpr int NSUM = C == KQ_Q2_K || C == KQ_Q3_K ? 2 : C == KQ_Q4_K || C == KQ_Q5_K || C == KQ_Q4_1 || C == KQ_Q5_1 ? 1 : 0;
  static constexpr int NF = 16 + NSUM;  // fragments per step
};
template <int C>
constexpr int mid_slot_bytes() { return MidGeom<C>::LROW * 32 > 4096 ? MidGeom<C>::LROW * 32 : 4096; }
template <int C>
constexpr int mid_table_bytes() {
  if constexpr (k_quant<C>() || fp4<C>()) return 0;
  else return CodeGeom<C>::GROUPED_GRID_BYTES + CodeGeom<C>::SPREAD_BYTES;
}

// Eight consecutive activations h (8-group pc of a row's step) to the step's fragments, 1 KiB each of [lane = 32 kg + row][8
// halves]; `step` is the step's first fragment plus 16 bytes per row of the block of 32.
// ORD 0 (q4_k / q5_k / q6_k): fragment 2 j + s, half kg = weights 32 j + 16 kg + 8 s .. of the step; ORD 1: fragment J,
// half kg = weights 16 J + 8 kg ..; both k0 k2 k1 k3 k4 k6 k5 k7 inside the eight; ORD 2: as ORD 1 with the positions of
// x[j], x[j + 16] interleaved over every 32 (ORD 3: x[j], x[j + 8] over every 16).  NSUM 1: fragment 16 = sums of the eight 32-wide blocks, kg 0 the f16 part hi,
// kg 1 the remainder lo, X = 32 (hi + lo); NSUM 2: fragments 16 / 17 = hi / lo of the sixteen 16-wide sums, X = 16 (hi + lo).
// Whole octets of lanes call together, lane by lane consecutive groups.  SWZ, for fragments in LDS: row r of half kg of fragment
// J < 16 lies in place r ^ (2 J + kg), so that the 32 groups of a row, written by 32 lanes at once, meet 32 different places.
template <int ORD, int NSUM, bool SWZ = false>
__device__ __forceinline__ void store_frags(uint8_t* step, int pc, const _Float16 (&h)[8], int row = 0) {
  auto at = [&](int q) { return step + 512 * q + (SWZ ? 16 * (row ^ q) - 16 * row : 0); };  // q = 2 J + kg
  if constexpr (ORD >= 2) {
    uint32_t own[4], par[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      own[e] = (uint32_t)__builtin_bit_cast(uint16_t, h[2 * e]) | ((uint32_t)__builtin_bit_cast(uint16_t, h[2 * e + 1]) << 16);
      // the neighbour two (ORD 3: one) groups on: quad_perm [2,3,0,1] or [1,0,3,2]
      par[e] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)own[e], ORD == 2 ? 0x4E : 0xB1, 0xf, 0xf, true);
    }
    const bool high = (pc & (ORD == 2 ? 2 : 1)) != 0;
    const uint32_t a0 = high ? par[2] : own[0], a1 = high ? par[3] : own[1];
    const uint32_t b0 = high ? own[2] : par[0], b1 = high ? own[3] : par[1];
    const u32x4 o = {(a0 & 0xffffu) | (b0 << 16), (a0 >> 16) | (b0 & 0xffff0000u), (a1 & 0xffffu) | (b1 << 16),
                     (a1 >> 16) | (b1 & 0xffff0000u)};
    const int pos = ORD == 2 ? 4 * (pc >> 2) + 2 * (pc & 1) + (high ? 1 : 0) : pc;
    *reinterpret_cast<u32x4*>(at(pos)) = o;
  } else {
    const int J = ORD == 0 ? 2 * (pc >> 2) + (pc & 1) : pc >> 1, kg = ORD == 0 ? (pc >> 1) & 1 : pc & 1;
    *reinterpret_cast<f16x8*>(at(2 * J + kg)) = f16x8{h[0], h[2], h[1], h[3], h[4], h[6], h[5], h[7]};
  }
  if constexpr (NSUM > 0) {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) s += (float)h[e];
    s += __shfl_xor(s, 1);
    if constexpr (NSUM == 1) s += __shfl_xor(s, 2);
    constexpr float unit = NSUM == 1 ? 32.0f : 16.0f;
    const _Float16 hi = (_Float16)(s * (1.0f / unit)), lo = (_Float16)((s - unit * (float)hi) * (1.0f / unit));
    if constexpr (NSUM == 1) {
      if ((pc & 3) == 0) {
        *reinterpret_cast<_Float16*>(step + 16 * 1024 + 2 * (pc >> 2)) = hi;
        *reinterpret_cast<_Float16*>(step + 16 * 1024 + 512 + 2 * (pc >> 2)) = lo;
      }
    } else if ((pc & 1) == 0) {
      const int sb = pc >> 1;
      *reinterpret_cast<_Float16*>(step + 16 * 1024 + 512 * (sb >> 3) + 2 * (sb & 7)) = hi;
      *reinterpret_cast<_Float16*>(step + 17 * 1024 + 512 * (sb >> 3) + 2 * (sb & 7)) = lo;
    }
  }
}

// Row bytes of a step from LDS into registers (codes of kq_codes.h).  The long blocks come in two halves, to leave
// room for the activation fragments; the short ones whole, byte b being dword b / 4 again once the last piece has been
// moved to where its bytes belong.
template <int C>
constexpr int row_parts() { return MidGeom<C>::BYTES >= 160 ? 2 : 1; }
template <int C, int P>
struct RowPart {
  using G = MidGeom<C>;
  static constexpr int LEN = G::BYTES / row_parts<C>(), BASE = P * LEN, NDW = (LEN + 15) / 16 * 4;
  RowRegs<NDW> r;
  template <int OFF>
  __device__ __forceinline__ uint32_t u32() const { return r.template u32<OFF - BASE>(); }
  template <int OFF>
  __device__ __forceinline__ uint32_t u16() const { return r.template u16<OFF - BASE>(); }
  template <int OFF>
  __device__ __forceinline__ uint32_t u8() const { return r.template u8<OFF - BASE>(); }
  __device__ __forceinline__ void load(const uint8_t* b) {
    if constexpr (row_parts<C>() == 2) {
      static_assert(row_parts<C>() == 1 || (G::BYTES % 16 == 0 && LEN % 8 == 0), "halves of whole pieces in 8-byte reads");
#pragma unroll
      for (int i = 0; i < LEN / 8; i++) {
        const u32x2 v = *reinterpret_cast<const u32x2*>(b + BASE + 8 * i);
        r.d[2 * i] = v[0];
        r.d[2 * i + 1] = v[1];
      }
    } else {
      constexpr int R = G::BYTES % 16;
      StaticFor<G::PIECES>::run([&](auto pc) {
        constexpr int p = decltype(pc)::value;
        const u32x4 v = *reinterpret_cast<const u32x4*>(b + 16 * p);
        constexpr int sh = p < G::PIECES - 1 || R == 0 ? 0 : 16 - R;
        const uint32_t e[5] = {v[0], v[1], v[2], v[3], 0u};
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int q = sh / 4 + i;
          r.d[4 * p + i] = q >= 4 ? 0u : sh % 4 == 0 ? e[q] : __builtin_amdgcn_alignbyte(e[q + 1], e[q], sh % 4);
        }
      });
    }
  }
};

// B operand of the fp4 codecs by the hardware's fp4 -> f16 conversion: a byte gives the pair of its two codes.  nvfp4:
// times the 16-weight scale, an f16 number (its bits (x & 0x7f) << 7 read the e4m3 value / 256; 0x7f decodes to 0), so
// nothing is left to do after the MFMA; mxfp4: the codes doubled, as the block scale expects them.
template <int C, int J, class R>
__device__ __forceinline__ f16x8 fp4_frag(const R& row, int kg) {
  constexpr int off = C == KQ_NVFP4 ? (J / 4) * 36 + 4 + 8 * (J & 3) : (J / 2) * 17 + 1 + 8 * (J & 1);
  const uint32_t w = pick(kg, row.template u32<off>(), row.template u32<off + 4>());
  constexpr float cs = C == KQ_NVFP4 ? 1.0f : 2.0f;
  f16x2 p[4];
  p[0] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, cs, 0);
  p[1] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, cs, 1);
  p[2] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, cs, 2);
  p[3] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, cs, 3);
  if constexpr (C == KQ_NVFP4) {
    const uint32_t x = row.template u8<(J / 4) * 36 + (J & 3)>();
    const uint32_t hb = x == 0x7fu ? 0u : (x & 0x7fu) << 7;
    const f16x2 sp = __builtin_bit_cast(f16x2, hb | (hb << 16)) * f16x2{(_Float16)256.0f, (_Float16)256.0f};
#pragma unroll
    for (int e = 0; e < 4; e++) p[e] *= sp;
  }
  return f16x8{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
}

// acc += (32 weight rows of the step in LDS at b_lane) . (32 activation rows in the fragments a)
template <int C>
__device__ __forceinline__ void mid_step(const uint8_t* b_lane, int kg, const f16x8 (&a)[MidGeom<C>::NF], const Tables& tabs,
                                         const kqfrag::KMasks& masks, int kvalid, f32x16& acc) {
  if constexpr (k_quant<C>()) {
    kqfrag::KRow<C> row;
    row.load(b_lane, kg);
    f32x16 part = f32x16{0};
    StaticFor<16>::run([&](auto jc) {
      constexpr int J = decltype(jc)::value;
      f16x8 b[2];
      row.template frag<J>(kg, masks, b);
      part = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[J], b[0], part, 0, 0, 0);
      if constexpr (kqfrag::KRow<C>::TERMS == 2) part = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[J], b[1], part, 0, 0, 0);
    });
#pragma unroll
    for (int i = 0; i < 16; i++) acc[i] = fmaf(row.d, part[i], acc[i]);
    if constexpr (kqfrag::KRow<C>::NSUM > 0) {
      const f16x8 m = row.template min_frag<0>(kg);
      part = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[16], m, f32x16{0}, 0, 0, 0);
      if constexpr (kqfrag::KRow<C>::NSUM == 2) part = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[17], m, part, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 16; i++) acc[i] = fmaf(row.dm, part[i], acc[i]);
    }
  } else {
    using G = CodeGeom<C>;
    constexpr int MPS = G::SB / 16, PARTS = row_parts<C>(), JP = 16 / PARTS;
    auto run = [&](auto full_c) {
      constexpr bool FULL = decltype(full_c)::value;
      f32x16 part[2];
      f16x8 mins = {};
      StaticFor<PARTS>::run([&](auto pc) {
        constexpr int P = decltype(pc)::value;
        RowPart<C, P> row;
        row.load(b_lane);
        StaticFor<JP>::run([&](auto jc) {
          constexpr int J = P * JP + decltype(jc)::value;
          if (FULL || 16 * J < kvalid) {  // uniform
            if constexpr (C == KQ_NVFP4) {
              acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[J], fp4_frag<C, J>(row, kg), acc, 0, 0, 0);
              return;
            }
            f16x8 b;
            if constexpr (C == KQ_MXFP4) b = fp4_frag<C, J>(row, kg);
            else b = codes<C, J>(row, kg, tabs);
            constexpr int sbi = J / MPS, slot = sbi & 1;
            if constexpr (J % MPS == 0)
              part[slot] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[J], b, f32x16{0}, 0, 0, 0);
            else
              part[slot] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[J], b, part[slot], 0, 0, 0);
            if constexpr (J % MPS == MPS - 1) {
              float mn;
              const float sc = block_scale<C, sbi>(row, mn);
#pragma unroll
              for (int i = 0; i < 16; i++) acc[i] = fmaf(sc, part[slot][i], acc[i]);
              if constexpr (G::HAS_MIN) mins[sbi] = (_Float16)mn;  // the f16 it came from
            }
          }
        });
      });
      if constexpr (G::HAS_MIN) {  // blocks past the end of K: minimum 0 on sums of zeros
        part[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[16], mins, f32x16{0}, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 16; i++) acc[i] = fmaf(32.0f, part[0][i], acc[i]);
      }
    };
    if (kvalid >= CK_STEP)
      run(std::true_type{});
    else
      run(std::false_type{});
  }
}

// The step of a block that holds a row of wide range: bf16 activations as they are, weights by the reference-order decoder
// from global memory in two bf16 terms (16 significant bits), the numerics of the any-codec kernel.  Rare, so small code
// rather than speed: q8_0 4096 x 4096, 32 rows, 32 us (ordinary rows 13, the any-codec kernel 18).
template <int C, class Args>
__device__ __forceinline__ void wide_step(const Args& a, int row0, int nrows, int mb, int st, int l32, int kg,
                                          uint32_t row_bytes, f32x16& acc) {
  using G = MidGeom<C>;
  typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
  const int m = 32 * mb + l32 < a.M ? 32 * mb + l32 : a.M - 1, n = row0 + (l32 < nrows ? l32 : nrows - 1);
  const uint16_t* x = a.x + (size_t)m * a.K;
  const uint8_t* w = a.w + (size_t)n * row_bytes;
  const int end = CK_STEP * (st + 1) < a.K ? CK_STEP * (st + 1) : a.K;
#pragma unroll 1
  for (int k0 = CK_STEP * st; k0 < end; k0 += 16) {  // K is a multiple of 32
    const int k = k0 + 8 * kg;
    float f[8];
    kq::decode8<C>(w + (size_t)(k / G::WPB) * G::BPB, k % G::WPB / 8, a.grids, f);
    bf16x8 hi, lo;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const uint32_t top = __builtin_bit_cast(uint32_t, f[e]) & 0xffff0000u;
      hi[e] = __builtin_bit_cast(__bf16, (uint16_t)(top >> 16));
      lo[e] = (__bf16)(f[e] - __builtin_bit_cast(float, top));
    }
    const bf16x8 xv = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(x + k));
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xv, hi, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xv, lo, acc, 0, 0, 0);
  }
}

}  // namespace kqmid
