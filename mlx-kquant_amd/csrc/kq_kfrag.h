// B operands of v_mfma_f32_32x32x16_f16 from one K-quant superblock of one weight row in LDS, for kernels that keep
// their activation fragments in registers.  Lane (row l % 32, K half kg = l / 32).  Numerics are those of kq_mma.h: exact
// integers sc_j q from a masked field and one packed fma, the block's d on the f32 sum of the superblock, the minimum
// term as an extra product of the sub-block minima with the split sub-block sums of the activations.
//
// LDS row: the block's 16-byte pieces in order, the last one holding the block's last 16 bytes.
#pragma once

#include "kq_mma.h"

namespace kqfrag {

using namespace kqmma;

// Masks as the instructions want them: (a & mask) | magic is one v_and_or_b32 if the magic is a vector register and the
// mask a scalar one the compiler cannot see through.
struct KMasks {
  uint32_t magic, m[8];
  template <int C>
  __device__ __forceinline__ void init() {
    magic = opaque_vgpr(0x64006400u);
    if constexpr (C == KQ_Q4_K || C == KQ_Q5_K) {
      m[0] = opaque_sgpr(0x000f000fu);
      m[1] = opaque_sgpr(0x00f000f0u);
    }
    if constexpr (C == KQ_Q5_K) {
      m[2] = opaque_sgpr(0x00100010u);
      m[3] = opaque_sgpr(0x01000100u);
    }
    if constexpr (C == KQ_Q6_K) {
      m[0] = opaque_sgpr(0x00f000f0u);
      m[1] = opaque_sgpr(0x03000300u);
    }
    if constexpr (C == KQ_Q2_K || C == KQ_Q3_K)
      for (int j = 0; j < 4; j++) m[j] = opaque_sgpr(0x00030003u << (2 * j));
    if constexpr (C == KQ_Q3_K)
      for (int j = 0; j < 4; j++) m[4 + j] = opaque_sgpr(0x00010001u << (2 * j + 2));
  }
};

template <int C>
struct KRow;

template <int C>
struct KRow45 {
  static constexpr int QS = C == KQ_Q4_K ? 16 : 48;
  static constexpr int TERMS = 1, NSUM = 1;
  static constexpr float XUNIT = 32.0f;  // X_j = 32 (hi_j + lo_j)
  uint4 qv[4];
  uint32_t hb[4], scw[2], mnw[2];
  float d, dm;
  __device__ __forceinline__ void load(const uint8_t* b, int kg) {
    const uint4 hdr = *reinterpret_cast<const uint4*>(b);
#pragma unroll
    for (int g = 0; g < 4; g++) qv[g] = *reinterpret_cast<const uint4*>(b + QS + 32 * g + 16 * kg);
    if constexpr (C == KQ_Q5_K) {
      const uint4 hv = *reinterpret_cast<const uint4*>(b + 16 + 16 * kg);
      hb[0] = hv.x;
      hb[1] = hv.y;
      hb[2] = hv.z;
      hb[3] = hv.w;
    }
    d = kq::h2f((uint16_t)(hdr.x & 0xffff));
    dm = kq::h2f((uint16_t)(hdr.x >> 16)) * -XUNIT;
    scw[0] = hdr.y & 0x3f3f3f3fu;
    scw[1] = (hdr.w & 0x0f0f0f0fu) | ((hdr.y >> 2) & 0x30303030u);
    mnw[0] = hdr.z & 0x3f3f3f3fu;
    mnw[1] = ((hdr.w >> 4) & 0x0f0f0f0fu) | ((hdr.z >> 2) & 0x30303030u);
  }
  // fragment J = 2 j + s: sub-block j, weights 16 kg + 8 s .. + 7 of it
  template <int J>
  __device__ __forceinline__ void frag(int, const KMasks& k, f16x8* out) const {
    constexpr int j = J >> 1, s = J & 1, g = j >> 1, h = j & 1;
    const uint32_t magic = k.magic;
    const uint32_t qw[4] = {qv[g].x, qv[g].y, qv[g].z, qv[g].w};
    const float scf = (float)((scw[j >> 2] >> (8 * (j & 3))) & 0xff);
    // low nibbles read 1024 + q, high nibbles (in place) 1024 + 16 q: the 16 goes into the scale
    const _Float16 sch = (_Float16)(h ? scf * 0.0625f : scf), off = (_Float16)(-(h ? 64.0f : 1024.0f) * scf);
    const f16x2 scp = {sch, sch}, offp = {off, off};
    const uint32_t mask = k.m[h];
    uint32_t fr[4] = {(qw[2 * s] & mask) | magic, ((qw[2 * s] >> 8) & mask) | magic, (qw[2 * s + 1] & mask) | magic,
                      ((qw[2 * s + 1] >> 8) & mask) | magic};
    if constexpr (C == KQ_Q5_K) {
      // fifth bit of weight (j, i) is bit j of qh[i]: to bit 4 beside a low nibble, bit 8 beside a high one in place
      constexpr int P = h ? 8 : 4;
      const uint32_t mbit = k.m[2 + h];
      auto place = [&](uint32_t word, int from) -> uint32_t { return from >= P ? word >> (from - P) : word << (P - from); };
      fr[0] |= place(hb[2 * s], j) & mbit;
      fr[1] |= place(hb[2 * s], j + 8) & mbit;
      fr[2] |= place(hb[2 * s + 1], j) & mbit;
      fr[3] |= place(hb[2 * s + 1], j + 8) & mbit;
    }
    f16x2 bq[4];
#pragma unroll
    for (int e = 0; e < 4; e++) bq[e] = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, fr[e]), scp, offp);
    out[0] = f16x8{bq[0][0], bq[0][1], bq[1][0], bq[1][1], bq[2][0], bq[2][1], bq[3][0], bq[3][1]};
  }
  // K slots 0..7 meet the hi halves of the sums, 8..15 the lo halves
  template <int>
  __device__ __forceinline__ f16x8 min_frag(int) const {
    f16x8 m;
#pragma unroll
    for (int j = 0; j < 8; j++) m[j] = (_Float16)(float)((mnw[j >> 2] >> (8 * (j & 3))) & 0xff);
    return m;
  }
};
template <>
struct KRow<KQ_Q4_K> : KRow45<KQ_Q4_K> {};
template <>
struct KRow<KQ_Q5_K> : KRow45<KQ_Q5_K> {};

// sc (q - 32) as two exact terms, sc ql and 16 sc (qh - 2)
template <>
struct KRow<KQ_Q6_K> {
  static constexpr int TERMS = 2, NSUM = 0;
  uint4 hv[2], qv[4], scv;
  float d, dm;
  __device__ __forceinline__ void load(const uint8_t* b, int kg) {
    scv = *reinterpret_cast<const uint4*>(b + 192);
#pragma unroll
    for (int hf = 0; hf < 2; hf++) {
      hv[hf] = *reinterpret_cast<const uint4*>(b + 128 + 32 * hf + 16 * kg);
#pragma unroll
      for (int qr = 0; qr < 2; qr++) qv[2 * hf + qr] = *reinterpret_cast<const uint4*>(b + 64 * hf + 32 * qr + 16 * kg);
    }
    d = kq::h2f((uint16_t)(*reinterpret_cast<const uint32_t*>(b + 220) >> 16));  // block bytes 194 .. 209 lie at 208
    dm = 0.f;
  }
  template <int J>
  __device__ __forceinline__ void frag(int kg, const KMasks& k, f16x8* out) const {
    constexpr int j = J >> 1, s = J & 1, hf = j >> 2, t4 = j & 3, qr = t4 & 1, h = t4 >> 1;
    const uint32_t magic = k.magic;
    const uint32_t scw[4] = {scv.x, scv.y, scv.z, scv.w};
    const uint32_t hw[4] = {hv[hf].x, hv[hf].y, hv[hf].z, hv[hf].w};
    const uint32_t qw[4] = {qv[2 * hf + qr].x, qv[2 * hf + qr].y, qv[2 * hf + qr].z, qv[2 * hf + qr].w};
    const float scf = (float)(int)__builtin_amdgcn_sbfe((int)scw[2 * hf + (t4 >> 1)], 8 * (2 * (t4 & 1) + kg), 8);
    const _Float16 sch = (_Float16)(scf * 0.0625f), ofl = (_Float16)(-64.0f * scf), ofh = (_Float16)(-96.0f * scf);
    const f16x2 scp = {sch, sch}, oflp = {ofl, ofl}, ofhp = {ofh, ofh};
    uint32_t fl[4], fh[4];
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const uint32_t q = qw[2 * s + e], hq = hw[2 * s + e];
      const uint32_t qe = h ? q : (q << 4), qo = h ? (q >> 8) : (q >> 4);
      const uint32_t he = hq << (8 - 2 * t4), ho = t4 ? (hq >> (2 * t4)) : hq;
      fl[2 * e] = (qe & k.m[0]) | magic;
      fl[2 * e + 1] = (qo & k.m[0]) | magic;
      fh[2 * e] = (he & k.m[1]) | magic;
      fh[2 * e + 1] = (ho & k.m[1]) | magic;
    }
    f16x2 bl[4], bh[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      bl[e] = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, fl[e]), scp, oflp);
      bh[e] = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, fh[e]), scp, ofhp);
    }
    out[0] = f16x8{bl[0][0], bl[0][1], bl[1][0], bl[1][1], bl[2][0], bl[2][1], bl[3][0], bl[3][1]};
    out[1] = f16x8{bh[0][0], bh[0][1], bh[1][0], bh[1][1], bh[2][0], bh[2][1], bh[3][0], bh[3][1]};
  }
};

// One fragment = one 16-weight sub-block = one scale.  The rest of the weight, -dmin m_s (q2_k) or -4 d sc_s (q3_k), goes
// through the sums: minima fragment 0 meets the hi halves, fragment 1 the lo halves, sub-blocks 8 kg .. + 7 each.
template <int C>
struct KRow23 {
  static constexpr int QS = C == KQ_Q2_K ? 16 : 32;
  static constexpr int TERMS = 1, NSUM = 2;
  static constexpr float XUNIT = 16.0f;
  uint2 qv[4], hv[2];
  uint32_t lsc[4];  // q2_k: scale / minimum bytes; q3_k: unpacked 6-bit scales
  float d, dm;
  __device__ __forceinline__ void load(const uint8_t* b, int kg) {
#pragma unroll
    for (int i = 0; i < 4; i++) qv[i] = *reinterpret_cast<const uint2*>(b + QS + 16 * i + 8 * kg);
    if constexpr (C == KQ_Q2_K) {
      const uint4 sv = *reinterpret_cast<const uint4*>(b);
      lsc[0] = sv.x;
      lsc[1] = sv.y;
      lsc[2] = sv.z;
      lsc[3] = sv.w;
      const uint32_t dd = *reinterpret_cast<const uint32_t*>(b + 92);
      d = kq::h2f((uint16_t)(dd & 0xffff));
      dm = kq::h2f((uint16_t)(dd >> 16)) * -XUNIT;
    } else {
#pragma unroll
      for (int h = 0; h < 2; h++) hv[h] = *reinterpret_cast<const uint2*>(b + 16 * h + 8 * kg);
      const uint4 t = *reinterpret_cast<const uint4*>(b + 96);  // block bytes 94 .. 109
      const uint32_t aux0 = __builtin_amdgcn_alignbyte(t.y, t.x, 2), aux1 = __builtin_amdgcn_alignbyte(t.z, t.y, 2);
      const uint32_t tmp = __builtin_amdgcn_alignbyte(t.w, t.z, 2);
      d = kq::h2f((uint16_t)(t.w >> 16));
      dm = d * -XUNIT;
      lsc[0] = (aux0 & 0x0f0f0f0fu) | ((tmp & 0x03030303u) << 4);
      lsc[1] = (aux1 & 0x0f0f0f0fu) | (((tmp >> 2) & 0x03030303u) << 4);
      lsc[2] = ((aux0 >> 4) & 0x0f0f0f0fu) | (((tmp >> 4) & 0x03030303u) << 4);
      lsc[3] = ((aux1 >> 4) & 0x0f0f0f0fu) | (((tmp >> 6) & 0x03030303u) << 4);
    }
  }
  template <int J>
  __device__ __forceinline__ void frag(int, const KMasks& k, f16x8* out) const {
    constexpr int p = J >> 3, g = J & 7, j = g >> 1, h = g & 1;
    const uint32_t magic = k.magic;
    const uint32_t mask = k.m[j];
    const uint32_t sb8 = (lsc[J >> 2] >> (8 * (J & 3))) & 0xff;
    const float scf = C == KQ_Q2_K ? (float)(sb8 & 15) : (float)(int)sb8 - 32.0f;
    constexpr float f = 1.0f / (float)(1 << (2 * j));  // the field reads 4^j q
    const _Float16 sch = (_Float16)(scf * f), off = (_Float16)(-1024.0f * f * scf);
    const f16x2 scp = {sch, sch}, offp = {off, off};
    const uint32_t w0 = qv[2 * p + h].x, w1 = qv[2 * p + h].y;
    uint32_t fr[4] = {(w0 & mask) | magic, ((w0 >> 8) & mask) | magic, (w1 & mask) | magic, ((w1 >> 8) & mask) | magic};
    if constexpr (C == KQ_Q3_K) {
      constexpr int from = 4 * p + j, to = 2 * j + 2;  // third bit: hmask bit 4 p + j, to the place beside the field
      const uint32_t mbit = k.m[4 + j];
      auto place = [&](uint32_t word, int fb) -> uint32_t { return fb >= to ? word >> (fb - to) : word << (to - fb); };
      fr[0] |= place(hv[h].x, from) & mbit;
      fr[1] |= place(hv[h].x, from + 8) & mbit;
      fr[2] |= place(hv[h].y, from) & mbit;
      fr[3] |= place(hv[h].y, from + 8) & mbit;
    }
    f16x2 bq[4];
#pragma unroll
    for (int e = 0; e < 4; e++) bq[e] = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, fr[e]), scp, offp);
    out[0] = f16x8{bq[0][0], bq[0][1], bq[1][0], bq[1][1], bq[2][0], bq[2][1], bq[3][0], bq[3][1]};
  }
  template <int>
  __device__ __forceinline__ f16x8 min_frag(int kg) const {
    f16x8 m;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const uint32_t w = pick(kg, lsc[j >> 2], lsc[2 + (j >> 2)]);
      const uint32_t b = (w >> (8 * (j & 3))) & 0xff;
      m[j] = C == KQ_Q2_K ? (_Float16)(float)(b >> 4) : (_Float16)(4.0f * ((float)(int)b - 32.0f));
    }
    return m;
  }

 private:
  __device__ static __forceinline__ uint32_t pick(int kg, uint32_t a, uint32_t b) { return kg ? b : a; }
};
template <>
struct KRow<KQ_Q2_K> : KRow23<KQ_Q2_K> {};
template <>
struct KRow<KQ_Q3_K> : KRow23<KQ_Q3_K> {};

}  // namespace kqfrag
