// Down projection of MoE decode with the routing mix in one launch: out[t] = sum over the slots s of scores[t][s] * (W_s . x[t][s]).
//
// The sums are those of gather_mix_generic_kernel (kq_generic.hip), bit for bit: f32 products of the activations as they are and
// the decoded weights, in the same order.  Virtual wave c of four takes the slots c, c + 4, ...; lane l of it the groups of 8 weights
// l, l + 64, ... of a row; a lane's sums are mixed by the slots' scores, added over the lanes by halves and over the four in turn.
//
// What bounds it: at one token latency (expert id -> address -> weights -> results), then the vector ALU (decode, product and sum of
// a weight in f32).  That kernel reads a weight's bytes one by one in the order of their use, a workgroup per output element.  Here:
//   * Workgroup = 8 waves, 8 weight rows: wave = virtual wave x half of the rows, so that a fetched activation serves four rows.
//   * What a wave will read (its slots' activations and, per slot, four rows, which lie one behind another) is requested at once
//     with direct-to-LDS loads, as many slots as fit (mix_depth); a slot that has been read makes room for the next.
//   * Weights are decoded from words in LDS instead of bytes from memory.
//   * A row's last 32 groups of 8, where K is an odd multiple of 256, would idle half of the lanes: they take two rows at once.
// us, top-8 on 128 experts of 2048 x 768, one token (without tiles): q6_k 7.6 (12.7), q4_k 7.7 (14.6), q8_0 7.6 (9.4); of q6_k's 9.6 before,
// 8-byte reads of half-word alignment were 1.1 and the idle lanes 0.6.  Longer slots, 64 experts: top-8 of 4096 x 1536 q6_k 15.4 (28.4),
// q4_k 15.8 (35.3); top-4 of 4096 x 2816 mxfp4 16.7 (26.8); top-2 of 4096 x 4096 q6_k 23.0 (26.3).  The streamed kernel's matrix
// instructions would take 10 us for the 33 M weights of 4096 x 2048 top-4 (here q6_k 15.7), in less precise sums.
#include <algorithm>

#include "kq_decode.h"
#include "kq_dma.h"
#include "kq_epilogue.h"

namespace {

using namespace kqdma;

constexpr int MX_CLASSES = 4, MX_HALVES = 2, MX_WAVES = MX_CLASSES * MX_HALVES, MX_R = 4, MX_ROWS = MX_R * MX_HALVES;
constexpr int MX_LDS = 160 * 1024 - (int)sizeof(float) * MX_CLASSES * MX_ROWS;

struct MixArgs {
  const uint16_t* x;       // [T][S][K]
  const uint8_t* w;        // [E][N][row bytes]
  const uint8_t* shexp_w;  // [N][row bytes] or null
  const uint32_t* idx;     // [T][routed]
  const float* scores;     // [T][S]
  const float* bias;       // [E][N] or null
  void* out;               // [T][N]
  const uint8_t* grids;
  int S, routed, E, N, K, tiles;
  int depth;               // regions of a wave: slots under way at once
  int64_t w_expert_stride;
};

// codebook of a codec, copied to LDS per wave
template <int C>
constexpr int mix_grid_bytes() { return C == KQ_IQ3_S || C == KQ_IQ2_XXS ? 2048 : 0; }
template <int C>
constexpr int mix_grid_at() { return C == KQ_IQ3_S ? KQ_GRID_IQ3S : KQ_GRID_IQ2XXS; }

// A region, LDS of a wave and slot: the slot's activations, four rows of weights, what 16-byte alignment adds and what words8 reads past them
__host__ __device__ constexpr int mix_region(int K, int row_bytes) { return 2 * K + ((MX_R * row_bytes + 15) & ~15) + 32; }

// 8 bytes of a codec's block.  Blocks of no whole number of words: from the three words that hold them (an 8-byte LDS read of
// half-word alignment takes several times as long).
template <int C>
__device__ __forceinline__ uint2 words8(const uint8_t* p) {
  uint2 v;
  if constexpr (kq_geom(C).bpb % 4 == 0) {
    __builtin_memcpy(&v, p, 8);
  } else {
    const uint32_t at = (uint32_t)reinterpret_cast<uintptr_t>(p) & 3;
    const uint32_t* d = reinterpret_cast<const uint32_t*>(p - at);
    v = make_uint2(__builtin_amdgcn_alignbyte(d[1], d[0], at), __builtin_amdgcn_alignbyte(d[2], d[1], at));
  }
  return v;
}
__device__ __forceinline__ uint16_t word2(const uint8_t* p) {
  uint16_t v;
  __builtin_memcpy(&v, p, 2);
  return v;
}
// entries of a table of 16 signed bytes for the four codes (0 .. 15) in the bytes of n
__device__ __forceinline__ uint32_t table4(uint64_t lo, uint64_t hi, uint32_t n) {
  const uint32_t sel = n & 0x07070707u, top = (n & 0x08080808u) >> 3, mask = (top << 8) - top;
  const uint32_t a = __builtin_amdgcn_perm((uint32_t)(lo >> 32), (uint32_t)lo, sel);
  const uint32_t b = __builtin_amdgcn_perm((uint32_t)(hi >> 32), (uint32_t)hi, sel);
  return (b & mask) | (a & ~mask);
}
// byte t as a number
__device__ __forceinline__ float ub(uint2 w, int t) { return (float)((t < 4 ? w.x >> (8 * t) : w.y >> (8 * (t - 4))) & 0xffu); }
__device__ __forceinline__ float sb(uint2 w, int t) { return (float)(int8_t)((t < 4 ? w.x >> (8 * t) : w.y >> (8 * (t - 4))) & 0xffu); }
__device__ __forceinline__ uint2 bits(uint2 q, int shift, uint32_t mask) {
  uint2 v = make_uint2((q.x >> shift) & mask, (q.y >> shift) & mask);
  asm("" : "+v"(v.x), "+v"(v.y));  // or every byte is extracted on its own
  return v;
}
// bytes below 128 less c each, as signed bytes
__device__ __forceinline__ uint2 less(uint2 q, uint32_t c) {
  const uint32_t add = (128u - c) * 0x01010101u;
  return make_uint2((q.x + add) ^ 0x80808080u, (q.y + add) ^ 0x80808080u);
}
__device__ __forceinline__ uint2 either(uint2 a, uint2 b) { return make_uint2(a.x | b.x, a.y | b.y); }
__device__ __forceinline__ uint2 up(uint2 a, int shift) { return make_uint2(a.x << shift, a.y << shift); }

// Weights 8 g .. 8 g + 7 of a block: kq::decode8 in two halves, its bytes fetched as words (so that the reads of several rows are
// under way together) and the same operations on the same values.
template <int C>
struct Group {
  uint2 q, h;              // codes, high bits (iq3_s, iq2_xxs: magnitudes)
  uint16_t d_bits, m_bits;  // f16 scales of the block
  uint32_t s[3];           // bytes of the group's scale (iq3_s, iq2_xxs: its signs)
  float db;                // iq3_s, iq2_xxs: the group's scale
  __device__ __forceinline__ void load(const uint8_t* b, int g, const uint8_t* grids) {
    const int w = 8 * g, half = w >> 7, r = w & 127, l0 = r & 31;  // of the codecs of two halves of 128
    if constexpr (C == KQ_Q8_0) {
      d_bits = word2(b);
      q = words8<C>(b + 2 + 8 * g);
    } else if constexpr (C == KQ_Q4_0 || C == KQ_IQ4_NL) {
      d_bits = word2(b);
      q = words8<C>(b + 2 + 8 * (g & 1));
    } else if constexpr (C == KQ_Q4_K || C == KQ_Q5_K) {
      d_bits = word2(b), m_bits = word2(b + 2);
      const int j = g >> 2, i0 = 8 * (g & 3);
      // scale j, min j (j < 4); their high bits, low bits of both (j > 3)
      s[0] = b[j < 4 ? 4 + j : j], s[1] = b[8 + (j & 3)], s[2] = b[8 + j];
      q = words8<C>(b + (C == KQ_Q4_K ? 16 : 48) + 32 * (j >> 1) + i0);
      if constexpr (C == KQ_Q5_K) h = words8<C>(b + 16 + i0);
    } else if constexpr (C == KQ_Q6_K) {
      d_bits = word2(b + 208);
      s[0] = b[192 + (w >> 4)];
      q = words8<C>(b + 64 * half + (((r >> 5) & 1) ? 32 : 0) + l0);
      h = words8<C>(b + 128 + 32 * half + l0);
    } else if constexpr (C == KQ_Q3_K) {
      const int is = w >> 4, k = is & 3, grp = is >> 2;
      d_bits = word2(b + 108);
      s[0] = b[96 + k + 4 * (grp & 1)], s[1] = b[104 + k];
      q = words8<C>(b + 32 + 32 * half + l0);
      h = words8<C>(b + l0);
    } else if constexpr (C == KQ_Q2_K) {
      d_bits = word2(b + 80), m_bits = word2(b + 82);
      s[0] = b[w >> 4];
      q = words8<C>(b + 16 + 32 * half + l0);
    } else if constexpr (C == KQ_IQ4_XS) {
      d_bits = word2(b);
      s[0] = b[4 + (g >> 3)], s[1] = word2(b + 2);
      q = words8<C>(b + 8 + 16 * (g >> 2) + 8 * (g & 1));
    } else if constexpr (C == KQ_MXFP4) {
      s[0] = b[0];
      q = words8<C>(b + 1 + 8 * (g & 1));
    } else if constexpr (C == KQ_NVFP4) {
      s[0] = b[g >> 1];
      q = words8<C>(b + 4 + 8 * (g >> 1));
    } else {
      static_assert(C == KQ_IQ3_S || C == KQ_IQ2_XXS, "no unit for this codec");
      kq::iq_group<C, false, true>(b, g, grids, q.x, q.y, s[0], db);
    }
  }
  __device__ __forceinline__ void weights(int g, float* o) const {
    const int w = 8 * g, half = w >> 7, si = (w & 127) >> 5;
    const float d = kq::h2f(d_bits), dmin = kq::h2f(m_bits);
    if constexpr (C == KQ_Q8_0) {
      for (int t = 0; t < 8; t++) o[t] = d * sb(q, t);
    } else if constexpr (C == KQ_Q4_0) {
      const uint2 v = less(bits(q, 4 * (g >> 1), 0x0f0f0f0fu), 8);
      for (int t = 0; t < 8; t++) o[t] = d * sb(v, t);
    } else if constexpr (C == KQ_Q4_K || C == KQ_Q5_K) {
      const int j = g >> 2;
      const uint32_t isc = j < 4 ? s[0] & 63 : (s[2] & 15) | ((s[0] >> 6) << 4);
      const uint32_t imn = j < 4 ? s[1] & 63 : (s[2] >> 4) | ((s[1] >> 6) << 4);
      const float sc = d * (float)isc, mn = dmin * (float)imn;
      uint2 v = bits(q, 4 * (j & 1), 0x0f0f0f0fu);
      if constexpr (C == KQ_Q5_K) v = either(v, up(bits(h, j, 0x01010101u), 4));
      for (int t = 0; t < 8; t++) o[t] = sc * ub(v, t) - mn;
    } else if constexpr (C == KQ_Q6_K) {
      const float dsc = d * (float)(int8_t)s[0];
      const uint2 v = less(either(bits(q, 4 * (si >> 1), 0x0f0f0f0fu), up(bits(h, 2 * si, 0x03030303u), 4)), 32);
      for (int t = 0; t < 8; t++) o[t] = dsc * sb(v, t);
    } else if constexpr (C == KQ_Q3_K) {
      const int grp = w >> 6;
      const int sc = (int)((grp & 2 ? s[0] >> 4 : s[0] & 15) | (((s[1] >> (2 * grp)) & 3) << 4));
      const float dl = d * (float)(sc - 32);
      const uint2 v = less(either(bits(q, 2 * si, 0x03030303u), up(bits(h, 4 * half + si, 0x01010101u), 2)), 4);
      for (int t = 0; t < 8; t++) o[t] = dl * sb(v, t);
    } else if constexpr (C == KQ_Q2_K) {
      const float dl = d * (float)(s[0] & 15), ml = dmin * (float)(s[0] >> 4);
      const uint2 v = bits(q, 2 * si, 0x03030303u);
      for (int t = 0; t < 8; t++) o[t] = dl * ub(v, t) - ml;
    } else if constexpr (C == KQ_IQ4_NL || C == KQ_IQ4_XS) {
      constexpr uint64_t lo = 0xF6EADDCFBFAD9881ull, hi = 0x7159453526190D01ull;  // as kq::kv_iq4nl
      float dl = d;
      if constexpr (C == KQ_IQ4_XS) {
        const int ib = g >> 2;
        dl = d * (float)((int)(((s[0] >> (4 * (ib & 1))) & 15) | (((s[1] >> (2 * ib)) & 3) << 4)) - 32);
      }
      const uint2 n = bits(q, C == KQ_IQ4_XS ? 4 * ((g >> 1) & 1) : 4 * (g >> 1), 0x0f0f0f0fu);
      const uint2 v = make_uint2(table4(lo, hi, n.x), table4(lo, hi, n.y));
      for (int t = 0; t < 8; t++) o[t] = dl * sb(v, t);
    } else if constexpr (C == KQ_MXFP4 || C == KQ_NVFP4) {
      constexpr uint64_t lo = 0x0C08060403020100ull, hi = 0xF4F8FAFCFDFEFF00ull;  // kq::kv_mxfp4: magnitudes, their negatives
      const float dl = C == KQ_MXFP4 ? kq::e8m0_half(s[0]) : kq::ue4m3_half(s[0]);
      const uint2 n = bits(q, C == KQ_MXFP4 ? 4 * (g >> 1) : 4 * (g & 1), 0x0f0f0f0fu);
      const uint2 v = make_uint2(table4(lo, hi, n.x), table4(lo, hi, n.y));
      for (int t = 0; t < 8; t++) o[t] = dl * sb(v, t);
    } else {
      for (int j = 0; j < 4; j++) {
        o[j] = db * (float)kq::byte_of(q.x, j) * kq::sgn(s[0], j);
        o[j + 4] = db * (float)kq::byte_of(q.y, j) * kq::sgn(s[0], j + 4);
      }
    }
  }
};

// a wave-uniform pointer, in scalar registers
__device__ __forceinline__ const uint8_t* uniform(const void* p) {
  const uintptr_t v = reinterpret_cast<uintptr_t>(p);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  return reinterpret_cast<const uint8_t*>((uintptr_t)hi << 32 | lo);
}

// the upper half of a's lanes against the lower half of b's
__device__ __forceinline__ void swap_halves(float a, float b, float& x, float& y) {
  const auto v = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
  const uint32_t v0 = v[0], v1 = v[1];
  x = __builtin_bit_cast(float, v0);
  y = __builtin_bit_cast(float, v1);
}

// at most n loads younger than what is waited for
__device__ __forceinline__ void wait_younger(int n) {
  if (n >= 16) vmwait<16>();
  else if (n >= 8) vmwait<8>();
  else if (n >= 4) vmwait<4>();
  else if (n >= 2) vmwait<2>();
  else if (n >= 1) vmwait<1>();
  else vmwait<0>();
}

template <int C, int DT>
__global__ __launch_bounds__(64 * MX_WAVES, 4) void mix_kernel(MixArgs a) {
  constexpr int WPB = kq_geom(C).wpb, BPB = kq_geom(C).bpb, GPB = WPB / 8;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ float part[MX_CLASSES][MX_ROWS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), cls = wave & 3, half = wave >> 2;
  const int S = a.S, K = a.K, N = a.N;
  const int t = __builtin_amdgcn_readfirstlane((int)blockIdx.x / a.tiles);
  const int row0 = ((int)blockIdx.x - t * a.tiles) * MX_ROWS + half * MX_R;  // the wave's rows; N is a multiple of 8
  const uint32_t row_bytes = (uint32_t)(K / WPB) * BPB;
  const int nsl = S > cls ? (S - cls + MX_CLASSES - 1) / MX_CLASSES : 0;  // the wave's slots, at most 8

  if (nsl > 0) {  // uniform over the wave
    // lane u: expert (~0: the shared one, ~1: outside the stack, not added) and score of the wave's slot u
    uint32_t u_expert = ~1u;
    float u_score = 0.f;
    if (lane < nsl) {
      const int s = cls + MX_CLASSES * lane;
      u_expert = s < a.routed ? a.idx[(size_t)t * a.routed + s] : ~0u;
      u_score = a.scores[(size_t)t * S + s];
      if (s < a.routed && u_expert >= (uint32_t)a.E) u_expert = ~1u;
    }
    auto expert = [&](int u) { return (uint32_t)__builtin_amdgcn_readlane((int)u_expert, u); };
    auto score_of = [&](int u) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, u_score), u)); };
    const int region = mix_region(K, (int)row_bytes);
    const uint32_t lds0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_addr(smem));
    const uint8_t* grids = nullptr;
    uint32_t first = 0;  // LDS offset of the first wave's first region
    if constexpr (mix_grid_bytes<C>() > 0) {
      first = MX_WAVES * mix_grid_bytes<C>();
      grids = smem + wave * mix_grid_bytes<C>() - mix_grid_at<C>();
      for (int o = 0; o < mix_grid_bytes<C>(); o += 1024)
        dma16(a.grids + mix_grid_at<C>() + o, 16 * lane, lds0 + wave * mix_grid_bytes<C>() + o);
    }
    const int classes = S < MX_CLASSES ? S : MX_CLASSES, depth = a.depth;
    auto region_of = [&](int u) { return first + (uint32_t)((half * classes + cls) * depth + (u < depth ? u : u % depth)) * region; };
    auto request_x = [&](int u) {
      const uint32_t to = lds0 + region_of(u);
      const uint8_t* xs = uniform(a.x + ((size_t)t * S + cls + MX_CLASSES * u) * K);
      for (int o = 0; o < K / 8; o += 64)
        if (o + lane < K / 8) dma16(xs, 16 * (o + lane), to + 16 * o);
    };
    const int ahead = nsl < depth ? nsl : depth;
    for (int u = 0; u < ahead; u++) request_x(u);
    // The rows of a slot are one run of bytes.  Fetched in 16-byte pieces: from the aligned address in front of it, where the matrix
    // has bytes in front and behind; the matrix's first rows from their start, its last up to their end.
    const uint32_t run = MX_R * row_bytes;
    auto run_of = [&](uint32_t e, uint32_t& lead) -> const uint8_t* {
      const uint8_t* p = (e == ~0u ? a.shexp_w : a.w + (e == ~1u ? 0 : (int64_t)e * a.w_expert_stride)) + (size_t)row0 * row_bytes;
      lead = row0 == 0 ? 0 : row0 + MX_R < N ? (uint32_t)reinterpret_cast<uintptr_t>(p) & 15 : (0u - run) & 15;
      return p - lead;
    };
    auto request_w = [&](int u) {
      const uint32_t to = lds0 + region_of(u);
      uint32_t lead;
      const uint8_t* p = uniform(run_of(expert(u), lead));
      const int pieces = (int)((lead + run + 15) / 16);
      for (int o = 0; o < pieces; o += 64)
        if (o + lane < pieces) dma16(p, 16 * (o + lane), to + 2 * K + 16 * o);
    };
    for (int u = 0; u < ahead; u++) request_w(u);
    const int slot_loads = (int)((run + 1023) / 1024);  // of a slot, or one more

    float tot[MX_R] = {};
    const int ngroups = K / 8, whole = ngroups & ~63, g = lane % GPB;
    for (int u = 0; u < nsl; u++) {
      wait_younger(((u + depth < nsl ? u + depth : nsl) - 1 - u) * slot_loads);
      const uint32_t e = expert(u);
      uint32_t lead;
      run_of(e, lead);
      const uint8_t* xs = smem + region_of(u);
      const uint8_t* ws = xs + 2 * K + lead;
      float v[MX_R] = {};
      // NR of v's rows: group gi of this lane's x times the blocks at w, `pitch` apart
      auto add = [&](const uint8_t* w, uint32_t pitch, int gi, auto& v) __attribute__((always_inline)) {
        constexpr int NR = sizeof(v) / sizeof(v[0]);
        const uint4 xv = *reinterpret_cast<const uint4*>(xs + 16 * gi);
        const uint32_t xw[4] = {xv.x, xv.y, xv.z, xv.w};
        Group<C> grp[NR];
#pragma unroll
        for (int r = 0; r < NR; r++) grp[r].load(w + r * pitch, g, grids);
        __builtin_amdgcn_sched_barrier(0);
        float xf[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          xf[2 * i] = DT == KQ_F16 ? kq::h2f((uint16_t)xw[i]) : __builtin_bit_cast(float, xw[i] << 16);
          xf[2 * i + 1] = DT == KQ_F16 ? kq::h2f((uint16_t)(xw[i] >> 16)) : __builtin_bit_cast(float, xw[i] & 0xffff0000u);
        }
#pragma unroll
        for (int r = 0; r < NR; r++) {
          float wv[8];
          grp[r].weights(g, wv);
#pragma unroll
          for (int i = 0; i < 8; i++) v[r] = fmaf(xf[i], wv[i], v[r]);
        }
      };
      const uint8_t* at = ws + (lane / GPB) * BPB;
      for (int gi = lane; gi < whole; gi += 64, at += 64 / GPB * BPB) add(at, row_bytes, gi, v);
      if (ngroups - whole == 32) {
        // the groups left over, of lanes 0 .. 31: the upper half of the lanes takes them for every other row
        const int l32 = lane & 31;
        const uint8_t* tail = ws + (lane >> 5) * row_bytes + (whole / GPB + l32 / GPB) * BPB;
        float lo[MX_R / 2], hi[MX_R / 2];  // rows 2 p and 2 p + 1: their lanes 0 .. 31, 32 .. 63
#pragma unroll
        for (int p = 0; p < MX_R / 2; p++) swap_halves(v[2 * p], v[2 * p + 1], lo[p], hi[p]);
        add(tail, 2 * row_bytes, whole + l32, lo);
#pragma unroll
        for (int p = 0; p < MX_R / 2; p++) swap_halves(lo[p], hi[p], v[2 * p], v[2 * p + 1]);
      } else if (whole + lane < ngroups) {
        add(at, row_bytes, whole + lane, v);
      }
      if (e != ~1u) {
#pragma unroll
        for (int r = 0; r < MX_R; r++) tot[r] = fmaf(score_of(u), v[r], tot[r]);
      }
      if (u + depth < nsl) {
        lgkm_drain();  // the region has been read
        request_x(u + depth);
        request_w(u + depth);
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
      for (int r = 0; r < MX_R; r++) tot[r] += __shfl_xor(tot[r], off);
    float mine = tot[0], btot = 0.f;  // lane r < 4: row r
#pragma unroll
    for (int r = 1; r < MX_R; r++) mine = lane == r ? tot[r] : mine;
    if (a.bias) {
      for (int u = 0; u < nsl; u++) {
        const uint32_t e = expert(u);
        if (e < (uint32_t)a.E && lane < MX_R) btot = fmaf(score_of(u), a.bias[(size_t)e * N + row0 + lane], btot);
      }
    }
    if (lane < MX_R) part[cls][half * MX_R + lane] = mine + btot;
  } else if (lane < MX_R) {
    part[cls][half * MX_R + lane] = 0.f;
  }
  __syncthreads();
  if (tid < MX_ROWS) {  // of wave 0
    float r = part[0][tid];
    for (int c = 1; c < MX_CLASSES; c++) r += part[c][tid];
    static_cast<uint16_t*>(a.out)[(size_t)t * N + row0 + tid] = DT == KQ_F16 ? kq::f2f16(r) : kq::f2bf16(r);
  }
}

// Regions per wave: all of its slots under way at once where they fit, fewer where that lets a second workgroup onto the CU that
// waits for one (64 experts of 4096 x 1024, top-8, 512 workgroups, us with all under way / with one: q8_0 14.0 / 9.9, q6_k 15.1 / 11.8);
// 0: not even one fits.
int mix_depth(int T, int S, int N, int K, int row_bytes, int grid_bytes) {
  const int waves = MX_HALVES * std::min(S, MX_CLASSES), slots = (S + MX_CLASSES - 1) / MX_CLASSES, each = waves * mix_region(K, row_bytes);
  const int fit = (MX_LDS - MX_WAVES * grid_bytes) / each, shared = (MX_LDS / 2 - MX_WAVES * grid_bytes) / each;
  const bool crowded = (int64_t)T * (N / MX_ROWS) > kq_num_cus();
  return std::min(slots, crowded && shared >= 1 ? shared : fit);
}

template <int C, int DT>
int launch(MixArgs a, int T, hipStream_t s) {
  const int row_bytes = a.K / kq_geom(C).wpb * kq_geom(C).bpb;
  a.depth = mix_depth(T, a.S, a.N, a.K, row_bytes, mix_grid_bytes<C>());
  const size_t lds = MX_WAVES * mix_grid_bytes<C>() + (size_t)MX_HALVES * std::min(a.S, MX_CLASSES) * a.depth * mix_region(a.K, row_bytes);
  auto kern = mix_kernel<C, DT>;
  KQ_SET_MAX_LDS_ONCE((kern), MX_LDS);
  hipLaunchKernelGGL(kern, dim3((unsigned)(T * a.tiles)), dim3(64 * MX_WAVES), lds, s, a);
  KQ_HIP_CHECK(hipGetLastError());
  return KQ_OK;
}

}  // namespace

bool kq_mix_fits(int S, int N, int K, int codec) {
  int grid_bytes = 0;
  switch (codec) {
    case KQ_IQ3_S: grid_bytes = mix_grid_bytes<KQ_IQ3_S>(); break;
    case KQ_IQ2_XXS: grid_bytes = mix_grid_bytes<KQ_IQ2_XXS>(); break;
    case KQ_Q2_K: case KQ_Q3_K: case KQ_Q4_K: case KQ_Q5_K: case KQ_Q6_K: case KQ_IQ4_XS: case KQ_Q8_0: case KQ_IQ4_NL: case KQ_Q4_0:
    case KQ_MXFP4: case KQ_NVFP4:
      break;
    default:
      return false;
  }
  const KqGeom geom = kq_geom(codec);
  if (S < 1 || S > 32 || N < MX_ROWS || N % MX_ROWS || K < geom.wpb || K % geom.wpb || K > MX_LDS / 2) return false;
  return mix_depth(1, S, N, K, K / geom.wpb * geom.bpb, grid_bytes) >= 1;
}

int kq_launch_mix(const void* x, const uint8_t* w, const uint8_t* shexp_w, const uint32_t* idx, const float* scores, const float* bias,
                  void* out, int T, int S, int E, int N, int K, int64_t w_expert_stride, int codec, int dtype, hipStream_t s) {
  if (!kq_mix_fits(S, N, K, codec) || E < 1 || (reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(w) & 1) ||
      (reinterpret_cast<uintptr_t>(shexp_w) & 1) || (w_expert_stride & 1))
    return KQ_ERR_UNSUPPORTED;
  MixArgs a{};
  a.x = static_cast<const uint16_t*>(x);
  a.w = w;
  a.shexp_w = shexp_w;
  a.idx = idx;
  a.scores = scores;
  a.bias = bias;
  a.out = out;
  a.S = S;
  a.routed = shexp_w ? S - 1 : S;
  a.E = E;
  a.N = N;
  a.K = K;
  a.tiles = N / MX_ROWS;
  a.w_expert_stride = w_expert_stride;
  a.grids = kq_device_grids();
  if (!a.grids) return KQ_ERR_HIP;
  switch (codec) {
#define KQ_CASE(c) \
  case c:          \
    return dtype == KQ_F16 ? launch<c, KQ_F16>(a, T, s) : launch<c, KQ_BF16>(a, T, s);
    KQ_CASE(KQ_Q2_K) KQ_CASE(KQ_Q3_K) KQ_CASE(KQ_Q4_K) KQ_CASE(KQ_Q5_K) KQ_CASE(KQ_Q6_K) KQ_CASE(KQ_IQ4_XS)
    KQ_CASE(KQ_IQ3_S) KQ_CASE(KQ_IQ2_XXS) KQ_CASE(KQ_Q8_0) KQ_CASE(KQ_IQ4_NL) KQ_CASE(KQ_Q4_0) KQ_CASE(KQ_MXFP4)
    KQ_CASE(KQ_NVFP4)
#undef KQ_CASE
  }
  return KQ_ERR_UNSUPPORTED;
}
