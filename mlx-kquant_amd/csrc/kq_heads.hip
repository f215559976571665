// gather_qmm of short contractions over few rows per expert, every codec, one launch: y[p] = x[row(p)] . W[expert(p)]^T with
// K of one or two steps of 256 (absorbed-MLA projections: 128 heads of 128 x 512, a few sequences).
//
// What bounds it: a chain of latencies.  The whole product is a microsecond of work, and the kernels that had these calls
// (a prepass that sorts the pairs and converts activations, then a kernel over the sorted segments) went through the memory
// six times one after the other: list, counts, segment, order, activations and weights, sums.  Here a workgroup knows its
// expert and its weight rows from its index, so the wire bytes travel while it looks for the expert's entries in the id list
// (a list of at most 1024 ids, read by every workgroup at once); then one load of the activations, which it converts itself.
//   * Workgroup = 4 waves; wave = one 32-row weight tile x one 256-weight step (mid_step of kq_mid.h, wire bytes through LDS),
//     so a workgroup covers four tiles or two; the steps of a tile meet in LDS at the end.
//   * Activations: up to 32 rows at a time as f16 fragments in LDS under a power of two per row and step.  A row with a nonzero
//     value that this does not hold (2^-31 of the step's largest, bf16), or with an infinity, is done in f32 instead.
//     More rows than 32 are further rounds, of other workgroups (kq_entries.h): 1024 entries of 8 rows on one of 64 experts
//     243 -> 31 us against rounds in series on the expert's own, 512 of one row on one of 128 100 -> 18.4, even shares 6.7 -> 6.7 (q8_0).
// 128 heads of 128 x 512, 4 / 16 / 32 rows each, us: q8_0 12.6 / 14.6 / 22.4 -> 6.7 / 7.7 / 9.8, q4_k 10.3 / 11.7 / 15.4 -> 6.3 / 7.4 / 10.0,
// q6_k 11.9 / 12.9 / 16.9 -> 6.9 / 7.8 / 9.8, the empty launch 2.4; 64 / 128 rows q8_0 28 / 61 -> 12.7 / 23.0, q4_k 22 / 45 -> 13.1 / 24.1.
#include <algorithm>

#include "kq_entries.h"
#include "kq_mid.h"

namespace {

using namespace kqmid;
using kqentries::MAX_ENTRIES;

constexpr int HD_WAVES = 4, HD_THREADS = 64 * HD_WAVES, HD_AHEAD = 4, HD_STEPS = 2;

struct HeadArgs {
  const uint16_t* x;
  const uint8_t* w;
  uint16_t* y;
  const uint32_t* lhs;
  const uint32_t* rhs;
  const uint8_t* grids;
  int B, M, N, K;
  int64_t x_batch_stride, w_expert_stride;
};

// The rows of a round that f16 does not hold, in f32 on the reference-order weights from global memory (the order of the sums
// aside, the arithmetic of the kernels that go entry by entry).  Rare, so small code rather than speed: a weight is decoded once
// for eight rows.
template <int C, int DT>
__device__ __forceinline__ void wide_rows_f32(const HeadArgs& a, uint32_t expert, uint32_t wide, const int64_t* x_off,
                                              const int64_t* y_row, int tid) {
  using G = MidGeom<C>;
  const int lg = a.K > CK_STEP ? 2 : 1, parts = 1 << lg;  // threads per weight row: 32 HD_WAVES / steps rows a workgroup
  const int part = tid & (parts - 1), n = (HD_THREADS >> lg) * (int)blockIdx.x + (tid >> lg);
  const bool live = n < a.N;
  const uint8_t* w = a.w + (size_t)expert * (size_t)a.w_expert_stride + (size_t)(live ? n : 0) * (size_t)(a.K / G::WPB) * G::BPB;
#pragma unroll 1
  for (int r0 = 0; r0 < 32; r0 += 8) {
    if (!((wide >> r0) & 0xff)) continue;  // uniform
    float sum[8] = {};
#pragma unroll 1
    for (int g = part; g < a.K / 8; g += parts) {
      float f[8];
      kq::decode8<C>(w + (size_t)(8 * g / G::WPB) * G::BPB, 8 * g % G::WPB / 8, a.grids, f);
#pragma unroll
      for (int r = 0; r < 8; r++) {
        if (!((wide >> (r0 + r)) & 1)) continue;  // uniform
        const u32x4 v = *reinterpret_cast<const u32x4*>(a.x + x_off[r0 + r] + 8 * g);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const uint16_t lo = (uint16_t)(v[e] & 0xffffu), hi = (uint16_t)(v[e] >> 16);
          sum[r] = fmaf(DT == KQ_BF16 ? kq::bf162f(lo) : kq::h2f(lo), f[2 * e], sum[r]);
          sum[r] = fmaf(DT == KQ_BF16 ? kq::bf162f(hi) : kq::h2f(hi), f[2 * e + 1], sum[r]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 8; r++) {
      if (!((wide >> (r0 + r)) & 1)) continue;
      for (int m = 1; m < parts; m <<= 1) sum[r] += __shfl_xor(sum[r], m);
      if (live && part == 0) a.y[(size_t)y_row[r0 + r] * a.N + n] = DT == KQ_F16 ? kq::f2f16(sum[r]) : kq::f2bf16(sum[r]);
    }
  }
}

template <int C, int DT>
__global__ __launch_bounds__(HD_THREADS, 2) void heads_kernel(HeadArgs a) {
  using G = MidGeom<C>;
  constexpr int SLOT = mid_slot_bytes<C>();
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  static_assert(HD_THREADS == kqentries::THREADS, "the search of the id list");
  __shared__ kqentries::Places places;
  __shared__ kqentries::Share share;
  __shared__ float xs[HD_STEPS][32];
  __shared__ int64_t x_off[32], y_row[32];
  __shared__ uint32_t wide_rows;  // rows of the round that f16 under a power of two does not hold, by bit
  const int N = a.N, K = a.K, nsteps = K / CK_STEP;
  uint8_t* slots = smem + mid_table_bytes<C>();
  uint8_t* frags = slots + HD_WAVES * SLOT;  // [step][fragment][lane][16]; the sums of the waves afterwards
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, kg = lane >> 5;
  uint32_t expert = blockIdx.y;

  // ---- this wave's wire bytes
  const int tpw = HD_WAVES / nsteps, t = wave / nsteps, st = wave - t * nsteps;
  const int row0 = 32 * ((int)blockIdx.x * tpw + t), nrows = N - row0 < 32 ? N - row0 : 32;
  const bool live = t < tpw && nrows > 0;
  auto request = [&]() {
    if (!live) return;
    const uint32_t row_bytes = (uint32_t)(K / G::WPB) * G::BPB;
    const uint8_t* base = a.w + (size_t)expert * (size_t)a.w_expert_stride + (size_t)row0 * row_bytes + (size_t)st * G::BYTES;
    const uint32_t l0 = lds_addr(slots + wave * SLOT);
    StaticFor<G::LOADS>::run([&](auto tc) {
      constexpr int T = decltype(tc)::value;
      const int i = lane + 64 * T, r = i / G::LP, p = i - r * G::LP;
      const int off = 16 * p < G::BYTES - 16 ? 16 * p : G::BYTES - 16;
      if (r < nrows) dma16(base, (uint32_t)r * row_bytes + (uint32_t)off, l0 + 1024 * T);
    });
  };
  kqfrag::KMasks masks;
  masks.init<C>();
  Tables tabs{smem, smem, 2};
  uint8_t* spread = smem + CodeGeom<C>::GROUPED_GRID_BYTES;
  if constexpr (mid_table_bytes<C>() > 0) tabs = Tables{CodeGeom<C>::PAIR_LUT ? smem + 4 * l32 : smem, spread, 7};

  // largest magnitude over the lane's 32, as the half's bits
  auto magnitude = [](u32x4 v) {
    u16x2 top = __builtin_bit_cast(u16x2, v[0] & 0x7fff7fffu);
#pragma unroll
    for (int e = 1; e < 4; e++) top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, v[e] & 0x7fff7fffu));
    int m = top[0] > top[1] ? top[0] : top[1];
    m = max(m, __builtin_amdgcn_update_dpp(0, m, 0xB1, 0xf, 0xf, true));   // quad_perm [1,0,3,2]
    m = max(m, __builtin_amdgcn_update_dpp(0, m, 0x4E, 0xf, 0xf, true));   // quad_perm [2,3,0,1]
    m = max(m, __builtin_amdgcn_update_dpp(0, m, 0x141, 0xf, 0xf, true));  // row_half_mirror
    m = max(m, __builtin_amdgcn_update_dpp(0, m, 0x140, 0xf, 0xf, true));  // row_mirror
    return (uint32_t)max(m, __shfl_xor(m, 16));
  };
  auto lo_f = [](uint32_t v) { return DT == KQ_BF16 ? __builtin_bit_cast(float, v << 16) : kq::h2f((uint16_t)(v & 0xffffu)); };
  auto hi_f = [](uint32_t v) { return DT == KQ_BF16 ? __builtin_bit_cast(float, v & 0xffff0000u) : kq::h2f((uint16_t)(v >> 16)); };
  uint32_t* entries = reinterpret_cast<uint32_t*>(frags + nsteps * (G::NF * 1024));  // per expert
  const int E = gridDim.y, Z = gridDim.z;
  auto barrier = [] { lds_barrier(); };
  auto round = [&](int r0, int rows, auto own) __attribute__((always_inline)) {  // rows r0 ... of the expert whose places and wire bytes are in LDS or on the way
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    lds_barrier();
    const int here = rows - r0 < 32 ? rows - r0 : 32;
    if (tid < here) {
      const int place = (r0 + tid) / a.M, m = r0 + tid - place * a.M;
      x_off[tid] = (int64_t)places.lhs_of[place] * a.x_batch_stride + (int64_t)m * K;
      y_row[tid] = (int64_t)places.entry_of[place] * a.M + m;
    }
    if (tid == 0) wide_rows = 0;
    lds_barrier();
    // ---- activations: 32 lanes per (row, step), eight rows of a step at a time, the loads of four such blocks in flight
    const int pc = tid & 31, rblocks = (here + 7) / 8, nblocks = rblocks * nsteps;
    const int per_block = rblocks == 1 ? 32 : rblocks == 2 ? 16 : rblocks == 3 ? 11 : 8;  // b / rblocks = b per_block / 32
    uint32_t lost_rows = 0;  // of the lane's, by bit
    for (int b0 = 0; b0 < nblocks; b0 += HD_AHEAD) {
      u32x4 v[HD_AHEAD];
#pragma unroll
      for (int u = 0; u < HD_AHEAD; u++) {
        const int b = b0 + u < nblocks ? b0 + u : nblocks - 1, s = b * per_block >> 5;
        const int row = 8 * (b - s * rblocks) + (tid >> 5);
        v[u] = *reinterpret_cast<const u32x4*>(a.x + x_off[row < here ? row : here - 1] + CK_STEP * s + 8 * pc);
      }
      if constexpr (decltype(own)::value) {
        if (b0 == 0) kqentries::note_left<32>(a.M, E, Z, tid, entries, share);
      }
#pragma unroll
      for (int u = 0; u < HD_AHEAD; u++) {
        const int b = b0 + u, s = b * per_block >> 5, row = 8 * (b - s * rblocks) + (tid >> 5);
        if (b >= nblocks) break;  // uniform
        const uint32_t mag = magnitude(v[u]);
        const float amax = DT == KQ_BF16 ? __builtin_bit_cast(float, mag << 16) : kq::h2f((uint16_t)mag);
        float inv = 1.f, scale = 1.f;
        const uint32_t eb = (__builtin_bit_cast(uint32_t, amax) >> 23) & 0xff;
        if (eb != 0 && eb != 0xff) {  // the largest magnitude into [2^14, 2^15); f16 rows only upwards
          int e = (int)eb - 127 - 14;
          if (e < -100) e = -100;
          if (DT == KQ_F16 && e > 0) e = 0;
          scale = __builtin_bit_cast(float, (uint32_t)(127 + e) << 23);
          inv = __builtin_bit_cast(float, (uint32_t)(127 - e) << 23);
        }
        // values below 2^-17 in the step's unit lose bits (RowRange of kq_mma.h); an infinity leaves the others unscaled
        bool lost = eb == 0xff;
        if constexpr (DT == KQ_BF16) {
          const uint32_t cut = ((__builtin_bit_cast(uint32_t, scale) >> 23) - 17) << 7;
          u16x2 low = {0xffff, 0xffff};
#pragma unroll
          for (int e = 0; e < 4; e++)
            low = __builtin_elementwise_min(low, (u16x2)(__builtin_bit_cast(u16x2, v[u][e] & 0x7fff7fffu) - (uint16_t)1));
          lost |= (uint32_t)(low[0] < low[1] ? low[0] : low[1]) < cut - 1;
        }
        _Float16 h[8];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          h[2 * e] = (_Float16)(lo_f(v[u][e]) * inv);
          h[2 * e + 1] = (_Float16)(hi_f(v[u][e]) * inv);
        }
        if (row >= here) continue;  // 32 lanes at a time
        lost_rows |= lost ? 1u << row : 0u;
        store_frags<G::ORD, G::NSUM, true>(frags + s * (G::NF * 1024) + 16 * row, pc, h, row);
        if (pc == 0) xs[s][row] = scale;
      }
    }
    if (__builtin_expect(lost_rows != 0, 0)) atomicOr(&wide_rows, lost_rows);
    vmwait<0>();  // the wire bytes
    lds_barrier();
    const uint32_t rows_here = here == 32 ? ~0u : (1u << here) - 1, wide = __builtin_amdgcn_readfirstlane(wide_rows) & rows_here;
    f32x16 acc = f32x16{0};
    if (live) {
      // places past the last row hold whatever lies there: their results are not stored
      f16x8 f[G::NF];
#pragma unroll
      for (int j = 0; j < G::NF; j++)
        f[j] = *reinterpret_cast<const f16x8*>(frags + (st * G::NF + j) * 1024 + 512 * kg +
                                               16 * (j < 16 ? l32 ^ (2 * j + kg) : l32));
      mid_step<C>(slots + wave * SLOT + l32 * G::LROW, kg, f, tabs, masks, CK_STEP, acc);
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const float4 v = *reinterpret_cast<const float4*>(&xs[st][8 * q + 4 * kg]);
        acc[4 * q + 0] *= v.x;
        acc[4 * q + 1] *= v.y;
        acc[4 * q + 2] *= v.z;
        acc[4 * q + 3] *= v.w;
      }
    }
    if (nsteps > 1) {  // the second step of a tile to its first
      float* sums = reinterpret_cast<float*>(frags) + t * 1024 + lane;
      lds_barrier();  // the fragments have been read
      if (live && st > 0) {
#pragma unroll
        for (int i = 0; i < 16; i++) sums[64 * i] = acc[i];
      }
      lds_barrier();
      if (live && st == 0) {
#pragma unroll
        for (int i = 0; i < 16; i++) acc[i] += sums[64 * i];
      }
    }
    if (live && st == 0 && l32 < nrows) {
      const uint32_t mine = (rows_here & ~wide) >> (4 * kg);
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int r0 = 8 * (i >> 2) + (i & 3);
        if ((mine >> r0) & 1) a.y[(size_t)y_row[r0 + 4 * kg] * N + row0 + l32] = DT == KQ_F16 ? kq::f2f16(acc[i]) : kq::f2bf16(acc[i]);
      }
    }
    if (__builtin_expect(wide != 0, 0)) wide_rows_f32<C, DT>(a, expert, wide, x_off, y_row, tid);
  };
  // A round of the workgroup's own expert, if it has one for it, then one that another expert leaves over.  The second is written
  // out: a loop around both kept the addresses of the first alive in it (172 registers where this takes 127, even shares 10 % longer).
  if (blockIdx.z == 0) request();
  const int r0 = 32 * blockIdx.z;
  int own_rows;
  {
    kqentries::Ids ids;
    ids.load(a.rhs, a.lhs, a.B, tid);
    if constexpr (mid_table_bytes<C>() > 0) build_tables<C, HD_THREADS, true>(smem, spread, a.grids, tid);
    own_rows = kqentries::find_and_count(ids, expert, a.B, E, tid, wave, places, entries, share, barrier) * a.M;
  }
  if (__builtin_expect(r0 < own_rows, 1)) {  // uniform
    if (blockIdx.z != 0) request();
    round(r0, own_rows, std::true_type{});
    if (__builtin_expect(!share.left || !kqentries::shares_rounds<32>(own_rows, a.B, a.M, E, Z), 1)) return;
  } else {
    vmwait<0>();  // nothing may be on its way into LDS when the workgroup ends
    lds_barrier();
    kqentries::note_left<32>(a.M, E, Z, tid, entries, share);
    lds_barrier();
    if (!share.left) return;
  }
  const uint32_t next = kqentries::share_rounds<32>(a.B, a.M, E, Z, blockIdx.y, blockIdx.z, tid, entries, share, barrier);
  if (next == kqentries::NO_ROUND) return;
  expert = next & (kqentries::MAX_EXPERTS - 1);
  request();
  int cold_tid = tid;
  asm volatile("" : "+v"(cold_tid));
  kqentries::Ids ids;
  ids.load(a.rhs, a.lhs, a.B, cold_tid);
  const int rows = ids.find(expert, a.B, cold_tid, wave, places, barrier) * a.M;
  round(32 * (int)(next >> kqentries::EXPERT_BITS), rows, std::false_type{});
}

template <int C, int DT>
int launch_heads(const HeadArgs& a, int E, hipStream_t s) {
  using G = MidGeom<C>;
  const int nsteps = a.K / CK_STEP, cols = 32 * (HD_WAVES / nsteps);
  constexpr size_t fixed = (size_t)mid_table_bytes<C>() + HD_WAVES * mid_slot_bytes<C>();
  static_assert(fixed + HD_STEPS * G::NF * 1024 + kqentries::count_bytes(kqentries::MAX_EXPERTS) + 9 * 1024 <= 160 * 1024, "LDS of a CU");
  // workgroups for the rounds of an average expert, and for more in long lists of random ids: those without one leave early
  const int64_t P = (int64_t)a.B * a.M;
  const int z = (int)std::min<int64_t>(8, std::max<int64_t>(1 + P / 2048, (P + 32 * E - 1) / (32 * E)));
  const size_t lds = fixed + (size_t)nsteps * G::NF * 1024 + kqentries::count_bytes(E);
  auto kern = heads_kernel<C, DT>;
  KQ_SET_MAX_LDS_ONCE((kern), fixed + HD_STEPS * G::NF * 1024 + kqentries::count_bytes(kqentries::MAX_EXPERTS));
  hipLaunchKernelGGL(kern, dim3((a.N + cols - 1) / cols, E, z), dim3(HD_THREADS), lds, s, a);
  KQ_HIP_CHECK(hipGetLastError());
  return KQ_OK;
}

}  // namespace

static bool heads_shape(int B, int M, int E, int N, int K, int codec) {
  if (codec < 0 || codec >= KQ_NUM_CODECS || B <= 0 || M <= 0 || E <= 0 || E > kqentries::MAX_EXPERTS || N <= 0 || B > MAX_ENTRIES) return false;
  if (K <= 0 || K % CK_STEP || K > HD_STEPS * CK_STEP || K % kq_geom(codec).wpb) return false;
  const int64_t row_bytes = (int64_t)(K / kq_geom(codec).wpb) * kq_geom(codec).bpb;
  if (row_bytes & 1) return false;  // the direct-to-LDS loads take 2-byte aligned addresses
  // Up to 16 rows the streamed kernel goes entry by entry (16 heads of 64 x 512: 3.4 us q4_k, 4.1 q8_0; here 4.4, 5.0).
  // Stacks of more weights than a few per lane and long rows are no matter of latency, and a workgroup of one tile converts its
  // activations for few products: 1000 random pairs, here / the grouped kernels, us: 128 x 2048 x 768 q4_k 109 / 37, q8_0 199 / 62,
  // 128 x 768 x 1024 86 / 24, 86 / 40; but 16 x 512 x 512 14 / 12, 14 / 17, 8 x 4096 x 256 19 / 16, 20 / 29, 128 x 128 x 512 7.8 / 11.2,
  // 8.1 / 13.9.  256 rows on each expert: 128 x 128 x 512 43 / 78, 41 / 108, 16 x 512 x 512 20 / 23, 22 / 30.
  const int64_t P = (int64_t)B * M;
  if ((int64_t)E * N * K > (int64_t)1 << 24 || P <= 16 || P > 256 * (int64_t)E) return false;
  return P <= 32 * (int64_t)E || N <= 256 || !kq_moe_grouped_supported((int)P, E, N, K, codec);
}

bool kq_heads_takes(const void* x, const void* w, int B, int M, int E, int N, int K, int64_t x_batch_stride, int64_t w_expert_stride,
                    int codec) {
  return heads_shape(B, M, E, N, K, codec) && !(reinterpret_cast<uintptr_t>(x) & 15) && !(x_batch_stride & 7) &&
         !(reinterpret_cast<uintptr_t>(w) & 1) && !(w_expert_stride & 1);
}

// KQ_ERR_UNSUPPORTED: nothing launched
int kq_launch_heads(const void* x, const uint8_t* w, const uint32_t* lhs, const uint32_t* rhs, void* out, int B, int M, int E,
                    int N, int K, int64_t x_batch_stride, int64_t w_expert_stride, int codec, int dtype, hipStream_t s) {
  if (!kq_heads_takes(x, w, B, M, E, N, K, x_batch_stride, w_expert_stride, codec)) return KQ_ERR_UNSUPPORTED;
  HeadArgs a{static_cast<const uint16_t*>(x), w, static_cast<uint16_t*>(out), lhs, rhs, kq_device_grids(), B, M, N, K,
             x_batch_stride, w_expert_stride};
  if (!a.grids) return KQ_ERR_HIP;
  switch (codec) {
#define KQ_CASE(c) \
  case c:          \
    return dtype == KQ_F16 ? launch_heads<c, KQ_F16>(a, E, s) : launch_heads<c, KQ_BF16>(a, E, s);
    KQ_CASE(KQ_Q2_K) KQ_CASE(KQ_Q3_K) KQ_CASE(KQ_Q4_K) KQ_CASE(KQ_Q5_K) KQ_CASE(KQ_Q6_K) KQ_CASE(KQ_Q4_0) KQ_CASE(KQ_Q4_1)
    KQ_CASE(KQ_Q5_0) KQ_CASE(KQ_Q5_1) KQ_CASE(KQ_Q8_0) KQ_CASE(KQ_IQ4_NL) KQ_CASE(KQ_IQ4_XS) KQ_CASE(KQ_IQ3_S)
    KQ_CASE(KQ_IQ3_XXS) KQ_CASE(KQ_IQ2_XXS) KQ_CASE(KQ_IQ2_XS) KQ_CASE(KQ_IQ2_S) KQ_CASE(KQ_IQ1_S) KQ_CASE(KQ_IQ1_M)
    KQ_CASE(KQ_MXFP4) KQ_CASE(KQ_NVFP4)
#undef KQ_CASE
  }
  return KQ_ERR_UNSUPPORTED;
}
