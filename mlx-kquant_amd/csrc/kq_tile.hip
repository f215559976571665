// Matmul of 33 rows and more, every codec: y[M,N] = x[M,K] . W^T on tiles of 128 weight rows x up to 128 activation rows.
//
// What bounds it: the streamed kernel of kq_mid.hip decodes a weight once per 32 activation rows and every wave reads its
// activation fragments from L2 for itself (17 KB per 4.6 KB of q4_k wire, 25 B a cycle and CU, which is what L2 gives).
// Here a decoded fragment feeds NB = 2 ... 4 matrix instructions and four waves share the activations through LDS:
//   * Workgroup = 8 waves: four own 32 weight rows each, times two that take the 256-weight steps in turn; the two halves'
//     sums meet in LDS at the end.  Tiles of 128 weight rows leave enough of them to fill the chip from a few hundred
//     activation rows on, and a workgroup's sums are 16 KB per block of 32 rows when K is cut over the grid.
//   * Activations (f16 in matrix-operand order, the prepass of kq_mid.hip) travel L2 -> LDS with direct-to-LDS loads in
//     quarter steps of 64 weights, DEPTH buffers per half, one barrier per quarter step.
//   * Wire bytes of a wave's own rows go to a private LDS slot one step ahead and from there into registers at the start of
//     the step, which frees the slot for the next one.
//   * Whole rounds of tiles run uncut; the K of the tiles left over is cut into ranges that fill the chip once more, and the
//     workgroup that finishes last adds the ranges' sums in order (as finish_tile of kq_mid.hip).
//   * A block of 32 rows that holds a row of wide range is done again by wide_step before its sums are stored.
// Measured, us with the prepass (before, on the kernel that had the call): iq4_xs 333 rows 14336 x 4096 89 (127), 4096 x 4096
// 39 (47), 768 rows 4096 x 14336 152 (474); q6_k 333 rows 4096 x 14336 108 (163); q4_k 1024 rows 4096 x 4096 57 (65).  On q4_k 1024
// rows of 28672 x 8192 a pair of steps of all eight waves takes 5.2 us = 0.8 PFLOP/s; taking out the
// activation loads, the wire loads, the LDS reads or the decode (timing only) gives 14, 7, 4 and 3 %: the stages add up.  A
// workgroup's fixed cost is 8 us at NB = 4 (11 with 2-byte stores and row scales loaded between them).
// Precision: exact f16 terms of the weights, f32 sums per scale block and of those.  Results that are not the correctly rounded ones,
// bf16, 1024 rows of 2048 x 4096 N(0, 1) activations (any-codec kernel / tall tiles that had the calls): q3_k 0.02 % (0.23 / -), q4_1 and q5_1 0.025 (0.031 /
// 0.049), q2_k 0.013 (0.034), mxfp4 0.006 (0.006 / 0.007), nvfp4 0.012 (0.010 / 0.013); q8_0, iq4_xs, iq3_s, iq1_m 0.01 - 0.02 (0.4 - 0.5).  A minimum's
// products cancel against the codes' where activations have a mean: of 0.3, q4_1 / q5_1 0.07 (0.03 / 0.05), q2_k 0.04 (0.03).  Activations
// are f16 under their row's power of two; of a bf16 row that does not count as wide one value in 4096 may have lost bits below 2^-31 of
// its largest (RowRange of kq_mma.h; N(0, 1): one in 10^9), which the any-codec kernel keeps.
#include <algorithm>
#include <cmath>

#include "kq_tile.h"

namespace {

using namespace kqmid;
using namespace kqtile;

constexpr int TL_NW = 4, TL_KS = 2, TL_WAVES = TL_NW * TL_KS, TL_TN = 32 * TL_NW;

struct TileArgs {
  const uint16_t* x;
  const uint8_t* xf;
  const float* rs;
  const uint8_t* w;
  uint16_t* y;
  const uint8_t* grids;
  int M, N, K, dtype;
  int vec;                      // rows of y are whole 16-byte pieces
  int mblocks, mtiles, ntiles;
  int whole;                    // tiles that one workgroup does alone; behind them come `splits` workgroups per tile
  int splits, steps_per_split;
  float* part;    // the ranges' sums of the cut tiles, [item][NB * 4][1024] f32
  int* counters;  // and the arrivals per cut tile, zero at the start
};

template <int C, int NB>
struct TileLds {
  using G = MidGeom<C>;
  static constexpr int TABLES = mid_table_bytes<C>(), WSLOT = 32 * G::LROW, WIRE = TL_WAVES * WSLOT;
  static constexpr int QUARTER = NB * 4096, SUMS = TL_KS * NB * G::NSUM * 1024;
  static constexpr int FIXED = TABLES + WIRE + SUMS + 64;
  static constexpr int DEPTH = FIXED + 3 * TL_KS * QUARTER <= 160 * 1024 ? 3 : 2;
  static constexpr int BYTES = FIXED + DEPTH * TL_KS * QUARTER;
  static_assert(BYTES <= 160 * 1024, "the tile does not fit the LDS of a CU");
  static_assert(WIRE + DEPTH * TL_KS * QUARTER >= NB * TL_NW * 4096, "room for the halves' sums");
};

template <int C, int NB>
__global__ __launch_bounds__(64 * TL_WAVES, 1) void tile_kernel(TileArgs a) {
  using G = MidGeom<C>;
  using L = TileLds<C, NB>;
  constexpr int D = L::DEPTH, NT = 64 * TL_WAVES, PARTS = k_quant<C>() ? 1 : row_parts<C>();
  constexpr int UW = PARTS == 2 ? 2 : 0;  // the quarter in which the wire slot is free for the next step
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  uint8_t* wire = smem + L::TABLES;
  uint8_t* acts = wire + L::WIRE;
  uint8_t* sums = acts + D * TL_KS * L::QUARTER;
  int* last = reinterpret_cast<int*>(sums + L::SUMS);
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, kg = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), grp = wave >> 2, nw = wave & 3;
  const int N = a.N, K = a.K, nsteps = K / CK_STEP;
  const uint32_t row_bytes = (uint32_t)(K / G::WPB) * G::BPB;

  // item -> tile and range of steps.  Tiles run over (group of 8 column tiles, row tile, column tile of the group):
  // workgroups go to the 8 XCDs in turn, so the row tiles of a column meet in one L2.
  const bool cut = (int)blockIdx.x >= a.whole;
  const int q = (int)blockIdx.x - a.whole;
  const int range = cut ? __builtin_amdgcn_readfirstlane(q % a.splits) : 0;
  const int t = cut ? a.whole + __builtin_amdgcn_readfirstlane(q / a.splits) : (int)blockIdx.x;
  const int s0 = cut ? range * a.steps_per_split : 0;
  const int s1 = cut && s0 + a.steps_per_split < nsteps ? s0 + a.steps_per_split : nsteps;
  const int g8 = __builtin_amdgcn_readfirstlane(t / (8 * a.mtiles)), rem = t - g8 * 8 * a.mtiles;
  const int width = a.ntiles - 8 * g8 < 8 ? a.ntiles - 8 * g8 : 8, rowt = __builtin_amdgcn_readfirstlane(rem / width);
  const int mb0 = rowt * NB, row0 = (8 * g8 + rem - rowt * width) * TL_TN + 32 * nw;  // row0: the wave's weight rows
  const int rowb = row0 < N ? row0 : N - 1;

  const uint32_t wire_lds = lds_addr(wire) + wave * L::WSLOT;
  const uint32_t acts_lds = lds_addr(acts) + grp * D * L::QUARTER + nw * 1024;
  const uint32_t sums_lds = lds_addr(sums) + grp * NB * G::NSUM * 1024;
  const uint8_t* wbase = a.w + (size_t)rowb * row_bytes;
  uint32_t voff[G::LOADS];
  StaticFor<G::LOADS>::run([&](auto tc) __attribute__((always_inline)) {
    constexpr int T = decltype(tc)::value;
    const int i = lane + 64 * T, r = i / G::LP, p = i - r * G::LP;
    const int off = 16 * p < G::BYTES - 16 ? 16 * p : G::BYTES - 16;
    voff[T] = (uint32_t)(rowb + r < N ? r : N - 1 - rowb) * row_bytes + (uint32_t)off;
  });
  auto request_wire = [&](int st) __attribute__((always_inline)) {
    StaticFor<G::LOADS>::run([&](auto tc) __attribute__((always_inline)) {
      constexpr int T = decltype(tc)::value;
      if (64 * T + lane < 32 * G::LP) dma16(wbase + (size_t)st * G::BYTES, voff[T], wire_lds + 1024 * T);
    });
  };
  // fragment 4 u + nw of every block (blocks past the last one: that one again), with quarter 3 the sums of block nw
  auto request_acts = [&](int st, int u, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
      const int mb = mb0 + nb < a.mblocks ? mb0 + nb : a.mblocks - 1;
      dma16(a.xf + (((size_t)mb * nsteps + st) * G::NF + 4 * u + nw) * 1024, 16 * lane, acts_lds + buf * L::QUARTER + nb * 4096);
    }
    if constexpr (G::NSUM > 0) {
      if (u == 3) {
        const int nb = nw < NB ? nw : NB - 1, mb = mb0 + nb < a.mblocks ? mb0 + nb : a.mblocks - 1;
#pragma unroll
        for (int s = 0; s < G::NSUM; s++)
          dma16(a.xf + (((size_t)mb * nsteps + st) * G::NF + 16 + s) * 1024, 16 * lane, sums_lds + (nb * G::NSUM + s) * 1024);
      }
    }
  };

  kqfrag::KMasks masks;
  masks.init<C>();
  Tables tabs{smem, smem, 2};
  int st = s0 + grp;
  if (st < s1) {
    request_wire(st);
#pragma unroll
    for (int u = 0; u < D - 1; u++) request_acts(st, u, u);
  }
  if constexpr (L::TABLES > 0) {
    uint8_t* spread = smem + CodeGeom<C>::GROUPED_GRID_BYTES;
    build_tables<C, NT, true>(smem, spread, a.grids, tid);
    tabs = Tables{CodeGeom<C>::PAIR_LUT ? smem + 4 * l32 : smem, spread, 7};
  }

  f32x16 acc[NB], part[NB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++) acc[nb] = part[nb] = f32x16{0};
  const uint8_t* wrow = wire + wave * L::WSLOT + l32 * G::LROW;
  const uint8_t* arow = acts + grp * D * L::QUARTER + 16 * lane;
  const uint8_t* srow = sums + grp * NB * G::NSUM * 1024 + 16 * lane;
  int buf = 0;
  // Both halves go through the same number of steps; one may have nothing in the last.  Loads of a wave land in order: the
  // counts are those issued behind the quarter waited for.
  for (int it = s0; it < s1; it += TL_KS, st += TL_KS) {
    const bool have = st < s1, more = st + TL_KS < s1;
    f16x8 mins = {};
    float fold = 0.f;
    auto quarter = [&](auto uc, const auto& row, auto&& at_start) __attribute__((always_inline)) {
      constexpr int U = decltype(uc)::value;
      constexpr int LATER = D == 2 || (U == 3) ? 0 : U == 2 ? NB + G::NSUM : NB;  // of this step's activations
      constexpr int NEXT = (D == 3 && U == 3 ? NB : 0) + ((UW == 0 && (U == 1 || (D == 3 && U == 2))) || (UW == 2 && U == 3) ? G::LOADS : 0);
      if (more) vmwait<LATER + NEXT>();
      else vmwait<LATER>();
      lds_barrier();
      if (!have) return;
      const int nbuf = buf + D - 1 < D ? buf + D - 1 : buf - 1;
      if constexpr (U + D - 1 < 4) request_acts(st, U + D - 1, nbuf);
      else if (more) request_acts(st + TL_KS, U + D - 5, nbuf);
      at_start();
      const uint8_t* act = arow + buf * L::QUARTER;
      tile_quarter<C, NB, U>(row, [&](int nb, int j) __attribute__((always_inline)) { return act + nb * 4096 + j * 1024; }, srow, kg, tabs,
                             masks, mins, fold, part, acc);
      buf = buf + 1 < D ? buf + 1 : 0;
    };
    auto nothing = [] {};
    auto refill = [&] {
      lgkm_drain();
      if (more) request_wire(st + TL_KS);
    };
    if constexpr (k_quant<C>()) {
      kqfrag::KRow<C> row;
      quarter(std::integral_constant<int, 0>{}, row, [&] { row.load(wrow, kg); refill(); });
      quarter(std::integral_constant<int, 1>{}, row, nothing);
      quarter(std::integral_constant<int, 2>{}, row, nothing);
      quarter(std::integral_constant<int, 3>{}, row, nothing);
    } else if constexpr (PARTS == 1) {
      RowPart<C, 0> row;
      quarter(std::integral_constant<int, 0>{}, row, [&] { row.load(wrow); refill(); });
      quarter(std::integral_constant<int, 1>{}, row, nothing);
      quarter(std::integral_constant<int, 2>{}, row, nothing);
      quarter(std::integral_constant<int, 3>{}, row, nothing);
    } else {
      RowPart<C, 0> r0;
      quarter(std::integral_constant<int, 0>{}, r0, [&] { r0.load(wrow); });
      quarter(std::integral_constant<int, 1>{}, r0, nothing);
      RowPart<C, PARTS - 1> r1;
      quarter(std::integral_constant<int, 2>{}, r1, [&] { r1.load(wrow); refill(); });
      quarter(std::integral_constant<int, 3>{}, r1, nothing);
    }
  }
  vmwait<0>();

  // blocks that hold a row of wide range, again
  uint32_t wide = 0;
  if (a.dtype == KQ_BF16) {
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
      const int m = 32 * (mb0 + nb) + l32;
      if (__builtin_amdgcn_ballot_w64(a.rs[m < a.M ? m : a.M - 1] < 0.f)) wide |= 1u << nb;
    }
  }
  if (__builtin_expect(wide != 0, 0)) {
#pragma unroll 1
    for (int nb = 0; nb < NB; nb++) {
      if (!((wide >> nb) & 1)) continue;
      f32x16 v = f32x16{0};
      if (row0 < N && mb0 + nb < a.mblocks) {
#pragma unroll 1
        for (int s = s0 + grp; s < s1; s += TL_KS) wide_step<C>(a, row0, N - row0 < 32 ? N - row0 : 32, mb0 + nb, s, l32, kg, row_bytes, v);
      }
#pragma unroll
      for (int c = 0; c < NB; c++)
        if (c == nb) acc[c] = v;
    }
  }

  // The halves' sums: each half finishes some of the blocks (0 ... H - 1 the first, the others the second) and hands over
  // the rest.
  constexpr int H = (NB + 1) / 2;
  float* meet = reinterpret_cast<float*>(wire);
  lds_barrier();
  StaticFor<NB>::run([&](auto nc) __attribute__((always_inline)) {
    constexpr int nb = decltype(nc)::value;
    if ((nb < H) == (grp == 1)) {
      float* to = meet + (nb * TL_NW + nw) * 1024 + lane;
#pragma unroll
      for (int i = 0; i < 16; i++) to[64 * i] = acc[nb][i];
    }
  });
  lds_barrier();
  // Row scales are fetched ahead: a load between two stores would wait for the stores in front of it.
  f32x16 scale[H];
#pragma unroll
  for (int h = 0; h < H; h++) {
    const int nb = grp == 0 ? h : H + h;
    const float* r = a.rs + 32 * (mb0 + nb < a.mblocks ? mb0 + nb : a.mblocks - 1) + 4 * kg;
#pragma unroll
    for (int i = 0; i < 16; i++) scale[h][i] = (wide >> nb) & 1 ? 1.f : r[8 * (i >> 2) + (i & 3)];
  }
  const bool f16 = a.dtype == KQ_F16;
  // Results go back into the slot their sums came from, [32 rows][32 columns] of 16 bits, rows 80 bytes apart, and from there
  // to y in 16-byte pieces of whole rows (2-byte stores, one per result, cost 1.7 us per block of 32 rows).
  constexpr int RROW = 80;
  auto put = [&](int nb, const f32x16& v, const f32x16& sc) __attribute__((always_inline)) {
    uint8_t* to = reinterpret_cast<uint8_t*>(meet + (nb * TL_NW + nw) * 1024) + 2 * l32 + 4 * kg * RROW;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const float r = v[i] * sc[i];
      *reinterpret_cast<uint16_t*>(to + (8 * (i >> 2) + (i & 3)) * RROW) = f16 ? kq::f2f16(r) : kq::f2bf16(r);
    }
  };
  const int n0 = row0 - 32 * nw;  // the tile's first weight row
  auto write_out = [&] {
    lds_barrier();
    const int r = tid >> 4, c = tid & 15, n = n0 + 8 * c;
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
      const int m = 32 * (mb0 + nb) + r;
      const u32x4 v = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint8_t*>(meet + (nb * TL_NW + (c >> 2)) * 1024) + r * RROW + 16 * (c & 3));
      if (m >= a.M) continue;
      uint16_t* y = a.y + (size_t)m * N + n;
      if (a.vec && n + 8 <= N) {
        *reinterpret_cast<u32x4*>(y) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 8; e++)
          if (n + e < N) y[e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
      }
    }
  };
  uint64_t* mine = reinterpret_cast<uint64_t*>(a.part + (size_t)q * (NB * TL_NW * 1024));
  StaticFor<NB>::run([&](auto nc) __attribute__((always_inline)) {
    constexpr int nb = decltype(nc)::value;
    if ((nb < H) == (grp == 0)) {
      const float* from = meet + (nb * TL_NW + nw) * 1024 + lane;
      f32x16 v;  // the first half's steps first
#pragma unroll
      for (int i = 0; i < 16; i++) v[i] = acc[nb][i] + from[64 * i];
      if (!cut) {
        put(nb, v, scale[nb < H ? nb : nb - H]);
      } else {
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
          const float lo = v[i], hi = v[i + 1];  // (a bit cast of a vector's element itself reads element 0)
          __hip_atomic_store(mine + (nb * TL_NW + nw) * 512 + 32 * i + lane,
                             (uint64_t)__builtin_bit_cast(uint32_t, lo) | ((uint64_t)__builtin_bit_cast(uint32_t, hi) << 32),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    }
  });
  if (!cut) {
    write_out();
    return;
  }
  vmwait<0>();
  lds_barrier();
  if (tid == 0)
    *last = __hip_atomic_fetch_add(a.counters + q / a.splits, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.splits - 1;
  lds_barrier();
  if (!*last) return;
  const uint64_t* p0 = reinterpret_cast<const uint64_t*>(a.part + (size_t)(q - range) * (NB * TL_NW * 1024));
  StaticFor<NB>::run([&](auto nc) __attribute__((always_inline)) {
    constexpr int nb = decltype(nc)::value;
    if ((nb < H) == (grp == 0)) {
      f32x16 v = f32x16{0};
      for (int r = 0; r < a.splits; r++) {
        const uint64_t* p = p0 + ((size_t)r * NB * TL_NW + nb * TL_NW + nw) * 512 + lane;
        uint64_t u[8];
#pragma unroll
        for (int i = 0; i < 8; i++) u[i] = __hip_atomic_load(p + 64 * i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] += __builtin_bit_cast(float, (uint32_t)(u[i >> 1] >> (32 * (i & 1))));
      }
      put(nb, v, scale[nb < H ? nb : nb - H]);
    }
  });
  write_out();
}

template <int C, int NB>
int launch_tile(const TileArgs& a, int grid, hipStream_t s) {
  auto kern = tile_kernel<C, NB>;
  KQ_SET_MAX_LDS_ONCE((kern), (TileLds<C, NB>::BYTES));
  hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * TL_WAVES), (TileLds<C, NB>::BYTES), s, a);
  KQ_HIP_CHECK(hipGetLastError());
  return KQ_OK;
}

template <int NB>
int dispatch_tile(const TileArgs& a, int grid, int codec, hipStream_t s) {
  switch (codec) {
#define KQ_CASE(c) \
  case c:          \
    return launch_tile<c, NB>(a, grid, s);
    KQ_CASE(KQ_Q2_K) KQ_CASE(KQ_Q3_K) KQ_CASE(KQ_Q4_K) KQ_CASE(KQ_Q5_K) KQ_CASE(KQ_Q6_K) KQ_CASE(KQ_Q4_0) KQ_CASE(KQ_Q4_1)
    KQ_CASE(KQ_Q5_0) KQ_CASE(KQ_Q5_1) KQ_CASE(KQ_Q8_0) KQ_CASE(KQ_IQ4_NL) KQ_CASE(KQ_IQ4_XS) KQ_CASE(KQ_IQ3_S)
    KQ_CASE(KQ_IQ3_XXS) KQ_CASE(KQ_IQ2_XXS) KQ_CASE(KQ_IQ2_XS) KQ_CASE(KQ_IQ2_S) KQ_CASE(KQ_IQ1_S) KQ_CASE(KQ_IQ1_M)
    KQ_CASE(KQ_MXFP4) KQ_CASE(KQ_NVFP4)
#undef KQ_CASE
  }
  return KQ_ERR_UNSUPPORTED;
}

}  // namespace

#define KQ_TILE_ENTRY_(nb) kq_tile_dispatch_##nb
#define KQ_TILE_ENTRY(nb) KQ_TILE_ENTRY_(nb)
int KQ_TILE_ENTRY(KQ_TILE_NB)(const void* args, int grid, int codec, hipStream_t s) {
  return dispatch_tile<KQ_TILE_NB>(*static_cast<const TileArgs*>(args), grid, codec, s);
}

#if KQ_TILE_NB == 4
int kq_tile_dispatch_2(const void* args, int grid, int codec, hipStream_t s);
int kq_tile_dispatch_3(const void* args, int grid, int codec, hipStream_t s);

static int g_tile_force = 0;  // 33: every call the kernel can run; another forced tile: none
void kq_tile_force(int rows) { g_tile_force = rows; }

namespace {

size_t tile_align(size_t v) { return (v + 255) & ~(size_t)255; }

// Tile height and ranges of a call: the cheapest by a model in us without the prepass, fitted over 819 calls of seven codecs
// (33 ... 1024 rows, ten matrices; the plan it picks is 0.9 % behind the best one on average).  A pair of steps costs 1.2 +
// 0.8 per block of 32 rows, a workgroup 4.6 + 0.9 per block besides, and the last arrival reads 0.44 per block and range.
struct TilePlan {
  int nb, mtiles, ntiles, whole, splits, steps_per_split, cut, grid;
  double cost;
};
TilePlan tile_plan(int M, int N, int K) {
  const int cus = kq_num_cus(), mblocks = (M + 31) / 32, nsteps = K / CK_STEP, ntiles = (N + TL_TN - 1) / TL_TN;
  TilePlan best{};
  for (int nb = 2; nb <= 4; nb++) {
    const int mtiles = (mblocks + nb - 1) / nb, tiles = mtiles * ntiles, whole = tiles / cus * cus, rest = tiles - whole;
    for (int splits = 1; splits <= 16 && splits * 2 <= nsteps; splits++) {
      if (splits > 1 && (rest == 0 || rest * splits > 2 * cus)) break;
      const int per = ((nsteps + splits - 1) / splits + 1) & ~1, sp = (nsteps + per - 1) / per;
      const double pairs = (nsteps + 1) / 2, step = 1.2 + 0.8 * nb, fix = 4.6 + 0.9 * nb;
      const double c = whole / cus * (pairs * step + fix) +
                       (rest ? (rest * sp + cus - 1) / cus * (per / 2 * step + fix) + (sp > 1 ? 0.44 * nb * sp : 0) : 0);
      if (!best.grid || c < best.cost) {
        best = TilePlan{nb, mtiles, ntiles, sp > 1 ? whole : tiles, sp, per, sp > 1 ? rest : 0, sp > 1 ? whole + rest * sp : tiles, c};
      }
    }
  }
  return best;
}

}  // namespace

// What share of its rounds' matrix work the codec's tall-tile kernel (a workgroup per CU, 256 weight rows) would do on real rows:
// 128-row tiles, or 256-row ones, which are `gain` times as fast for their size.
static double tall_share(int M, int N, double gain) {
  const double cus = kq_num_cus(), nt = (N + 255) / 256, work = (double)M * N / (128.0 * 256.0);
  const double r128 = std::ceil((M + 127) / 128 * nt / cus), r256 = std::ceil((M + 255) / 256 * nt / cus);
  return std::max(work / (r128 * cus), gain * work / (2.0 * r256 * cus));
}

bool kq_tile_supported(int M, int N, int K, int codec) {
  if (g_tile_force != 0 && g_tile_force != 33) return false;
  // (nothing of K beyond 32768 has been measured: the kernels that had it keep it)
  if (codec < 0 || codec >= KQ_NUM_CODECS || M <= 32 || N < 8 || K < 2 * CK_STEP || K > 32768 || K % CK_STEP) return false;
  const int64_t row_bytes = (int64_t)(K / kq_geom(codec).wpb) * kq_geom(codec).bpb;
  if (row_bytes * 32 >= ((int64_t)1 << 31) || (int64_t)N * ((M + 31) / 32) >= ((int64_t)1 << 31)) return false;
  if (g_tile_force == 33) return true;
  // Against the streamed kernel: its time is 2 us + 3 per step a wave of it goes through, whatever the codec (without the
  // prepass, which both have).  Over 378 calls of 33 ... 128 rows this picks the faster one to 0.2 %.  Here / there: 4096 x 4096,
  // 64 rows 1.39, 96 1.10, 160 0.95, 256 0.82, 400 0.70; 14336 x 4096, 48 rows 0.78, 160 0.62; 2048 x 2048, 256 rows 1.2, 400 0.85.
  if (kq_mid_supported(M, N, K, codec)) return tile_plan(M, N, K).cost < 2.0 + 3.0 * kq_mid_wave_steps(M, N, K);
  // Against the tall tiles, 21 codecs, 160 ... 2048 rows of five matrices: by how much of those tiles' rounds is work.
  const int64_t cus = kq_num_cus(), nt = (N + 255) / 256, t256 = (M + 255) / 256 * nt, t128 = (M + 127) / 128 * nt;
  switch (codec) {
    case KQ_Q4_K:
    case KQ_Q5_K:
      // 256-row tiles from three quarters of a round on: 28672 x 8192, 400 rows (224 tiles) 1.15, 1.21; 14336 x 4096, 700 rows
      // (168) 0.87, 1024 rows (224) 1.11, 1.19.  128-row tiles in full rounds: 4096 x 4096, 2048 rows 1.15, 1.19, 1536 (192) 0.93.
      return !(4 * t256 >= 3 * cus || (t128 >= cus && tall_share(M, N, 0) > 0.9));
    case KQ_Q6_K:  // 14336 x 4096, 400 rows (0.68) 1.00, 448 (0.77) 1.05, 700 (0.66) 0.98, 1024 (0.96) 1.10
      return tall_share(M, N, 1.1) < 0.74;
    case KQ_Q2_K:
    case KQ_Q3_K:  // 28672 x 8192, 1536 rows (0.87) 0.98, 2048 (1.0) 1.07; 4096 x 4096, 1536 rows (no tall tiles) 0.43, 2048 (1.0) 1.10
      return !(t128 >= cus && tall_share(M, N, 0) > 0.9);
    case KQ_IQ2_XS:
    case KQ_IQ2_S:
    case KQ_IQ1_M:  // a scale per 16 weights to fold: 28672 x 8192, 96 rows (0.33) 0.59, 160 (0.55) 1.16; 14336 x 4096, 256 rows (0.44) 0.78
      return tall_share(M, N, 1.12) < 0.52;
    case KQ_IQ1_S:
    case KQ_IQ2_XXS:
    case KQ_IQ3_S:  // 28672 x 8192, 160 rows (0.55) 0.97; 14336 x 4096, 400 rows (0.68) 1.12
      return tall_share(M, N, 1.12) < 0.62;
    case KQ_IQ3_XXS:
    case KQ_MXFP4:
    case KQ_NVFP4:  // 14336 x 4096, 400 rows (0.68) 1.00, 1.07, 0.98, 700 (0.67) 1.03, 0.96, 0.90, 1024 (0.98) 1.25, 1.17, 1.09
      return tall_share(M, N, 1.12) < 0.74;
  }
  // Two or three terms per weight on the tall tiles against a scale folded per 32 weights here: 28672 x 8192, 2048 rows q8_0 0.94,
  // q5_0 0.95, q4_0 0.90, iq4_nl 0.87, q4_1 0.69, q5_1 0.74, iq4_xs 0.84; 400 rows 0.91, 0.93, 0.84, 0.82, 0.66, 0.72, 0.75.
  return true;
}

size_t kq_tile_workspace_bytes(int M, int N, int K) {
  const size_t mb = (M + 31) / 32, nsteps = K / CK_STEP;
  const TilePlan p = tile_plan(M, N, K);
  return tile_align(mb * nsteps * 18 * 1024) + tile_align(mb * 32 * 4) + tile_align((size_t)p.cut * 4) +
         (size_t)p.cut * p.splits * p.nb * TL_NW * 4096;
}

int kq_launch_tile(const void* x, const uint8_t* w, void* y, int M, int N, int K, int codec, int dtype, void* ws, hipStream_t s) {
  if (!kq_tile_supported(M, N, K, codec) || (reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(ws) & 15) ||
      (reinterpret_cast<uintptr_t>(w) & 1))
    return KQ_ERR_UNSUPPORTED;
  const size_t mb = (M + 31) / 32, nsteps = K / CK_STEP;
  const TilePlan p = tile_plan(M, N, K);
  uint8_t* xf = static_cast<uint8_t*>(ws);
  float* rs = reinterpret_cast<float*>(xf + tile_align(mb * nsteps * 18 * 1024));
  TileArgs a{};
  a.x = static_cast<const uint16_t*>(x);
  a.xf = xf;
  a.rs = rs;
  a.w = w;
  a.y = static_cast<uint16_t*>(y);
  a.grids = kq_device_grids();
  if (!a.grids) return KQ_ERR_HIP;
  a.M = M;
  a.N = N;
  a.K = K;
  a.dtype = dtype;
  a.vec = (N & 7) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
  a.mblocks = (int)mb;
  a.mtiles = p.mtiles;
  a.ntiles = p.ntiles;
  a.whole = p.whole;
  a.splits = p.splits;
  a.steps_per_split = p.steps_per_split;
  a.counters = reinterpret_cast<int*>(reinterpret_cast<uint8_t*>(rs) + tile_align(mb * 32 * 4));
  a.part = reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(a.counters) + tile_align((size_t)p.cut * 4));
  const int rc = kq_launch_mid_prepass(x, xf, rs, a.counters, p.cut, M, K, codec, dtype, s);
  if (rc != KQ_OK) return rc;
  return p.nb == 2 ? kq_tile_dispatch_2(&a, p.grid, codec, s) : p.nb == 3 ? kq_tile_dispatch_3(&a, p.grid, codec, s)
                                                                          : kq_tile_dispatch_4(&a, p.grid, codec, s);
}
#endif
