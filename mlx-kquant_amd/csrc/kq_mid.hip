// Matmul of 9 ... 512 activation rows, every codec: y[M,N] = x[M,K] . W^T between the streamed skinny kernel (M <= 8)
// and the tile GEMMs.
//
// What bounds it: the weight bytes (HBM).  A call of 32 rows does 64 operations per weight, a tenth of what the matrix
// cores could do in the time the weights take to arrive, so the kernel is built like the skinny ones: every wave streams
// wire bytes on its own, and no barrier sits in the stream.
//   * Workgroup = 8 waves on one tile of up to 32 weight rows; wave w takes the 256-weight steps w, w + 8, ...; the
//     waves' sums meet in LDS at the end of the tile.  Workgroups are persistent (one per CU) and a wave's next step,
//     of this tile or the next one, is already on its way while one is multiplied.
//   * A matrix of fewer tiles than CUs cuts its steps into ranges of eight or more, one workgroup each.  The workgroup
//     of a tile that finishes last adds the others' sums, in the order of the ranges (finish_tile): no launch behind.
//   * Wire bytes go to wave-private LDS with direct-to-LDS loads, two slots per wave.
//   * Activations: a prepass writes them as f16 in matrix-operand order, 1 KiB per (32 rows, 16 weights of K), so a
//     fragment is one coalesced 16-byte load per lane straight into registers (L2 serves every tile after the first).
//     Loads of a wave return in order, so fragments and wire bytes of the next step are requested together and waited
//     for together.
//   * bf16 activations become f16 under their row's power of two: exact down to 2^-31 of the row's largest value.  A row of
//     wider range (a value as large as a mask's beside ordinary ones) is flagged by the prepass, and its block of 32 rows
//     takes the activations as they are (wide_step).
//   * 33 rows and more run as blocks of 32 rows: the blocks of a tile are neighbours in launch order on one XCD, so that
//     the second one finds the wire bytes in its L2.
// Measured: see the routing in kq_mid_supported.
#include <algorithm>

#include "kq_mid.h"

namespace {

using namespace kqmid;
using kqmma::RowRange;

// ------------------------------------------------------------------ activation prepass
// One workgroup per activation row m: f16 values scaled by the row's power of two (rs[m]) into fragment order,
//   xf[(m / 32 * nsteps + step) * NF + J][lane = 32 kg + m % 32][8 halves]
// (orders: store_frags in kq_mid.h).
// Rows past M are not written: what they hold reaches output rows that are not stored.
// rs[m] is negative for a wide row (RowRange).
constexpr int MP_THREADS = 512, MP_REGS = 4;

// Row of a workgroup.  Eight neighbouring rows write the 16-byte eighths of the same 128-byte lines, and workgroups go to the
// eight XCDs in turn: rows are dealt so that those eight meet in one L2, which then writes back whole lines.  K = 4096, us in a
// trace, row m on workgroup m before: 32 rows 3.2 -> 2.4, 333 rows 5.2 -> 4.5, 1024 rows 10.2 -> 6.7.
__device__ __forceinline__ int prepass_row_of(int b) { return 64 * (b >> 6) + 8 * (b & 7) + ((b >> 3) & 7); }
constexpr int prepass_grid(int M) { return (M + 63) & ~63; }

template <int DT, int ORD, int NSUM>
__global__ __launch_bounds__(MP_THREADS) void mid_prepass_kernel(const uint16_t* __restrict__ x, uint8_t* __restrict__ xf,
                                                                 float* __restrict__ rs, int M, int K, int nsteps,
                                                                 int* __restrict__ counters, int ncounters) {
  constexpr int NF = 16 + NSUM;
  __shared__ float red[MP_THREADS / 64];
  __shared__ uint32_t range_lds[MP_THREADS / 64 + 2];
  const int tid = threadIdx.x;
  // arrival counters of the main kernel's cut tiles
  for (int i = blockIdx.x * MP_THREADS + tid; i < ncounters; i += gridDim.x * MP_THREADS) counters[i] = 0;
  const int m = prepass_row_of(blockIdx.x);
  if (m >= M) return;
  const uint16_t* xi = x + (size_t)m * K;
  const int ngroups = 32 * nsteps;  // 8-weight groups, the step K ends in zero-filled
  auto fetch = [&](int g) -> u32x4 {
    return 8 * g < K ? *reinterpret_cast<const u32x4*>(xi + 8 * g) : u32x4{0, 0, 0, 0};
  };
  u32x4 keep[MP_REGS];
#pragma unroll
  for (int r = 0; r < MP_REGS; r++) {
    const int g = tid + MP_THREADS * r;
    keep[r] = g < ngroups ? fetch(g) : u32x4{0, 0, 0, 0};
  }
  // The row's power of two puts its largest magnitude into [2^14, 2^15), f16 rows too where that scales up (exact): the
  // hi / lo sums below need room under them.  Left as they came, f16 rows of 6e-5 had their sums rounded to 2^-24, 0.18 % of
  // a q4_1 result.
  float inv = 1.f, scale = 1.f, amax = 0.f;
  auto lo_f = [](uint32_t v) { return DT == KQ_BF16 ? __builtin_bit_cast(float, v << 16) : kq::h2f((uint16_t)(v & 0xffffu)); };
  auto hi_f = [](uint32_t v) { return DT == KQ_BF16 ? __builtin_bit_cast(float, v & 0xffff0000u) : kq::h2f((uint16_t)(v >> 16)); };
  auto take = [&](u32x4 v) {
#pragma unroll
    for (int e = 0; e < 4; e++) amax = fmaxf(amax, fmaxf(fabsf(lo_f(v[e])), fabsf(hi_f(v[e]))));
  };
#pragma unroll
  for (int r = 0; r < MP_REGS; r++) take(keep[r]);
  for (int g = tid + MP_THREADS * MP_REGS; g < ngroups; g += MP_THREADS) take(fetch(g));
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
  if ((tid & 63) == 0) red[tid >> 6] = amax;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < MP_THREADS / 64; w++) amax = fmaxf(amax, red[w]);
  const uint32_t eb = (__builtin_bit_cast(uint32_t, amax) >> 23) & 0xff;
  if (eb != 0 && eb != 0xff) {
    int e = (int)eb - 127 - 14;
    if (e < -100) e = -100;
    if (DT == KQ_F16 && e > 0) e = 0;
    scale = __builtin_bit_cast(float, (uint32_t)(127 + e) << 23);
    inv = __builtin_bit_cast(float, (uint32_t)(127 - e) << 23);
  }
  RowRange range;
  uint8_t* base = xf + (size_t)(m >> 5) * nsteps * NF * 1024 + 16 * (m & 31);
  auto convert = [&](int g, u32x4 v) {  // whole octets of lanes stay together
    _Float16 h[8];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      if constexpr (DT == KQ_BF16) range.take(v[e]);
      h[2 * e] = (_Float16)(lo_f(v[e]) * inv);
      h[2 * e + 1] = (_Float16)(hi_f(v[e]) * inv);
    }
    store_frags<ORD, NSUM>(base + (size_t)(g >> 5) * NF * 1024, g & 31, h);
  };
#pragma unroll
  for (int r = 0; r < MP_REGS; r++) {
    const int g = tid + MP_THREADS * r;
    if (g < ngroups) convert(g, keep[r]);
  }
  for (int g = tid + MP_THREADS * MP_REGS; g < ngroups; g += MP_THREADS) convert(g, fetch(g));
  bool wide = false;
  if constexpr (DT == KQ_BF16) wide = range.wide<MP_THREADS / 64>(scale, eb == 0xff, xi, K, tid, range_lds);
  if (tid == 0) rs[m] = wide ? -scale : scale;
}

// ------------------------------------------------------------------ main kernel
constexpr int MID_WAVES = 8;

struct MidArgs {
  const uint16_t* x;
  const uint8_t* xf;
  const float* rs;
  const uint8_t* w;
  uint16_t* y;
  const uint8_t* grids;
  int M, N, K;
  int rpt;       // weight rows per tile (<= 32): fewer than 32 levels the rows over the workgroups
  int items;     // tiles x 32-row blocks of activations x ranges of steps
  int mblocks;
  int splits, steps_per_split;
  float* part;    // splits > 1: the ranges' sums, [item][1024] f32
  int* counters;  // and the arrivals of every (tile, block), zero at the start
};


__device__ __forceinline__ void mid_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int C, int DT>
__global__ __launch_bounds__(64 * MID_WAVES, 1) void mid_kernel(MidArgs a) {
  using G = MidGeom<C>;
  constexpr int SLOT = mid_slot_bytes<C>(), NW = MID_WAVES, NT = 64 * NW;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  uint8_t* ring = smem + mid_table_bytes<C>();
  int* which = reinterpret_cast<int*>(ring + NW * 2 * SLOT);  // [NW] slot a wave's sums lie in, [NW] = last arrival
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, kg = lane >> 5;
  const int N = a.N, K = a.K, rpt = a.rpt, mblocks = a.mblocks, G_x = gridDim.x;
  const int nsteps = (K + CK_STEP - 1) / CK_STEP;
  const uint32_t row_bytes = (uint32_t)(K / G::WPB) * G::BPB;
  const uint32_t slot_lds = lds_addr(ring + wave * 2 * SLOT);

  kqfrag::KMasks masks;
  masks.init<C>();
  Tables tabs{smem, smem, 2};
  if constexpr (mid_table_bytes<C>() > 0) {
    uint8_t* spread = smem + CodeGeom<C>::GROUPED_GRID_BYTES;
    build_tables<C, NT, true>(smem, spread, a.grids, tid);
    tabs = Tables{CodeGeom<C>::PAIR_LUT ? smem + 4 * l32 : smem, spread, 7};
    lds_barrier();
  }

  // a position of the stream: item (tile, block of activation rows, range of steps) and step of the item's range
  struct Pos {
    int id, st, end;
  };
  // (tile, block)s run over (group of 8 tiles, block, tile of the group): workgroups go to the 8 XCDs in turn, so the
  // blocks of a tile meet in one L2
  auto tile_of = [&](int id, int& tile, int& mb) {
    const int t = id / a.splits, g = t / (8 * mblocks), r = t - g * 8 * mblocks;
    mb = r >> 3;
    tile = 8 * g + (r & 7);
  };
  const int ntiles = (N + rpt - 1) / rpt;
  auto first = [&](int id) {
    int tile, mb;
    tile_of(id, tile, mb);
    const int s0 = (id % a.splits) * a.steps_per_split;
    const int s1 = s0 + a.steps_per_split < nsteps ? s0 + a.steps_per_split : nsteps;
    // st >= end: this wave has no step in the item (or the item is a gap) and only joins the barriers
    return Pos{id, s0 + wave, tile < ntiles ? s1 : 0};
  };
  auto advance = [&](Pos p) {
    p.st += NW;
    return p.st < p.end ? p : first(p.id + G_x);
  };
  uint32_t voff[G::LOADS];
  StaticFor<G::LOADS>::run([&](auto tc) {
    constexpr int T = decltype(tc)::value;
    const int i = lane + 64 * T, r = i / G::LP, p = i - r * G::LP;
    const int off = 16 * p < G::BYTES - 16 ? 16 * p : G::BYTES - 16;
    voff[T] = (uint32_t)r * row_bytes + (uint32_t)off;
  });
  // rs of a block's rows, one per lane
  auto row_scale = [&](int mb) { return a.rs[32 * mb + l32 < a.M ? 32 * mb + l32 : a.M - 1]; };
  auto request = [&](Pos p, int slot, f16x8 (&an)[G::NF], float& rsn) {
    int tile, mb;
    tile_of(p.id, tile, mb);
    if constexpr (DT == KQ_BF16) rsn = row_scale(mb);
    if (p.st >= p.end) return;
    const int row0 = tile * rpt, nrows = N - row0 < rpt ? N - row0 : rpt;
    const uint8_t* base = a.w + (size_t)row0 * row_bytes + (size_t)p.st * G::BYTES;
    const uint32_t l0 = slot_lds + slot * SLOT;
    // The row that ends the matrix inside this step: nothing past its last byte is read (the rows before it read on into the
    // next one, as everywhere), and what would lie there is not used.  Its last, partial piece is the 16 bytes up to the end,
    // shifted.
    const bool ragged_end = (K & (CK_STEP - 1)) != 0 && p.st == nsteps - 1 && row0 + nrows == N;
    const int valid = ragged_end ? (K - CK_STEP * p.st) / G::WPB * G::BPB : 0;  // bytes of the step in that row, 17 or more
    const int npieces = ragged_end ? (nrows - 1) * G::LP + valid / 16 : nrows * G::LP;
    StaticFor<G::LOADS>::run([&](auto tc) {
      constexpr int T = decltype(tc)::value;
      if (64 * T + lane < npieces) dma16(base, voff[T], l0 + 1024 * T);
    });
    if (__builtin_expect(valid % 16, 0)) {
      if (lane == 0) {
        const u32x4 end = *reinterpret_cast<const u32x4_a1*>(base + (size_t)(nrows - 1) * row_bytes + valid - 16);
        *reinterpret_cast<u32x4*>(ring + wave * 2 * SLOT + slot * SLOT + 16 * npieces) = shr_bytes(end, 16 - valid % 16);
      }
      mid_wave_sync();
    }
    const uint8_t* fr = a.xf + ((size_t)mb * nsteps + p.st) * (G::NF * 1024) + 16 * lane;
#pragma unroll
    for (int j = 0; j < G::NF; j++) an[j] = *reinterpret_cast<const f16x8*>(fr + 1024 * j);
  };

  f32x16 acc = f32x16{0};
  auto finish_tile = [&](int id, int slot, bool wide) {
    // the waves' sums meet in the slots just read (a wave's other slot may be receiving its next step)
    float* mine = reinterpret_cast<float*>(ring + (wave * 2 + slot) * SLOT);
#pragma unroll
    for (int i = 0; i < 16; i++) mine[i * 64 + lane] = acc[i];
    acc = f32x16{0};
    if (lane == 0) which[wave] = slot;
    lds_barrier();
    int tile, mb;
    tile_of(id, tile, mb);
    const int row0 = tile * rpt, nrows = N - row0 < rpt ? N - row0 : rpt;
    auto store = [&](int e, float v) {
      const int i = e >> 6, l = e & 63;
      const int m = 32 * mb + 8 * (i >> 2) + 4 * (l >> 5) + (i & 3), c = l & 31;
      if (m < a.M && c < nrows && tile < ntiles) {
        if (!wide) v *= a.rs[m];
        a.y[(size_t)m * N + row0 + c] = DT == KQ_F16 ? kq::f2f16(v) : kq::f2bf16(v);
      }
    };
    static_assert(1024 % NT == 0, "whole passes over the tile");
    float v[1024 / NT];
#pragma unroll
    for (int k = 0; k < 1024 / NT; k++) {
      v[k] = 0.f;
#pragma unroll
      for (int w = 0; w < NW; w++) v[k] += reinterpret_cast<const float*>(ring + (w * 2 + which[w]) * SLOT)[tid + NT * k];
    }
    if (a.splits == 1) {
#pragma unroll
      for (int k = 0; k < 1024 / NT; k++) store(tid + NT * k, v[k]);
      lds_barrier();
      return;
    }
    // The ranges of a tile are added by the workgroup that arrives last.  The sums travel in device-scope atomic
    // stores and loads, which bypass the L2s (one per XCD, not coherent with each other); a wave counts as arrived
    // once its stores have been acknowledged.  No fence: that would write back a whole L2.
    float* part = a.part + (size_t)id * 1024;
#pragma unroll
    for (int k = 0; k < 1024 / NT; k++)
      __hip_atomic_store(part + tid + NT * k, v[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    vmwait<0>();
    lds_barrier();
    if (tid == 0)
      which[NW] = __hip_atomic_fetch_add(a.counters + id / a.splits, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.splits - 1;
    lds_barrier();
    if (which[NW]) {
      const float* p0 = a.part + (size_t)(id - id % a.splits) * 1024;
#pragma unroll
      for (int k = 0; k < 1024 / NT; k++) {
        float sum = 0.f;
        for (int r = 0; r < a.splits; r++)
          sum += __hip_atomic_load(p0 + (size_t)r * 1024 + tid + NT * k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        store(tid + NT * k, sum);
      }
    }
    lds_barrier();
  };

  f16x8 a0[G::NF], a1[G::NF];
#pragma unroll
  for (int j = 0; j < G::NF; j++) a0[j] = a1[j] = f16x8{};
  float rs0 = 0.f, rs1 = 0.f;
  Pos cur = first(blockIdx.x);
  request(cur, 0, a0, rs0);
  // one step: wait for it, ask for the next one, multiply
  auto body = [&](f16x8 (&ac)[G::NF], f16x8 (&an)[G::NF], float& rsc, float& rsn, int slot) -> bool {
    vmwait<0>();
    lgkm_drain();  // the other slot has been read: it may be filled again
#pragma unroll
    for (int j = 0; j < G::NF; j++) asm volatile("" : "+v"(ac[j]));
    const Pos nxt = advance(cur);
    const bool more = nxt.id < a.items;
    bool wide = false;
    if constexpr (DT == KQ_BF16) wide = __builtin_amdgcn_ballot_w64(rsc < 0.f) != 0;
    if (__builtin_expect(wide && cur.st < cur.end, 0)) {  // before the request: its registers are free here
      int tile, mb;
      tile_of(cur.id, tile, mb);
      const int row0 = tile * rpt;
      wide_step<C>(a, row0, N - row0 < rpt ? N - row0 : rpt, mb, cur.st, l32, kg, row_bytes, acc);
    }
    if (more) request(nxt, slot ^ 1, an, rsn);
    if (__builtin_expect(cur.st < cur.end && !wide, 1))
      mid_step<C>(ring + (wave * 2 + slot) * SLOT + l32 * G::LROW, kg, ac, tabs, masks, K - CK_STEP * cur.st, acc);
    if (nxt.id != cur.id) {
      mid_wave_sync();
      finish_tile(cur.id, slot, wide);
    }
    cur = nxt;
    return more;
  };
  while (true) {
    if (!body(a0, a1, rs0, rs1, 0)) break;
    if (!body(a1, a0, rs1, rs0, 1)) break;
  }
}

size_t mid_align(size_t v) { return (v + 255) & ~(size_t)255; }

// Tiles, ranges and workgroups of a call.  At least one tile per CU: 32-row tiles dealt out in rounds, levelled to the
// same number of rows.  Fewer: the steps are cut into ranges of two or more per wave, as many as fill the CUs; a K too
// short for that takes shorter tiles (some lanes then decode for nobody, but more CUs pull).  q4_k, 32 rows, us, prepass
// included: 4096 rows of K = 14336 on 16-row tiles 23.5, cut in two 20.7; of K = 4096 (one step per wave when cut) 11.2
// and 11.7.
struct MidPlan {
  int rpt, ntiles, splits, steps_per_split, items, grid;
};
MidPlan mid_plan(int M, int N, int K) {
  MidPlan p;
  const int cus = kq_num_cus(), mblocks = (M + 31) / 32, nsteps = (K + CK_STEP - 1) / CK_STEP;
  const int t32 = (N + 31) / 32 * mblocks;
  p.splits = 1;
  if (t32 < cus) p.splits = std::max(1, std::min(cus / t32, nsteps / (2 * MID_WAVES)));
  p.steps_per_split = (nsteps + p.splits - 1) / p.splits;
  p.splits = (nsteps + p.steps_per_split - 1) / p.steps_per_split;
  p.rpt = 32;
  if (p.splits == 1) {
    const int64_t rounds = (t32 + cus - 1) / cus;
    const int rpt = (int)((((int64_t)N * mblocks + cus * rounds - 1) / (cus * rounds) + 3) & ~3);
    p.rpt = rpt < 8 ? 8 : rpt > 32 ? 32 : rpt;
    // (the last tile and the last group of eight may be partly empty)
    while (p.rpt < 32 && (int64_t)((N + p.rpt - 1) / p.rpt + 7) / 8 * 8 * mblocks > cus * rounds) p.rpt += 4;
  }
  p.ntiles = (N + p.rpt - 1) / p.rpt;
  p.items = (p.ntiles + 7) / 8 * 8 * mblocks * p.splits;  // gaps in the last group of eight tiles included
  p.grid = p.items < cus ? p.items : cus;
  return p;
}

template <int C, int DT>
int launch_prepass(const void* x, uint8_t* xf, float* rs, int* counters, int ncounters, int M, int K, hipStream_t s) {
  using G = MidGeom<C>;
  hipLaunchKernelGGL((mid_prepass_kernel<DT, G::ORD, G::NSUM>), dim3(prepass_grid(M)), dim3(MP_THREADS), 0, s,
                     static_cast<const uint16_t*>(x), xf, rs, M, K, (K + CK_STEP - 1) / CK_STEP, counters, ncounters);
  KQ_HIP_CHECK(hipGetLastError());
  return KQ_OK;
}

template <int C, int DT>
int launch_mid(const void* x, MidArgs a, uint8_t* xf, float* rs, hipStream_t s) {
  constexpr size_t lds = (size_t)mid_table_bytes<C>() + (size_t)MID_WAVES * 2 * mid_slot_bytes<C>() + 64;
  static_assert(lds <= 160 * 1024, "the ring does not fit the LDS of a CU");
  const MidPlan p = mid_plan(a.M, a.N, a.K);
  a.rpt = p.rpt;
  a.items = p.items;
  a.splits = p.splits;
  a.steps_per_split = p.steps_per_split;
  const int ncounters = p.splits > 1 ? p.items / p.splits : 0;
  a.part = reinterpret_cast<float*>(a.counters + mid_align((size_t)ncounters * 4) / 4);
  const int rc = launch_prepass<C, DT>(x, xf, rs, a.counters, ncounters, a.M, a.K, s);
  if (rc != KQ_OK) return rc;
  auto kern = mid_kernel<C, DT>;
  KQ_SET_MAX_LDS_ONCE((kern), lds);
  hipLaunchKernelGGL(kern, dim3(p.grid), dim3(64 * MID_WAVES), lds, s, a);
  KQ_HIP_CHECK(hipGetLastError());
  return KQ_OK;
}

}  // namespace

static int g_mid_tile = 0;  // 32: every call the kernel can run; another forced tile: none
void kq_mid_force_tile(int rows) { g_mid_tile = rows; }

// Codecs that the any-codec kernel decodes fast: one table entry of eight weights per index.
static bool short_any_decode(int codec) {
  return codec == KQ_IQ1_S || codec == KQ_IQ1_M || codec == KQ_IQ2_XXS || codec == KQ_IQ2_XS;
}

bool kq_mid_supported(int M, int N, int K, int codec) {
  if (g_mid_tile != 0 && g_mid_tile != 32) return false;
  if (codec < 0 || codec >= KQ_NUM_CODECS || M <= 8 || N < 8 || K < CK_STEP || K % kq_geom(codec).wpb) return false;
  const int64_t row_bytes = (int64_t)(K / kq_geom(codec).wpb) * kq_geom(codec).bpb;
  if (row_bytes & 1) return false;  // the direct-to-LDS loads take 2-byte aligned addresses
  if (row_bytes * 32 >= ((int64_t)1 << 31) || (int64_t)N * ((M + 31) / 32) >= ((int64_t)1 << 31)) return false;
  if (g_mid_tile == 32) return M <= KQ_MID_MAX_ROWS;
  // Against the tile GEMMs, us at 32 / 64 / 128 rows: q4_k 4096^2 11 / 13 / 18 (64-row kernel 19 / 23 / 25), 28672 x 8192
  // 55 / 84 / 149 (64 / 70 / 114): from two row blocks on the tile GEMM of the K-quants with exact integers is ahead on
  // the large matrices, where a weight decoded once per 64 rows counts.  The any-codec kernel the others have there is
  // behind on every shape: mxfp4 28672 x 8192 56 / 85 / 147 (131 / 164 / 298), q8_0 77 / 113 / 193 (114 / 136 / 229).
  // Matrices of up to 4096 rows leave that GEMM with too few tiles up to 192 activation rows.  Here over there, 128 and 192
  // rows, q4_k: K = 4096, 1024 rows 0.68, 0.66, 2048 rows 0.62, 0.82, 4096 rows 0.74, 0.79, K = 14336, 4096 rows 0.97, 0.93; q6_k 0.73,
  // 0.71, 0.69, 0.91, 0.89, 0.87, 1.03, 0.94.  Past that a line in rows no longer tells: K = 4096, 6144 rows 0.81, 0.85, 8192 0.92,
  // 0.97, 11008 0.96, 0.95, 14336 1.05, 1.10, 5120 x 13824 1.08, 1.08, 8192 x 8192 1.01, 0.97; those calls stay there.
  const bool tile_gemm = codec == KQ_Q4_K || codec == KQ_Q5_K || codec == KQ_Q6_K;
  if (tile_gemm) return M <= 32 || (M <= 64 && (int64_t)N * K <= (int64_t)64 << 20) || (M <= 192 && N <= 4096);
  // Against the any-codec kernel's 128-row tiles with its short decode for these codecs: a weight decoded once per 128 rows
  // instead of once per 32 wins where its last tile is (nearly) full and it has the tiles to cut K into whole rounds.  Here /
  // there, us: iq2_xs 128 rows 8192 x 8192 68 / 61, 14336 x 4096 64 / 60, 256 rows 4096 x 14336 114 / 96, 8192 x 4096 76 / 62, 400 rows
  // 4096 x 4096 70 / 59, 512 80 / 62; but 160 rows 8192 x 8192 82 / 98 and 1024 x 4096, 256 rows, 16 / 22.  The others at 512 rows
  // of 4096 x 4096: iq1_m 74 / 63, iq1_s 66 / 60, iq2_xxs 71 / 65, but of 2880 x 2816 (92 tiles, no whole rounds) 0.92 ... 0.85 of
  // it, as at 256 rows of 4096 x 4096.
  if (short_any_decode(codec)) {
    const int64_t tiles = (int64_t)((M + 127) / 128) * ((N + 127) / 128);
    const int blocks = (M + 31) / 32, full = (M + 127) / 128 * 4;
    if (4 * tiles >= kq_num_cus()) {
      const bool whole = 2 * kq_num_cus() % tiles == 0;
      if (codec == KQ_IQ2_XS && M > 96 && (8 * blocks >= 7 * full || (whole && 5 * blocks >= 4 * full))) return false;
      if (M > 384 && blocks == full && whole) return false;
    }
  }
  if (M <= 128) return true;
  // 129 ... 512 rows: until the codec's tall tiles fill enough of the chip (one workgroup per CU and no K split there, so
  // an unfilled round costs a whole one).  us here / on tall tiles / on the any-codec kernel, which had these calls:
  // mxfp4 4096 x 14336 256 rows 76 / 235 / 147, 512 rows 161 / 236 / 266, 14336 x 4096 333 rows 111 / 84 / 282; iq3_s
  // 14336 x 4096 192 rows 89 / 87 / 154; q8_0 14336 x 4096 256 rows 101 / 97 / 130, 333 rows 137 / 103 / 210.
  // The kernel that would take the call is asked itself: it has conditions on K and M of its own.
  return M <= KQ_MID_MAX_ROWS && !kq_gemm2_low_supported(M, N, K, codec) && !kq_gemm3b_supported(M, N, K, codec) &&
         !kq_gemm3f_supported(M, N, K, codec) && !kq_gemm3i_supported(M, N, K, codec);
}

// Whether the tall-tile GEMM of a codec (kq_gemm3b / 3f / 3i.hip: 128 x 256 tiles, a workgroup per CU) has the tiles to beat
// the streamed kernel: three fifths of a round for two or three terms per weight, seven sixteenths for one term.
// Above the rows of the streamed kernel the alternative is the any-codec kernel.  Tall tiles against it, by tiles of 256 CUs
// (640 ... 1400 rows of 1024 ... 8192 weight rows; an unfilled round costs a whole one): mxfp4 48 tiles 1.00, 60 0.88, nvfp4
// 40 0.81; q8_0 / q5_0 60 1.25, 64 1.29, 72 0.91, 80 0.95 ... 1.01, q4_0 / iq4_nl 64 1.13 ... 1.19, 72 0.80; iq2_s / iq3_s /
// iq3_xxs 64 1.02 ... 1.12, 72 0.84 ... 0.92; iq1_s / iq1_m / iq2_xs / iq2_xxs, whose any-codec decode is short, 64 1.31 ... 1.36,
// 72 1.02 ... 1.08, 80 0.88 ... 0.96; q4_1 / q5_1 with their third term 96 0.91 ... 1.10, 128 1.06 ... 1.19, 132 0.90, 140 0.63.
bool kq_tall_fills(int M, int N, int codec) {
  const int64_t tiles = (int64_t)((M + 127) / 128) * ((N + 255) / 256), cus = kq_num_cus();
  const bool three = codec == KQ_Q4_1 || codec == KQ_Q5_1;
  if (M > KQ_MID_MAX_ROWS) {
    const bool fp4 = codec == KQ_MXFP4 || codec == KQ_NVFP4;
    return three ? 2 * tiles > cus : 32 * tiles >= (fp4 ? 8 : short_any_decode(codec) ? 10 : 9) * cus;
  }
  const bool two = codec == KQ_Q8_0 || codec == KQ_Q4_0 || codec == KQ_IQ4_NL || codec == KQ_Q5_0;
  return two || three ? 5 * tiles >= 3 * cus : 16 * tiles >= 7 * cus;
}

KqRedo kq_tall_redo(void* ws, int M, int N, int K) {
  if (4 * (int64_t)((M + 127) / 128) * ((N + 255) / 256) >= 3 * (int64_t)kq_num_cus()) return KqRedo{nullptr, nullptr};
  int* rows = reinterpret_cast<int*>(static_cast<uint8_t*>(ws) + (size_t)M * K * 2 + (size_t)M * 4);
  return KqRedo{rows, rows + M};
}

// Steps that a wave goes through one after the other.
int kq_mid_wave_steps(int M, int N, int K) {
  const MidPlan p = mid_plan(M, N, K);
  return (p.items + p.grid - 1) / p.grid * ((p.steps_per_split + MID_WAVES - 1) / MID_WAVES);
}

size_t kq_mid_workspace_bytes(int M, int N, int K) {
  const size_t mb = (M + 31) / 32, nsteps = (K + CK_STEP - 1) / CK_STEP;
  const MidPlan p = mid_plan(M, N, K);
  const size_t cut = p.splits > 1 ? mid_align((size_t)(p.items / p.splits) * 4) + (size_t)p.items * 4096 : 0;
  return mid_align(mb * nsteps * 18 * 1024) + mid_align(mb * 32 * 4) + cut;
}

int kq_launch_mid(const void* x, const uint8_t* w, void* y, int M, int N, int K, int codec, int dtype, void* ws, hipStream_t s) {
  if (!kq_mid_supported(M, N, K, codec) || (reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(ws) & 15) ||
      (reinterpret_cast<uintptr_t>(w) & 1) || (K & 7))
    return KQ_ERR_UNSUPPORTED;
  const size_t mb = (M + 31) / 32, nsteps = (K + CK_STEP - 1) / CK_STEP;
  uint8_t* xf = static_cast<uint8_t*>(ws);
  float* rs = reinterpret_cast<float*>(xf + mid_align(mb * nsteps * 18 * 1024));
  MidArgs a{};
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
  a.mblocks = (int)mb;
  a.counters = reinterpret_cast<int*>(reinterpret_cast<uint8_t*>(rs) + mid_align(mb * 32 * 4));
  switch (codec) {
#define KQ_CASE(c) \
  case c:          \
    return dtype == KQ_F16 ? launch_mid<c, KQ_F16>(x, a, xf, rs, s) : launch_mid<c, KQ_BF16>(x, a, xf, rs, s);
    KQ_CASE(KQ_Q2_K) KQ_CASE(KQ_Q3_K) KQ_CASE(KQ_Q4_K) KQ_CASE(KQ_Q5_K) KQ_CASE(KQ_Q6_K) KQ_CASE(KQ_Q4_0) KQ_CASE(KQ_Q4_1)
    KQ_CASE(KQ_Q5_0) KQ_CASE(KQ_Q5_1) KQ_CASE(KQ_Q8_0) KQ_CASE(KQ_IQ4_NL) KQ_CASE(KQ_IQ4_XS) KQ_CASE(KQ_IQ3_S)
    KQ_CASE(KQ_IQ3_XXS) KQ_CASE(KQ_IQ2_XXS) KQ_CASE(KQ_IQ2_XS) KQ_CASE(KQ_IQ2_S) KQ_CASE(KQ_IQ1_S) KQ_CASE(KQ_IQ1_M)
    KQ_CASE(KQ_MXFP4) KQ_CASE(KQ_NVFP4)
#undef KQ_CASE
  }
  return KQ_ERR_UNSUPPORTED;
}

int kq_launch_mid_prepass(const void* x, uint8_t* xf, float* rs, int* counters, int ncounters, int M, int K, int codec, int dtype,
                          hipStream_t s) {
  switch (codec) {
#define KQ_CASE(c) \
  case c:          \
    return dtype == KQ_F16 ? launch_prepass<c, KQ_F16>(x, xf, rs, counters, ncounters, M, K, s) \
                           : launch_prepass<c, KQ_BF16>(x, xf, rs, counters, ncounters, M, K, s);
    KQ_CASE(KQ_Q2_K) KQ_CASE(KQ_Q3_K) KQ_CASE(KQ_Q4_K) KQ_CASE(KQ_Q5_K) KQ_CASE(KQ_Q6_K) KQ_CASE(KQ_Q4_0) KQ_CASE(KQ_Q4_1)
    KQ_CASE(KQ_Q5_0) KQ_CASE(KQ_Q5_1) KQ_CASE(KQ_Q8_0) KQ_CASE(KQ_IQ4_NL) KQ_CASE(KQ_IQ4_XS) KQ_CASE(KQ_IQ3_S)
    KQ_CASE(KQ_IQ3_XXS) KQ_CASE(KQ_IQ2_XXS) KQ_CASE(KQ_IQ2_XS) KQ_CASE(KQ_IQ2_S) KQ_CASE(KQ_IQ1_S) KQ_CASE(KQ_IQ1_M)
    KQ_CASE(KQ_MXFP4) KQ_CASE(KQ_NVFP4)
#undef KQ_CASE
  }
  return KQ_ERR_UNSUPPORTED;
}
