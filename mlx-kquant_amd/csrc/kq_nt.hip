// transpose = false on the matrix cores: y[m, n] = sum_k x[m, k] * W[k, n], W stored as K wire rows of N weights
// (the orientation of the reference's qmm_n, src/kquant_matmul.cpp:455-527, and of its gathered form
// src/kquant_gather.cpp:470-746 with transpose = false: MLA's absorbed projections and the LoRA vjp).
//
// The reduction runs over wire ROWS, so a decoded 8-weight group (8 consecutive n of one row k) is not an MFMA
// operand by itself: an operand wants 8 consecutive k of one column.  The kernel gets there without any
// transpose: lane (c = lane % 16, h = lane / 16) decodes the SAME 8-column group c of 8 consecutive rows
// k0 + 8h ... k0 + 8h + 7; value t of those eight groups, taken over the rows, is the B operand of MFMA number t
// (v_mfma_f32_16x16x32_bf16: 32 rows of K a step), whose 16 columns are then the strided set {8c + t}.  Eight
// accumulator tiles (t = 0 ... 7) cover 128 consecutive output columns, and the eight results of a lane for one
// output row are 8 consecutive columns: one 16-byte store.
//
// Numerics: every decoded weight (f32, reference order, kq_decode.h) is split into two bf16 terms (16 mantissa
// bits), f16 activations into two exact bf16 terms, bf16 activations are used as they are; the MFMA forms exact
// products and sums in f32.
//
// Workgroup = 4 waves on one (entry, 16 or 32 activation rows, 128 columns) tile; the waves take the 32-row steps
// of K in turn and their accumulators meet in LDS.  A wave copies the 32 row pieces of its step (the wire bytes of
// the tile's columns, contiguous per row; for the 256-weight codecs the whole superblock, which two column tiles
// share) into its own LDS area with dword loads issued one step ahead, and the decoders read the bytes from there:
// decoding straight from global memory costs about 130 byte-wide loads a step.  Calls of 96 rows and more run
// gemm_nt_wide_kernel below, which decodes a step once for 128 activation rows, or from 512 rows on, where its tiles fill the
// chip (nt_tall), gemm_nt_tall_kernel (256 rows).
#include <algorithm>
#include <type_traits>

#include "kq_decode.h"
#include "kq_dma.h"
#include "kq_entries.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32_a1 __attribute__((aligned(1)));  // the hardware serves unaligned dword loads

constexpr int NT_WAVES = 4, NT_THREADS = 64 * NT_WAVES;
constexpr int NT_KSTEP = 32, NT_COLS = 128;
// Codecs whose 32-row form does not fit 256 registers (it spills up to 248 bytes per lane) take 64-row tiles on one
// wave per SIMD beyond 32 rows (q6_k 4096 x 4096, 512 rows: 292 -> 146 us); for the others the 64-row form measured
// level or slower (q8_0 93 -> 111 us).
constexpr bool nt_wide(int codec) { return codec == KQ_Q6_K; }
// Calls of this many activation rows take the kernel that decodes a step once for 128 rows
#ifndef KQ_NT_SHARED_ROWS
#define KQ_NT_SHARED_ROWS 96
#endif
constexpr int NT_SHARED_ROWS = KQ_NT_SHARED_ROWS;

struct NtArgs {
  const void* x;
  const uint8_t* w;
  void* y;
  const uint32_t* lhs;
  const uint32_t* rhs;
  int M, N, K, E, B;
  int64_t x_batch_stride, w_expert_stride;
  int x_vec;  // activation rows can be read 16 bytes at a time (K % 8 == 0, aligned base and stride)
  // dense calls with few tiles: grid z cuts the K steps into ksplit ranges whose f32 partial sums go to `part`
  // ([ksplit, M, N]) and are added by nt_reduce_kernel
  int ksplit, steps_per_split;
  float* part;
  bool tall;  // 256-row tiles
};

__device__ __forceinline__ uint32_t pack_hi(float a, float b) {
  // upper halves of two f32 = their bf16 truncations, a in the low half
  return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302u);
}
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_rne(float a, float b) {
  // two f32 rounded to nearest-even bf16 (v_cvt_pk_bf16_f32), a in the low half
  const bf16x2 v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float trunc_bf16(float a) {
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, a) & 0xffff0000u);
}

template <int C>
struct NtGeom {
  static constexpr int WPB = kq_geom(C).wpb, BPB = kq_geom(C).bpb, GPB = WPB / 8;
  static constexpr bool SUPER = WPB > NT_COLS;          // two column tiles share the row piece of a superblock
  static constexpr int PCOLS = SUPER ? WPB : NT_COLS;    // columns a row piece covers
  static constexpr int PIECE = PCOLS / WPB * BPB;        // ... and its wire bytes
  static constexpr int PDW = 2 * ((PIECE + 7) / 8), STRIDE = 4 * PDW;  // rows 8-byte aligned in LDS
  static constexpr int NDW = (NT_KSTEP * PDW + 63) / 64;  // dwords a lane copies per step
  static constexpr int STAGE_BYTES = NT_WAVES * NT_KSTEP * STRIDE;
};

// MR = 16-row groups of activations per workgroup (1: up to 16 rows, 2: 32, 4: 64 rows on one wave per SIMD, for
// calls of many rows: every decoded weight then feeds four MFMAs)
// MERGE (gathered calls of few rows per entry that name the experts more than once): grid z counts experts, and a workgroup
// multiplies 16 MR rows of its expert's entries (grid y of them), then some that a larger expert leaves over (kq_entries.h).  It
// asks for its first wire bytes before it looks for the entries in the id list.  128 heads of 128 -> 512, us, 4 x 1 / 8 x 1 / 8 x 4
// (sequences x rows), against a workgroup per entry that looked for the others of its expert: q8_0 12.8 / 26.4 / 32.7 ->
// 8.8 / 9.1 / 12.0, q4_k 14.2 / 27.7 / 34.5 -> 9.6 / 9.9 / 12.1, q6_k 15.9 / 29.5 / 37.6 -> 10.9 / 11.3 / 13.9.  1024 entries of 8
// rows, 64 experts, q8_0: all on one 66 -> 33 (427 with its rounds in series on its own workgroups), half of them 54 -> 34, random
// ids 53 -> 31; of one row 46 -> 16, 32 -> 16, 30 -> 16 (in series 276, 140, 12).
template <int C, int DT, int MR, bool MERGE = false>
__global__ __launch_bounds__(NT_THREADS, MR == 4 ? 1 : 2) void gemm_nt_mfma_kernel(NtArgs a, const uint8_t* __restrict__ grids) {
  using G = NtGeom<C>;
  constexpr int BPB = G::BPB, GPB = G::GPB, PDW = G::PDW, STRIDE = G::STRIDE, NDW = G::NDW;
  constexpr int RED_BYTES = 2 * 32 * MR * 64 * 4;  // two waves' accumulators; shares the space of the staging areas
  __shared__ __attribute__((aligned(16))) uint8_t lds[G::STAGE_BYTES > RED_BYTES ? G::STAGE_BYTES : RED_BYTES];
  float* red = reinterpret_cast<float*>(lds);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, h = lane >> 4;
  const int item = a.ksplit > 1 || MERGE ? 0 : blockIdx.z, split = a.ksplit > 1 ? blockIdx.z : 0;
  const uint32_t e = MERGE ? blockIdx.z : a.rhs ? a.rhs[item] : 0u;
  if (e >= (uint32_t)a.E) return;  // the whole workgroup leaves: the entry's output rows stay untouched
  static_assert(!MERGE || MR <= 2, "rows of a round");
  static_assert(!MERGE || NT_THREADS == kqentries::THREADS, "the search of the id list");
  __shared__ std::conditional_t<MERGE, kqentries::Places, int> places;
  __shared__ std::conditional_t<MERGE, kqentries::Share, int> share;
  __shared__ uint32_t entries[MERGE ? kqentries::count_bytes(kqentries::MAX_ENTRIES / 2) / 4 : 1];  // per expert (nt_merge)
  __shared__ int64_t x_off[MERGE ? 16 * MR : 1], y_row[MERGE ? 16 * MR : 1];
  const int tile = blockIdx.x;
  const int ngroups = a.N / 8;
  const int gi = tile * 16 + c;  // this lane's 8-column group
  const bool col_ok = gi < ngroups;
  const size_t row_bytes = (size_t)(a.N / G::WPB) * BPB;
  const int pi = G::SUPER ? tile >> 1 : tile;  // row piece the tile reads
  // group inside the piece; lanes past the last column decode the last group and store nothing
  const int gp = (col_ok ? gi : ngroups - 1) - pi * (G::PCOLS / 8);
  const uint8_t* wt = a.w + (size_t)e * (size_t)a.w_expert_stride + (size_t)pi * G::PIECE;  // MERGE: of the round's expert
  const int cols_here = a.N - G::PCOLS * pi < G::PCOLS ? a.N - G::PCOLS * pi : G::PCOLS;
  const int piece_here = cols_here / G::WPB * BPB;  // the last piece of a 32-weight codec may be shorter
  uint8_t* stage = lds + wave * NT_KSTEP * STRIDE;
  const uint8_t* blk = stage + (gp / GPB) * BPB;
  const int g = gp % GPB, klast = a.K - 1;
  const uint16_t* xr[MR];
  uint32_t wreg[NDW], xreg[MR][4];
  // Rows past K repeat the last row (their activations are zero).  No branch stands between the loads, so they are
  // all in flight together: a lane past the end of the step or of a short piece reads a clamped address, and the
  // last bytes of a piece come out of the dword that ends with the piece, shifted (never a byte past a row's end).
  auto fetch_w = [&](int st) {
    int l = lane;
    // the addresses are not kept from one use to the next: most merged waves have one step, and 27 addresses of q6_k spilled 76
    // registers over the loop of rounds
    if constexpr (MERGE) asm volatile("" : "+v"(l));
#pragma unroll
    for (int j = 0; j < NDW; j++) {
      const int idx = l + 64 * j < NT_KSTEP * PDW ? l + 64 * j : NT_KSTEP * PDW - 1;
      const int row = idx / PDW, boff = 4 * (idx - row * PDW);
      const int eoff = boff < piece_here - 4 ? boff : piece_here - 4;
      const int k = NT_KSTEP * st + row < a.K ? NT_KSTEP * st + row : klast;
      const uint32_t v = *reinterpret_cast<const u32_a1*>(wt + (size_t)k * row_bytes + eoff);
      wreg[j] = v >> (8 * ((boff - eoff) & 3));
    }
  };
  auto fetch_x = [&](int st) {
    const int k0 = NT_KSTEP * st + 8 * h;
#pragma unroll
    for (int q = 0; q < MR; q++) {
#pragma unroll
      for (int j = 0; j < 4; j++) xreg[q][j] = 0u;
      if (a.x_vec) {  // K is a multiple of 8 here: a group of 8 lies inside the row or past it
        const uint4 v = *reinterpret_cast<const uint4*>(xr[q] + (k0 < a.K ? k0 : 0));
        const bool in = k0 < a.K;
        xreg[q][0] = in ? v.x : 0u, xreg[q][1] = in ? v.y : 0u, xreg[q][2] = in ? v.z : 0u, xreg[q][3] = in ? v.w : 0u;
      } else {
#pragma unroll
        for (int i = 0; i < 8; i++)
          if (k0 + i < a.K) xreg[q][i >> 1] |= (uint32_t)xr[q][k0 + i] << (16 * (i & 1));
      }
    }
  };

  const int steps_all = (a.K + NT_KSTEP - 1) / NT_KSTEP;
  const int st_begin = split * a.steps_per_split;
  const int nsteps = st_begin + a.steps_per_split < steps_all ? st_begin + a.steps_per_split : steps_all;
  int rows = a.M, m0 = 16 * MR * blockIdx.y;
  if constexpr (MERGE) {
    if (blockIdx.y == 0 && st_begin + wave < nsteps) fetch_w(st_begin + wave);
    kqentries::Ids ids;
    ids.load(a.rhs, a.lhs, a.B, threadIdx.x);
    rows = kqentries::find_and_count(ids, e, a.B, a.E, threadIdx.x, wave, places, entries, share, [] { __syncthreads(); }) * a.M;
    if (m0 >= rows) {  // uniform
      __syncthreads();
      kqentries::note_left<16 * MR>(a.M, a.E, gridDim.y, threadIdx.x, entries, share);
      __syncthreads();
      if (!share.left) return;
    }
  }
  // MERGE: a round of the workgroup's own expert, if it has one for it, then one that another expert leaves over
  bool fetched = MERGE && blockIdx.y == 0, own = !MERGE || m0 < rows, others = false;
#pragma unroll 1
  for (;;) {
    int tid = threadIdx.x;
    if constexpr (MERGE) {
      if (__builtin_expect(!own, 0)) {
        asm volatile("" : "+v"(tid));  // what the search derives from it is not kept from one round to the next
        const uint32_t next = kqentries::share_rounds<16 * MR>(a.B, a.M, a.E, gridDim.y, e, blockIdx.y, tid, entries, share,
                                                               [] { __syncthreads(); });
        if (next == kqentries::NO_ROUND) return;
        others = true;
        const uint32_t expert = next & (kqentries::MAX_EXPERTS - 1);
        m0 = 16 * MR * (int)(next >> kqentries::EXPERT_BITS);
        wt = a.w + (size_t)expert * (size_t)a.w_expert_stride + (size_t)pi * G::PIECE;
        kqentries::Ids ids;
        ids.load(a.rhs, a.lhs, a.B, tid);
        rows = ids.find(expert, a.B, tid, wave, places, [] { __syncthreads(); }) * a.M;
        fetched = false;
      }
      __syncthreads();
      if (tid < 16 * MR) {  // rows past the last repeat it, never stored
        const int r = m0 + tid < rows ? m0 + tid : rows - 1, place = r / a.M, m = r - place * a.M;
        x_off[tid] = (int64_t)places.lhs_of[place] * a.x_batch_stride + (int64_t)m * a.K;
        y_row[tid] = (int64_t)places.entry_of[place] * a.M + m;
      }
      __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < MR; q++) {
      if constexpr (MERGE) {
        xr[q] = static_cast<const uint16_t*>(a.x) + x_off[16 * q + c];
      } else {
        const int mrow = m0 + 16 * q + c < a.M ? m0 + 16 * q + c : a.M - 1;  // rows past the last repeat it, never stored
        xr[q] = static_cast<const uint16_t*>(a.x) + (a.lhs ? (size_t)a.lhs[item] * (size_t)a.x_batch_stride : 0) + (size_t)mrow * a.K;
      }
    }
    f32x4 acc[MR][8];
#pragma unroll
    for (int q = 0; q < MR; q++)
#pragma unroll
      for (int t = 0; t < 8; t++) acc[q][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (st_begin + wave < nsteps) {
      if (!fetched) fetch_w(st_begin + wave);
      fetch_x(st_begin + wave);
    }
    if constexpr (MERGE) {
      if (own) kqentries::note_left<16 * MR>(a.M, a.E, gridDim.y, tid, entries, share);
    }
    for (int st = st_begin + wave; st < nsteps; st += NT_WAVES) {
#pragma unroll
      for (int j = 0; j < NDW; j++) {
        const int idx = lane + 64 * j;
        if (idx < NT_KSTEP * PDW) *reinterpret_cast<uint32_t*>(stage + 4 * idx) = wreg[j];
      }
      bf16x8 ah[MR], al[MR];
#pragma unroll
      for (int q = 0; q < MR; q++) {
        if constexpr (DT == KQ_BF16) {
          ah[q] = __builtin_bit_cast(bf16x8, make_uint4(xreg[q][0], xreg[q][1], xreg[q][2], xreg[q][3]));
        } else {
          uint32_t hi[4], lo[4];
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const float f0 = kq::h2f((uint16_t)(xreg[q][j] & 0xffffu)), f1 = kq::h2f((uint16_t)(xreg[q][j] >> 16));
            hi[j] = pack_hi(f0, f1);
            lo[j] = pack_hi(f0 - trunc_bf16(f0), f1 - trunc_bf16(f1));  // exact: 11 significant bits in all
          }
          ah[q] = __builtin_bit_cast(bf16x8, make_uint4(hi[0], hi[1], hi[2], hi[3]));
          al[q] = __builtin_bit_cast(bf16x8, make_uint4(lo[0], lo[1], lo[2], lo[3]));
        }
      }
      if (st + NT_WAVES < nsteps) {
        fetch_w(st + NT_WAVES);
        fetch_x(st + NT_WAVES);
      }
      // weights: rows 8h ... 8h + 7 of the step, column group of this lane, split into bf16 hi / lo and regrouped by
      // column
      uint32_t bh[8][4], bl[8][4];
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        float w0[8], w1[8];
        kq::decode8<C>(blk + (8 * h + i) * STRIDE, g, grids, w0);
        kq::decode8<C>(blk + (8 * h + i + 1) * STRIDE, g, grids, w1);
#pragma unroll
        for (int t = 0; t < 8; t++) {
          bh[t][i >> 1] = pack_hi(w0[t], w1[t]);
          bl[t][i >> 1] = pack_rne(w0[t] - trunc_bf16(w0[t]), w1[t] - trunc_bf16(w1[t]));
        }
      }
#pragma unroll
      for (int t = 0; t < 8; t++) {
        const bf16x8 wh = __builtin_bit_cast(bf16x8, make_uint4(bh[t][0], bh[t][1], bh[t][2], bh[t][3]));
        const bf16x8 wl = __builtin_bit_cast(bf16x8, make_uint4(bl[t][0], bl[t][1], bl[t][2], bl[t][3]));
#pragma unroll
        for (int q = 0; q < MR; q++) {
          acc[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[q], wh, acc[q][t], 0, 0, 0);
          acc[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[q], wl, acc[q][t], 0, 0, 0);
          if constexpr (DT == KQ_F16) acc[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[q], wh, acc[q][t], 0, 0, 0);
        }
      }
    }

    if (nsteps - st_begin > 1) {  // uniform over the workgroup: waves 2, 3 -> waves 0, 1, then wave 1 -> wave 0
      constexpr int NACC = 32 * MR;
      __syncthreads();  // every wave is done with its staging area
      float* mine = red + (size_t)(wave & 1) * NACC * 64 + lane;
      auto put = [&](float* dst) {
#pragma unroll
        for (int q = 0; q < MR; q++)
#pragma unroll
          for (int t = 0; t < 8; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) dst[((q * 8 + t) * 4 + r) * 64] = acc[q][t][r];
      };
      auto add = [&](const float* src) {
#pragma unroll
        for (int q = 0; q < MR; q++)
#pragma unroll
          for (int t = 0; t < 8; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[q][t][r] += src[((q * 8 + t) * 4 + r) * 64];
      };
      if (wave >= 2) put(mine);
      __syncthreads();
      if (wave < 2) add(mine);
      __syncthreads();
      if (wave == 1) put(red + lane);
      __syncthreads();
      if (wave == 0) add(red + lane);
    }
    if constexpr (!MERGE) {
      if (wave != 0 || !col_ok) return;
    }
    if (!MERGE && a.ksplit > 1) {
      float* pb = a.part + (size_t)split * a.M * a.N + 8 * (size_t)gi;
#pragma unroll
      for (int q = 0; q < MR; q++) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int m = m0 + 16 * q + 4 * h + r;
          if (m < a.M) {
            float4* o = reinterpret_cast<float4*>(pb + (size_t)m * a.N);
            o[0] = make_float4(acc[q][0][r], acc[q][1][r], acc[q][2][r], acc[q][3][r]);
            o[1] = make_float4(acc[q][4][r], acc[q][5][r], acc[q][6][r], acc[q][7][r]);
          }
        }
      }
      return;
    }
    uint16_t* yb = static_cast<uint16_t*>(a.y) + 8 * (size_t)gi;
    if (wave == 0 && col_ok)
#pragma unroll
    for (int q = 0; q < MR; q++) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int m = m0 + 16 * q + 4 * h + r;
        if (m < rows) {
          uint32_t o[4];
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const float v0 = acc[q][2 * j][r], v1 = acc[q][2 * j + 1][r];
            const uint16_t lo = DT == KQ_F16 ? kq::f2f16(v0) : kq::f2bf16(v0);
            const uint16_t hi = DT == KQ_F16 ? kq::f2f16(v1) : kq::f2bf16(v1);
            o[j] = (uint32_t)lo | ((uint32_t)hi << 16);
          }
          const size_t row = MERGE ? (size_t)y_row[m - m0] : (size_t)item * a.M + m;
          *reinterpret_cast<uint4*>(yb + row * a.N) = make_uint4(o[0], o[1], o[2], o[3]);
        }
      }
    }
    if constexpr (!MERGE) {
      return;
    } else {
      __syncthreads();  // the sums have been read: the staging areas may be filled again; share.left is known
      if (others || !share.left || !kqentries::shares_rounds<16 * MR>(rows, a.B, a.M, a.E, gridDim.y)) return;
      own = false;
    }
  }
}

// Many activation rows: 128 (MRW = 2) or 256 (MRW = 4) rows x 128 columns per workgroup.  Every wave owns a quarter
// of the rows and the four walk the
// K steps together, so the 4096 weights of a step are decoded ONCE per workgroup instead of once per 32 rows: wave w
// decodes rows 8w ... 8w + 7 of the step's 32 (lane (c, part): rows 8w + 2 part, + 1 of column group c), writes them
// as packed bf16 pairs where the MFMA operands of all four waves lie (LDS, [k group h][t][c] x 16 bytes, hi and lo
// planes), and after one barrier every wave reads its 16 operands back.  Staging and operand buffers are double:
// one barrier per step.
template <int C, int DT, int MRW, bool VEC>
__global__ __launch_bounds__(NT_THREADS, 2) void gemm_nt_wide_kernel(NtArgs a, const uint8_t* __restrict__ grids) {
  using G = NtGeom<C>;
  constexpr int BPB = G::BPB, GPB = G::GPB, PDW = G::PDW, STRIDE = G::STRIDE;
  constexpr int STG = NT_KSTEP * STRIDE;               // one staging buffer: the step's 32 row pieces
  constexpr int NDWW = (NT_KSTEP * PDW + NT_THREADS - 1) / NT_THREADS;  // dwords a thread copies per step
  constexpr int PLANE = 4 * 8 * 16 * 16;               // one operand plane: [h][t][c] x 16 bytes
  constexpr int OPB = 2 * PLANE;                       // hi + lo
  __shared__ __attribute__((aligned(16))) uint8_t lds[2 * STG + 2 * OPB];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c = lane & 15, h = lane >> 4;  // h: k group as operand reader, row pair as decoder
  const int item = a.ksplit > 1 ? 0 : blockIdx.z, split = a.ksplit > 1 ? blockIdx.z : 0;
  const uint32_t e = a.rhs ? a.rhs[item] : 0u;
  if (e >= (uint32_t)a.E) return;  // the whole workgroup leaves: the entry's output rows stay untouched
  const int tile = blockIdx.x;
  const int ngroups = a.N / 8;
  const int gi = tile * 16 + c;
  const bool col_ok = gi < ngroups;
  const size_t row_bytes = (size_t)(a.N / G::WPB) * BPB;
  const int pi = G::SUPER ? tile >> 1 : tile;
  const int gp = (col_ok ? gi : ngroups - 1) - pi * (G::PCOLS / 8);
  const uint8_t* wt = a.w + (size_t)e * (size_t)a.w_expert_stride + (size_t)pi * G::PIECE;
  const int cols_here = a.N - G::PCOLS * pi < G::PCOLS ? a.N - G::PCOLS * pi : G::PCOLS;
  const int piece_here = cols_here / G::WPB * BPB;
  const int blk_off = (gp / GPB) * BPB + (8 * wave + 2 * h) * STRIDE;  // this lane's first row inside a staging buffer
  const int g = gp % GPB, klast = a.K - 1;
  const int m0 = blockIdx.y * (64 * MRW) + 16 * MRW * wave;
  const uint16_t* xr[MRW];
#pragma unroll
  for (int q = 0; q < MRW; q++) {
    const int mrow = m0 + 16 * q + c < a.M ? m0 + 16 * q + c : a.M - 1;
    xr[q] = static_cast<const uint16_t*>(a.x) + (a.lhs ? (size_t)a.lhs[item] * (size_t)a.x_batch_stride : 0) +
            (size_t)mrow * a.K;
  }
  f32x4 acc[MRW][8];
#pragma unroll
  for (int q = 0; q < MRW; q++)
#pragma unroll
    for (int t = 0; t < 8; t++) acc[q][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  uint32_t wreg[NDWW], xreg[MRW][4];
  auto fetch = [&](int st) {  // as in gemm_nt_mfma_kernel, the step's pieces spread over the whole workgroup
#pragma unroll
    for (int j = 0; j < NDWW; j++) {
      const int idx = tid + NT_THREADS * j < NT_KSTEP * PDW ? tid + NT_THREADS * j : NT_KSTEP * PDW - 1;
      const int row = idx / PDW, boff = 4 * (idx - row * PDW);
      const int eoff = boff < piece_here - 4 ? boff : piece_here - 4;
      const int k = NT_KSTEP * st + row < a.K ? NT_KSTEP * st + row : klast;
      wreg[j] = *reinterpret_cast<const u32_a1*>(wt + (size_t)k * row_bytes + eoff);
    }
    const int k0 = NT_KSTEP * st + 8 * h;
#pragma unroll
    for (int q = 0; q < MRW; q++) {
      if constexpr (VEC) {
        const uint4 v = *reinterpret_cast<const uint4*>(xr[q] + (k0 < a.K ? k0 : 0));
        xreg[q][0] = v.x, xreg[q][1] = v.y, xreg[q][2] = v.z, xreg[q][3] = v.w;
      } else {
#pragma unroll
        for (int j = 0; j < 4; j++) xreg[q][j] = 0u;
#pragma unroll
        for (int i = 0; i < 8; i++)
          if (k0 + i < a.K) xreg[q][i >> 1] |= (uint32_t)xr[q][k0 + i] << (16 * (i & 1));
      }
    }
  };
  auto park = [&](uint8_t* stage) {
#pragma unroll
    for (int j = 0; j < NDWW; j++) {
      const int idx = tid + NT_THREADS * j;
      const int boff = 4 * (idx % PDW), eoff = boff < piece_here - 4 ? boff : piece_here - 4;
      if (idx < NT_KSTEP * PDW) *reinterpret_cast<uint32_t*>(stage + 4 * idx) = wreg[j] >> (8 * ((boff - eoff) & 3));
    }
  };

  const int steps_all = (a.K + NT_KSTEP - 1) / NT_KSTEP;
  const int st_begin = split * a.steps_per_split;
  const int nsteps = st_begin + a.steps_per_split < steps_all ? st_begin + a.steps_per_split : steps_all;
  if (st_begin < nsteps) {
    fetch(st_begin);
    park(lds);
  }
  for (int st = st_begin; st < nsteps; st++) {
    const int b = (st - st_begin) & 1;
    const uint8_t* stage = lds + b * STG;
    uint8_t* opnd = lds + 2 * STG + b * OPB;
    bf16x8 ah[MRW], al[MRW];
#pragma unroll
    for (int q = 0; q < MRW; q++) {
      if (VEC && NT_KSTEP * st + NT_KSTEP > a.K && NT_KSTEP * st + 8 * h >= a.K) xreg[q][0] = xreg[q][1] = xreg[q][2] = xreg[q][3] = 0u;
      if constexpr (DT == KQ_BF16) {
        ah[q] = __builtin_bit_cast(bf16x8, make_uint4(xreg[q][0], xreg[q][1], xreg[q][2], xreg[q][3]));
      } else {
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const float f0 = kq::h2f((uint16_t)(xreg[q][j] & 0xffffu)), f1 = kq::h2f((uint16_t)(xreg[q][j] >> 16));
          hi[j] = pack_hi(f0, f1);
          lo[j] = pack_hi(f0 - trunc_bf16(f0), f1 - trunc_bf16(f1));
        }
        ah[q] = __builtin_bit_cast(bf16x8, make_uint4(hi[0], hi[1], hi[2], hi[3]));
        al[q] = __builtin_bit_cast(bf16x8, make_uint4(lo[0], lo[1], lo[2], lo[3]));
      }
    }
    if (st == st_begin) __syncthreads();  // the first staging buffer is complete (later ones: the barrier below)
    // Under a branch, unlike the 256-row kernel's: as one block of code with the decode (the last step fetched again) the codecs of
    // short decode lost a tenth.  us, one block / branch: q8_0 600 rows 4096 x 14336 (reduction x outputs) 277 / 246, 128 rows
    // 14336 x 4096 67 / 56, q6_k 2048 rows 4096 x 4096 252 / 222, q4_0 96 ... 511 rows 0.94 of it, q4_k level
    if (st + 1 < nsteps) fetch(st + 1);
    {  // decode this lane's two rows and put them where the operands lie
      float w0[8], w1[8];
      kq::decode8<C>(stage + blk_off, g, grids, w0);
      kq::decode8<C>(stage + blk_off + STRIDE, g, grids, w1);
      uint8_t* dst = opnd + ((wave * 8) * 16 + c) * 16 + 4 * h;
#pragma unroll
      for (int t = 0; t < 8; t++) {
        *reinterpret_cast<uint32_t*>(dst + t * 256) = pack_hi(w0[t], w1[t]);
        *reinterpret_cast<uint32_t*>(dst + t * 256 + PLANE) =
            pack_rne(w0[t] - trunc_bf16(w0[t]), w1[t] - trunc_bf16(w1[t]));
      }
    }
    if (st + 1 < nsteps) park(lds + (b ^ 1) * STG);
    __syncthreads();  // operands of this step are complete; the other staging buffer is written
    const uint8_t* src = opnd + ((h * 8) * 16 + c) * 16;
#pragma unroll
    for (int t = 0; t < 8; t++) {
      const bf16x8 wh = *reinterpret_cast<const bf16x8*>(src + t * 256);
      const bf16x8 wl = *reinterpret_cast<const bf16x8*>(src + t * 256 + PLANE);
#pragma unroll
      for (int q = 0; q < MRW; q++) {
        acc[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[q], wh, acc[q][t], 0, 0, 0);
        acc[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[q], wl, acc[q][t], 0, 0, 0);
        if constexpr (DT == KQ_F16) acc[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[q], wh, acc[q][t], 0, 0, 0);
      }
    }
  }

  if (!col_ok) return;
  if (a.ksplit > 1) {
    float* pb = a.part + (size_t)split * a.M * a.N + 8 * (size_t)gi;
#pragma unroll
    for (int q = 0; q < MRW; q++) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int m = m0 + 16 * q + 4 * h + r;
        if (m < a.M) {
          float4* o = reinterpret_cast<float4*>(pb + (size_t)m * a.N);
          o[0] = make_float4(acc[q][0][r], acc[q][1][r], acc[q][2][r], acc[q][3][r]);
          o[1] = make_float4(acc[q][4][r], acc[q][5][r], acc[q][6][r], acc[q][7][r]);
        }
      }
    }
    return;
  }
  uint16_t* yb = static_cast<uint16_t*>(a.y) + (size_t)item * a.M * a.N + 8 * (size_t)gi;
#pragma unroll
  for (int q = 0; q < MRW; q++) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = m0 + 16 * q + 4 * h + r;
      if (m < a.M) {
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const float v0 = acc[q][2 * j][r], v1 = acc[q][2 * j + 1][r];
          const uint16_t lo = DT == KQ_F16 ? kq::f2f16(v0) : kq::f2bf16(v0);
          const uint16_t hi = DT == KQ_F16 ? kq::f2f16(v1) : kq::f2bf16(v1);
          o[j] = (uint32_t)lo | ((uint32_t)hi << 16);
        }
        *reinterpret_cast<uint4*>(yb + (size_t)m * a.N) = make_uint4(o[0], o[1], o[2], o[3]);
      }
    }
  }
}

// Many activation rows: 256 rows x 128 columns per workgroup of eight waves, 64 rows of K a step.  The 8192 weights of a
// step are decoded once for all 256 rows: wave w decodes rows 8w ... 8w + 7 of the step's 64 (lane (c, h): rows 8w + 2h,
// + 1 of column group c) into operand order as above.  A wave multiplies 64 rows with half of the columns (t = 4 wc ...
// 4 wc + 3), so an operand read feeds eight MFMAs and is made by four waves instead of by all.  Operands of step s + 1
// are decoded in the interval that multiplies step s, the two waves of a SIMD in opposite order, so that one decodes
// while the other multiplies; wire bytes are two steps ahead, one barrier per step.
// The step's activations come with direct-to-LDS loads one step ahead, rows 128 bytes apart with 16-byte piece p of row r at place
// p ^ (r & 7): two waves share a row, and no register waits for them.  (Loaded into registers by each wave, 64-byte pieces of 16 rows
// a load, they cost a quarter of the time: 4096 x 4096, us, q4_k 1024 / 2048 rows 118 / 185 -> 96 / 149, q8_0 110 / 185 -> 86 / 138,
// q6_k 122 / 207 -> 101 / 165.)  146 - 157 KB of LDS: one workgroup per CU.
// Bound by the stages of a step one after another: leaving out one (timing only, before the change above) gave 15 % for the decode, 4 for the
// wire loads, 12 for the second bf16 term's products.  8-byte instead of byte-wise LDS reads in the K-quant decoders
// gave 2 % on q4_k, 0 on q5_k and q6_k, and spilled in the narrow kernels: not kept.  128-row tiles of the same form were
// slower: 124 and 246 us (q4_k 1024 and 2048 rows, against 108 and 180 then).
constexpr int TALL_WAVES = 8, TALL_THREADS = 64 * TALL_WAVES, TALL_K = 64, TALL_RG = 4;

template <int C, int DT>
__global__ __launch_bounds__(TALL_THREADS, 2) void gemm_nt_tall_kernel(NtArgs a, const uint8_t* __restrict__ grids) {
  using G = NtGeom<C>;
  constexpr int BPB = G::BPB, GPB = G::GPB, PDW = G::PDW, STRIDE = G::STRIDE, RG = TALL_RG;
  constexpr int STG = TALL_K * STRIDE;                                      // one staging buffer: the step's row pieces
  constexpr int NDWW = (TALL_K * PDW + TALL_THREADS - 1) / TALL_THREADS;    // dwords a thread copies per step
  constexpr int PLANE = (TALL_K / 8) * 8 * 16 * 16;                         // one operand plane
  constexpr int OPB = 2 * PLANE;                                            // hi + lo
  constexpr int XB = 64 * RG * 2 * TALL_K;                                  // the step's activations
  __shared__ __attribute__((aligned(16))) uint8_t lds[2 * STG + 2 * OPB + 2 * XB];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave & 3, wc = wave >> 2;
  const int c = lane & 15, h = lane >> 4;  // h: k group as operand reader, row pair as decoder
  const int item = a.ksplit > 1 ? 0 : blockIdx.z, split = a.ksplit > 1 ? blockIdx.z : 0;
  const uint32_t e = a.rhs ? a.rhs[item] : 0u;
  if (e >= (uint32_t)a.E) return;  // the whole workgroup leaves: the entry's output rows stay untouched
  const int tile = blockIdx.x;
  const int ngroups = a.N / 8;
  const int gi = tile * 16 + c;
  const bool col_ok = gi < ngroups;
  const size_t row_bytes = (size_t)(a.N / G::WPB) * BPB;
  const int pi = G::SUPER ? tile >> 1 : tile;
  const int gp = (col_ok ? gi : ngroups - 1) - pi * (G::PCOLS / 8);
  const uint8_t* wt = a.w + (size_t)e * (size_t)a.w_expert_stride + (size_t)pi * G::PIECE;
  const int cols_here = a.N - G::PCOLS * pi < G::PCOLS ? a.N - G::PCOLS * pi : G::PCOLS;
  const int piece_here = cols_here / G::WPB * BPB;
  const int blk_off = (gp / GPB) * BPB + (8 * wave + 2 * h) * STRIDE;  // this lane's first row inside a staging buffer
  const int g = gp % GPB, klast = a.K - 1;
  const int m0 = blockIdx.y * (64 * RG) + 16 * RG * wr;
  const uint8_t* xr[RG];  // this lane's rows of the wave's four loads of 8 rows
#pragma unroll
  for (int q = 0; q < RG; q++) {
    const int mrow = blockIdx.y * (64 * RG) + 32 * wave + 8 * q + (lane >> 3);
    xr[q] = reinterpret_cast<const uint8_t*>(static_cast<const uint16_t*>(a.x) + (a.lhs ? (size_t)a.lhs[item] * (size_t)a.x_batch_stride : 0) +
                                             (size_t)(mrow < a.M ? mrow : a.M - 1) * a.K);
  }
  const int xpiece = (lane & 7) ^ (lane >> 3);  // 16-byte piece p of a row lies at place p ^ (row & 7)
  f32x4 acc[RG][4];
#pragma unroll
  for (int q = 0; q < RG; q++)
#pragma unroll
    for (int t = 0; t < 4; t++) acc[q][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  uint32_t wreg[NDWW];
  auto fetch_w = [&](int st) {  // as in gemm_nt_mfma_kernel, the step's pieces spread over the whole workgroup
#pragma unroll
    for (int j = 0; j < NDWW; j++) {
      const int idx = tid + TALL_THREADS * j < TALL_K * PDW ? tid + TALL_THREADS * j : TALL_K * PDW - 1;
      const int row = idx / PDW, boff = 4 * (idx - row * PDW);
      const int eoff = boff < piece_here - 4 ? boff : piece_here - 4;
      const int k = TALL_K * st + row < a.K ? TALL_K * st + row : klast;
      wreg[j] = *reinterpret_cast<const u32_a1*>(wt + (size_t)k * row_bytes + eoff);
    }
  };
  auto park = [&](uint8_t* stage) {
#pragma unroll
    for (int j = 0; j < NDWW; j++) {
      const int idx = tid + TALL_THREADS * j;
      const int boff = 4 * (idx % PDW), eoff = boff < piece_here - 4 ? boff : piece_here - 4;
      if (idx < TALL_K * PDW) *reinterpret_cast<uint32_t*>(stage + 4 * idx) = wreg[j] >> (8 * ((boff - eoff) & 3));
    }
  };
  uint8_t* const xs = lds + 2 * STG + 2 * OPB;
  const uint32_t xs_lds = kqdma::lds_addr(xs) + 4096 * (uint32_t)__builtin_amdgcn_readfirstlane(wave);
  auto fetch_x = [&](int st, int b) {
    const int k = TALL_K * st + 8 * xpiece;
    const int koff = k < a.K ? 2 * k : 0;  // K is a multiple of 8: a group of 8 lies inside the row or past it (masked by multiply)
#pragma unroll
    for (int q = 0; q < RG; q++) kqdma::dma16_at(xr[q] + koff, xs_lds + b * XB + 1024 * q);
  };
  auto decode = [&](const uint8_t* stage, uint8_t* opnd) {
    float w0[8], w1[8];
    kq::decode8<C>(stage + blk_off, g, grids, w0);
    kq::decode8<C>(stage + blk_off + STRIDE, g, grids, w1);
    uint8_t* dst = opnd + ((wave * 8) * 16 + c) * 16 + 4 * h;
#pragma unroll
    for (int t = 0; t < 8; t++) {
      *reinterpret_cast<uint32_t*>(dst + t * 256) = pack_hi(w0[t], w1[t]);
      *reinterpret_cast<uint32_t*>(dst + t * 256 + PLANE) = pack_rne(w0[t] - trunc_bf16(w0[t]), w1[t] - trunc_bf16(w1[t]));
    }
  };
  auto multiply = [&](int st, const uint8_t* opnd, const uint8_t* xb) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
      if (s && TALL_K * st + 32 >= a.K) break;  // rows past K are multiplied (by zero) up to the next multiple of 32 only
      bf16x8 ah[RG], al[RG];
#pragma unroll
      for (int q = 0; q < RG; q++) {
        const uint4 xv = *reinterpret_cast<const uint4*>(xb + (16 * RG * wr + 16 * q + c) * (2 * TALL_K) + 16 * ((4 * s + h) ^ (c & 7)));
        uint32_t v[4] = {xv.x, xv.y, xv.z, xv.w};
        if (TALL_K * st + TALL_K > a.K && TALL_K * st + 32 * s + 8 * h >= a.K) v[0] = v[1] = v[2] = v[3] = 0u;
        if constexpr (DT == KQ_BF16) {
          ah[q] = __builtin_bit_cast(bf16x8, make_uint4(v[0], v[1], v[2], v[3]));
        } else {
          uint32_t hi[4], lo[4];
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const float f0 = kq::h2f((uint16_t)(v[j] & 0xffffu)), f1 = kq::h2f((uint16_t)(v[j] >> 16));
            hi[j] = pack_hi(f0, f1);
            lo[j] = pack_hi(f0 - trunc_bf16(f0), f1 - trunc_bf16(f1));
          }
          ah[q] = __builtin_bit_cast(bf16x8, make_uint4(hi[0], hi[1], hi[2], hi[3]));
          al[q] = __builtin_bit_cast(bf16x8, make_uint4(lo[0], lo[1], lo[2], lo[3]));
        }
      }
      const uint8_t* src = opnd + (((4 * s + h) * 8 + 4 * wc) * 16 + c) * 16;
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const bf16x8 wh = *reinterpret_cast<const bf16x8*>(src + t * 256);
        const bf16x8 wl = *reinterpret_cast<const bf16x8*>(src + t * 256 + PLANE);
#pragma unroll
        for (int q = 0; q < RG; q++) acc[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[q], wh, acc[q][t], 0, 0, 0);
#pragma unroll
        for (int q = 0; q < RG; q++) acc[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[q], wl, acc[q][t], 0, 0, 0);
        if constexpr (DT == KQ_F16) {
#pragma unroll
          for (int q = 0; q < RG; q++) acc[q][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[q], wh, acc[q][t], 0, 0, 0);
        }
      }
    }
  };

  const int steps_all = (a.K + TALL_K - 1) / TALL_K;
  const int st_begin = split * a.steps_per_split;
  const int nsteps = st_begin + a.steps_per_split < steps_all ? st_begin + a.steps_per_split : steps_all;
  uint8_t* const ops = lds + 2 * STG;
  if (st_begin < nsteps) {
    fetch_x(st_begin, 0);
    fetch_w(st_begin);
    park(lds);
    if (st_begin + 1 < nsteps) fetch_w(st_begin + 1);
    __syncthreads();
    decode(lds, ops);
    if (st_begin + 1 < nsteps) park(lds + STG);
    kqdma::vmwait<0>();
    __syncthreads();
  }
  for (int st = st_begin; st < nsteps; st++) {
    const int b = (st - st_begin) & 1;
    // (no branch around the loads: past the range they repeat its last step)
    fetch_x(st + 1 < nsteps ? st + 1 : nsteps - 1, b ^ 1);
    fetch_w(st + 2 < nsteps ? st + 2 : nsteps - 1);
    // read here: staging of step st + 1, operands and activations of st.  Written here: operands and activations of st + 1, staging
    // of st + 2, whose buffers were last read before the previous barrier
    if (wc == 0) {
      multiply(st, ops + b * OPB, xs + b * XB);
      if (st + 1 < nsteps) decode(lds + (b ^ 1) * STG, ops + (b ^ 1) * OPB);
    } else {
      if (st + 1 < nsteps) decode(lds + (b ^ 1) * STG, ops + (b ^ 1) * OPB);
      multiply(st, ops + b * OPB, xs + b * XB);
    }
    if (st + 2 < nsteps) park(lds + b * STG);
    kqdma::vmwait<0>();
    __syncthreads();
  }

  if (!col_ok) return;
  const size_t col = 8 * (size_t)gi + 4 * wc;
#pragma unroll
  for (int q = 0; q < RG; q++) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = m0 + 16 * q + 4 * h + r;
      if (m < a.M) {
        if (a.ksplit > 1) {
          *reinterpret_cast<float4*>(a.part + ((size_t)split * a.M + m) * a.N + col) =
              make_float4(acc[q][0][r], acc[q][1][r], acc[q][2][r], acc[q][3][r]);
        } else {
          uint32_t o[2];
#pragma unroll
          for (int j = 0; j < 2; j++) {
            const float v0 = acc[q][2 * j][r], v1 = acc[q][2 * j + 1][r];
            const uint16_t lo = DT == KQ_F16 ? kq::f2f16(v0) : kq::f2bf16(v0);
            const uint16_t hi = DT == KQ_F16 ? kq::f2f16(v1) : kq::f2bf16(v1);
            o[j] = (uint32_t)lo | ((uint32_t)hi << 16);
          }
          *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.y) + ((size_t)item * a.M + m) * a.N + col) = make_uint2(o[0], o[1]);
        }
      }
    }
  }
}

// y[i] = sum over the K ranges of part[s][i], 8 outputs per thread, ranges added in order
template <int DT>
__global__ __launch_bounds__(256) void nt_reduce_kernel(const float* __restrict__ part, void* __restrict__ y,
                                                        size_t groups, int ksplit) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= groups) return;
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < ksplit; s++) {
    const float4* p = reinterpret_cast<const float4*>(part + ((size_t)s * groups + i) * 8);
    const float4 lo = p[0], hi = p[1];
    v[0] += lo.x, v[1] += lo.y, v[2] += lo.z, v[3] += lo.w, v[4] += hi.x, v[5] += hi.y, v[6] += hi.z, v[7] += hi.w;
  }
  uint32_t o[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const uint16_t lo = DT == KQ_F16 ? kq::f2f16(v[2 * j]) : kq::f2bf16(v[2 * j]);
    const uint16_t hi = DT == KQ_F16 ? kq::f2f16(v[2 * j + 1]) : kq::f2bf16(v[2 * j + 1]);
    o[j] = (uint32_t)lo | ((uint32_t)hi << 16);
  }
  reinterpret_cast<uint4*>(y)[i] = make_uint4(o[0], o[1], o[2], o[3]);
}

// K ranges of a dense call.  256-row tiles: one workgroup per CU.  Otherwise enough workgroups for two per CU (8192 x 8192,
// 500 rows, 256 tiles in two ranges: q8_0 227 us, uncut 410), at least eight steps each.
int nt_ranges(int M, int N, int K, bool tall) {
  const int cols = (N + NT_COLS - 1) / NT_COLS;
  if (tall) {
    const int64_t tiles = (int64_t)cols * ((M + 64 * TALL_RG - 1) / (64 * TALL_RG));
    const int steps = (K + TALL_K - 1) / TALL_K;
    const int64_t s = std::min<int64_t>(256 / tiles, steps / 4);
    return s < 2 ? 1 : (int)s;
  }
  const int rows = M <= 16 ? 16 : M < NT_SHARED_ROWS ? 32 : 128;  // activation rows per workgroup
  const int64_t tiles = (int64_t)cols * ((M + rows - 1) / rows);
  const int steps = (K + NT_KSTEP - 1) / NT_KSTEP;
  if (tiles >= (rows == 128 ? 512 : 256) || steps < 16) return 1;
  int s = (int)((512 + tiles - 1) / tiles);
  if (s > steps / 8) s = steps / 8;
  if (s > 32) s = 32;
  return s < 2 ? 1 : s;
}

// Calls of the 256-row kernel: 512 rows and more of aligned activations, K long enough for its pipeline, and not more than
// 19 % over the 128-row kernel by the work of their busiest CU, in 64-row steps of K (that kernel takes longer for a step than the
// count says).  256-row tiles run one per CU, so an unfilled round costs a whole one, and two steps more to fill the pipeline; of the
// 128-row tiles two run per CU, each half a step per 32 rows, and a last round evens out but for a quarter.  Measured / by this,
// 256-row over 128-row kernel, middle of eight codecs, rows, reduction x outputs: 1800 4096 x 4096 0.73 / 0.96, 512 4096 x 4096 0.89 / 1.09,
// 600 8192 x 2048 0.85 / 1.09, 768 4096 x 4096 0.87 / 1.13, 1024 2048 x 6144 0.88 / 1.18, 1500 2048 x 8192 1.08 / 1.20, 1400 4096 x 4096 0.97 /
// 1.25, 8192 x 8192 1.05 / 1.25, 600 4096 x 4096 1.02 / 1.37, 4096 x 14336 1.09 / 1.52; the codecs lie within 5 % of that (q3_k 8 % above at 600 rows of 4096 x 14336).  Ranges of
// fewer than eight steps hardly leave the filling of the pipeline (2048 rows of 1024 x 1024, four steps, 1.09 / 1.33) and keep to 5 %, q2_k
// and q4_1 to -5 %.  Never for the codebook codecs, whose table reads from eight waves decoding together make the 256-row
// kernel 1.3 - 1.5 times the other (1.1 where it is best; both before activations went through LDS).
// cut: K may be cut over the grid; entries: 1 for a dense call.
constexpr bool nt_codebook(int codec) {
  return codec == KQ_IQ1_S || codec == KQ_IQ1_M || codec == KQ_IQ2_XXS || codec == KQ_IQ2_XS || codec == KQ_IQ2_S ||
         codec == KQ_IQ3_XXS || codec == KQ_IQ3_S;
}
bool nt_tall(int codec, int M, int N, int K, bool cut, int entries) {
  if (M < 512 || K < 512 || (K & 7) || nt_codebook(codec)) return false;
  const int64_t cols = (int64_t)((N + NT_COLS - 1) / NT_COLS) * entries;
  const int st = cut ? nt_ranges(M, N, K, true) : 1, sw = cut ? nt_ranges(M, N, K, false) : 1;
  const int64_t tall_wgs = cols * ((M + 64 * TALL_RG - 1) / (64 * TALL_RG)) * st;
  const double rounds = (double)(cols * ((M + 127) / 128) * sw) / 512, steps = (double)K / TALL_K;
  const double tall = (double)((tall_wgs + 255) / 256) * (steps / st + 2);
  const double wide = (rounds <= 1 ? 1 : rounds + 0.25) * (steps / sw + 0.5);
  return tall <= (steps / st < 8 ? codec == KQ_Q2_K || codec == KQ_Q4_1 ? 0.95 : 1.05 : 1.19) * wide;
}

// Entries of one expert share tiles (gathered calls in which an expert comes twice on average, of a list short enough to be
// searched by every workgroup): where the rows of an entry fill half a tile at most, or a tile (two of the codec that spills
// without) and the unmerged workgroups would be more than two rounds of two per CU.  Merged / not, us, entries of 16 rows,
// four sequences: 128 heads of 128 x 512 q8_0 21.8 / 24.2, q4_k 22.6 / 27.9, 64 of 192 x 512 13.6 / 16.7, 16.4 / 21.0, but 32 of
// 128 x 256 8.6 / 6.3, 8.9 / 6.8, 16 of 192 x 512 q6_k 12.8 / 11.3; of 32 rows, two sequences, 128 heads q8_0 21.3 / 18.5, q6_k 25.0 / 30.1.
bool nt_merge(int M, int B, int E, int N, int codec, bool gathered) {
  if (!gathered || E < 1 || B < 2 * E || B > kqentries::MAX_ENTRIES) return false;
  return M <= 8 || ((M <= 16 || (M <= 32 && nt_wide(codec))) && (int64_t)B * ((N + NT_COLS - 1) / NT_COLS) >= 4 * kq_num_cus());
}

template <int C>
struct NtRun {
  template <int DT>
  static void reduce(const NtArgs& a, hipStream_t s) {
    if (a.ksplit <= 1) return;
    const size_t groups = (size_t)a.M * a.N / 8;
    hipLaunchKernelGGL((nt_reduce_kernel<DT>), dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, s, a.part, a.y, groups,
                       a.ksplit);
  }
  template <int DT, int MR, bool MERGE = false>
  static void go(const NtArgs& a, int B, const uint8_t* grids, hipStream_t s) {
    dim3 grid((a.N + NT_COLS - 1) / NT_COLS, (a.M + 16 * MR - 1) / (16 * MR), a.ksplit > 1 ? a.ksplit : B);
    if (MERGE) {
      // workgroups for the rounds of an average expert; half as many again for random ids where they all run at once
      const int64_t rows = (int64_t)B * a.M, more = (3 * rows / 2 + 16 * MR * a.E - 1) / (16 * MR * a.E);
      grid.y = (unsigned)(grid.x * a.E * more <= kq_num_cus() ? more : (rows + 16 * MR * a.E - 1) / (16 * MR * a.E));
      grid.z = a.E;
    }
    hipLaunchKernelGGL((gemm_nt_mfma_kernel<C, DT, MR, MERGE>), grid, dim3(NT_THREADS), 0, s, a, grids);
    reduce<DT>(a, s);
  }
  template <int DT, bool VEC>
  static void go_shared(const NtArgs& a, int B, const uint8_t* grids, hipStream_t s) {
    // (256-row tiles on four waves, MRW = 4, measured slower: 316 against 223 us at 2048 rows of 4096 x 4096 q4_k; their
    // 212 - 250 registers leave two workgroups per CU where the 128-row form runs three)
    dim3 grid((a.N + NT_COLS - 1) / NT_COLS, (a.M + 127) / 128, a.ksplit > 1 ? a.ksplit : B);
    hipLaunchKernelGGL((gemm_nt_wide_kernel<C, DT, 2, VEC>), grid, dim3(NT_THREADS), 0, s, a, grids);
    reduce<DT>(a, s);
  }
  template <int DT>
  static void go_tall(const NtArgs& a, int B, const uint8_t* grids, hipStream_t s) {
    dim3 grid((a.N + NT_COLS - 1) / NT_COLS, (a.M + 64 * TALL_RG - 1) / (64 * TALL_RG), a.ksplit > 1 ? a.ksplit : B);
    hipLaunchKernelGGL((gemm_nt_tall_kernel<C, DT>), grid, dim3(TALL_THREADS), 0, s, a, grids);
    reduce<DT>(a, s);
  }
  template <int DT>
  static void many_rows(const NtArgs& a, int B, const uint8_t* grids, hipStream_t s) {
    if constexpr (!nt_codebook(C))
      if (a.tall) return go_tall<DT>(a, B, grids, s);
    if (a.x_vec) go_shared<DT, true>(a, B, grids, s);
    else go_shared<DT, false>(a, B, grids, s);
  }
  static int run(const NtArgs& a, int B, int dt, const uint8_t* grids, hipStream_t s) {
    if (a.M >= NT_SHARED_ROWS) {
      dt == KQ_F16 ? many_rows<KQ_F16>(a, B, grids, s) : many_rows<KQ_BF16>(a, B, grids, s);
    } else if (nt_merge(a.M, B, a.E, a.N, C, a.rhs != nullptr)) {
      if ((int64_t)B * a.M <= 16 * (int64_t)a.E)
        dt == KQ_F16 ? go<KQ_F16, 1, true>(a, B, grids, s) : go<KQ_BF16, 1, true>(a, B, grids, s);
      else
        dt == KQ_F16 ? go<KQ_F16, 2, true>(a, B, grids, s) : go<KQ_BF16, 2, true>(a, B, grids, s);
    } else if (a.M <= 16) {
      dt == KQ_F16 ? go<KQ_F16, 1>(a, B, grids, s) : go<KQ_BF16, 1>(a, B, grids, s);
    } else if (nt_wide(C) && a.M > 32) {
      if constexpr (nt_wide(C)) dt == KQ_F16 ? go<KQ_F16, 4>(a, B, grids, s) : go<KQ_BF16, 4>(a, B, grids, s);
    } else {
      dt == KQ_F16 ? go<KQ_F16, 2>(a, B, grids, s) : go<KQ_BF16, 2>(a, B, grids, s);
    }
    KQ_HIP_CHECK(hipGetLastError());
    return KQ_OK;
  }
};

template <template <int> class F, typename... A>
int nt_dispatch(int codec, const A&... a) {
  switch (codec) {
#define KQ_CASE(c) \
  case c:          \
    return F<c>::run(a...);
    KQ_CASE(KQ_Q2_K) KQ_CASE(KQ_Q3_K) KQ_CASE(KQ_Q4_K) KQ_CASE(KQ_Q5_K) KQ_CASE(KQ_Q6_K) KQ_CASE(KQ_Q4_0)
    KQ_CASE(KQ_Q4_1) KQ_CASE(KQ_Q5_0) KQ_CASE(KQ_Q5_1) KQ_CASE(KQ_Q8_0) KQ_CASE(KQ_IQ4_NL) KQ_CASE(KQ_IQ4_XS)
    KQ_CASE(KQ_IQ3_S) KQ_CASE(KQ_IQ3_XXS) KQ_CASE(KQ_IQ2_XXS) KQ_CASE(KQ_IQ2_XS) KQ_CASE(KQ_IQ2_S)
    KQ_CASE(KQ_IQ1_S) KQ_CASE(KQ_IQ1_M) KQ_CASE(KQ_MXFP4) KQ_CASE(KQ_NVFP4)
#undef KQ_CASE
  }
  return KQ_ERR_UNSUPPORTED;
}

}  // namespace

// f32 partial sums of a dense call whose K range is cut (0: the call runs uncut)
size_t kq_nt_workspace_bytes(int M, int N, int K, int codec) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int s = nt_ranges(M, N, K, nt_tall(codec, M, N, K, true, 1));
  return s > 1 ? (size_t)s * M * N * 4 : 0;
}

// Dense (lhs = rhs = null, B = 1, E = 1) or gathered.  KQ_ERR_UNSUPPORTED (nothing launched) when the output is
// not 16-byte aligned or the grid does not fit: the caller then runs the plain vector kernel.  A dense call cuts
// its K range when `ws` holds kq_nt_workspace_bytes and is 16-byte aligned; without it the call runs uncut.
int kq_launch_nt_mfma(const void* x, const uint8_t* w, const uint32_t* lhs, const uint32_t* rhs, void* out, int B,
                      int M, int E, int N, int K, int64_t x_batch_stride, int64_t w_expert_stride, int codec, int dtype,
                      void* ws, size_t ws_bytes, hipStream_t s) {
  if (B <= 0 || M <= 0 || N <= 0 || K <= 0 || (N & 7)) return KQ_ERR_UNSUPPORTED;
  if (B > 65535 || (M + 15) / 16 > 65535) return KQ_ERR_UNSUPPORTED;
  if (reinterpret_cast<uintptr_t>(out) & 15) return KQ_ERR_UNSUPPORTED;
  const uint8_t* grids = kq_device_grids();
  if (!grids) return KQ_ERR_HIP;
  NtArgs a{x, w, out, lhs, rhs, M, N, K, E, B, x_batch_stride, w_expert_stride, 0, 1, 0, nullptr, false};
  a.x_vec = !(K & 7) && !(reinterpret_cast<uintptr_t>(x) & 15) && !(x_batch_stride & 7);
  // K is cut into the ranges that kq_nt_workspace_bytes was asked for, into what fits where unaligned activations turn the call
  // to the 128-row kernel, or not at all
  bool cut = !rhs && B == 1 && ws && !(reinterpret_cast<uintptr_t>(ws) & 15);
  a.tall = a.x_vec && nt_tall(codec, M, N, K, cut, B);
  int sp = cut ? nt_ranges(M, N, K, a.tall) : 1;
  const size_t fit = ws_bytes / ((size_t)M * N * 4);
  if ((size_t)sp > fit && sp > 1) {
    cut = fit >= 2 && !a.tall && !a.x_vec;
    sp = cut ? (int)fit : 1;
    a.tall = !cut && a.x_vec && nt_tall(codec, M, N, K, false, B);
  }
  const int kstep = a.tall ? TALL_K : NT_KSTEP, steps = (K + kstep - 1) / kstep;
  a.steps_per_split = steps;
  if (cut && sp > 1) {
    a.steps_per_split = (steps + sp - 1) / sp;
    a.ksplit = (steps + a.steps_per_split - 1) / a.steps_per_split;
    a.part = static_cast<float*>(ws);
  }
  return nt_dispatch<NtRun>(codec, a, B, dtype, grids, s);
}
