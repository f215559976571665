// Skinny-M matmul (M <= 8) on the matrix cores for the legacy, IQ and fp4 codecs:
// y[m, n] = sum_k x[m, k] W[n, k] with W in q8_0, q4_0/1, q5_0/1, iq4_nl, iq4_xs, iq3_s, iq3_xxs,
// iq2_xxs, iq2_xs, iq2_s, iq1_s, iq1_m, mxfp4 or nvfp4 wire form.
//
// Numerics.  Every one of these codecs stores a weight as (block scale) x (small code): an int8, a
// nibble minus a zero point, an entry of a 16-value table, a codebook magnitude with a sign, or a
// ternary value +- 1/8.  The codes are exact in f16, so they go into v_mfma_f32_32x32x16_f16 as they
// are, one scale block (16 or 32 weights) per accumulator set, and the block scale multiplies the f32
// partial sum afterwards: products are exact and everything else is f32, so the result differs from
// the f32 reference (src/kquant_cpu_decode.cpp:1010-1065) by summation order only.  q4_1 / q5_1 add
// their block minimum times the block's activation sum.  bf16 activations are converted to f16 per
// (row, 256-wide K step) with an exact power-of-two scale so that they cannot overflow.
//
// Tiling.  Workgroup = 8 waves that share 32 weight rows (the MFMA's 32 columns) and split K: wave w
// takes the 256-weight steps w, w + 8, ... entirely on its own -- wire bytes and activations of a step
// are fetched one step ahead with 16-byte loads and parked in wave-private LDS, so no workgroup
// barrier sits in the weight stream -- and the eight partial sums meet in LDS at the end.  Codebooks
// live in LDS as f16 tables built once per workgroup.  A lane copies its row's step bytes into
// registers with conflict-free 16-byte LDS reads and picks exactly the 8 codes its MFMA B operand
// needs (row l % 32, K half l / 32) at compile-time offsets, so nothing decoded is shared or stored.
//
// The batched MoE ops (more than 16 (token, expert) pairs) use the same decode in a workgroup-tiled
// grouped kernel (further down): 32 gathered pairs of one expert x 128 weight rows per workgroup.
#include "kq_codes.h"
#include "kq_epilogue.h"
#include "kq_moe_sort.h"

namespace {

using namespace kqcodes;

constexpr int CK_WAVES = 8;          // waves per workgroup: they share 32 weight rows and split K
constexpr int XA_STRIDE = 512 + 32;  // bytes per activation row of one step in LDS (rows 8 banks apart)
constexpr int CK_MAXM = 8;

// LDS of one wave: wire bytes of a step (32 rows), f16 activations (mb rows), row scales, block sums
template <int C>
constexpr int wave_lds_bytes(int mb) {
  return 32 * CodeGeom<C>::LROW + mb * XA_STRIDE + CK_MAXM * 4 + 8 * CK_MAXM * 4;
}

// ------------------------------------------------------------------ kernel
struct CkArgs {
  const void* x;  // [M][K]
  const uint8_t* w;
  void* y;        // [M][N]
  const uint16_t* bias;  // [N] in the activation dtype, added in f32 before the rounding; or null
  const uint8_t* grids;
  int M, N, K;
  // gathered calls (GMODE 1 / 2), one item per blockIdx.y: activation row x + (lhs ? lhs[item] : item / x_div) *
  // x_item_stride, matrix w (+ w2 for the GLU) + rhs[item] * w_expert_stride, f32 biases [E][N], output row
  // through the out map
  const uint8_t* w2;
  const uint32_t* lhs;
  const uint32_t* rhs;
  const float* fbias;
  const float* fbias2;
  int x_div, act;
  int64_t x_item_stride, w_expert_stride;
  float limit, alpha;
  KqOutMap om;
  int E;  // gathered calls: items whose expert id is >= E are skipped (output rows left untouched)
};

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Workgroup = CK_WAVES waves that share 32 weight rows and split K: wave w takes the 256-weight steps
// w, w + CK_WAVES, ... on its own (wave-private LDS buffers, no workgroup barrier in the stream), and
// the partial sums meet in LDS at the end.  MB = activation rows the LDS buffers are sized for.
// GMODE 0: one dense matrix.  GMODE 1: gathered, one (activation row, expert matrix) item per blockIdx.y.
// GMODE 2: gathered GLU: the tile's 32 rows are 16 gate rows and the same 16 up rows, the epilogue act(g) * u runs
// on the reduced sums before the single rounding.
// WV = waves per workgroup.  Gathered launches (many small workgroups, short K) need the whole grid resident at
// once: the codecs whose kernel stays under 128 registers get there with 8 waves (two workgroups per CU), the
// others use 4-wave workgroups (iq4_xs 11.9 + 8.9 -> 10.3 + 6.3 us for the GLU + down of 8 experts of 768 x 2048;
// iq1_s went the other way, 6.8 + 5.0 -> 8.1 + 5.8 us, hence the split).  Dense launches use 8 waves, except
// single-row calls of those larger kernels with more row tiles than CUs, where 4-wave workgroups measured 7 - 15 %
// faster (iq4_xs 128256 x 4096: 127 -> 110 us) and 20 - 40 % slower with fewer tiles.
template <int C>
constexpr bool ck_small() {
  return C == KQ_IQ2_XXS || C == KQ_IQ2_XS || C == KQ_IQ2_S || C == KQ_IQ1_S || C == KQ_IQ1_M;
}
template <int C, int GMODE>
constexpr int ck_waves() {
  return (GMODE && !ck_small<C>()) ? 4 : CK_WAVES;
}

template <int C, int DT, int MB, int GMODE, int WV>
__global__ __launch_bounds__((64 * WV), (WV == 4 ? 2 : 1)) void codes_skinny_kernel(CkArgs a) {
  constexpr int NWAVES = WV, NTHREADS = 64 * NWAVES;
  using G = CodeGeom<C>;
  constexpr int TILE_N = GMODE == 2 ? 16 : 32;  // output columns per workgroup
  constexpr int WPT = (32 * G::PIECES + 63) / 64;  // wire pieces per lane and step
  constexpr int XPT = MB >= 2 ? MB / 2 : 1;        // activation pieces per lane and step (rows lane / 32 + 2 t)
  constexpr int WAVE_LDS = wave_lds_bytes<C>(MB);
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  uint8_t* grid_lds = smem;
  uint8_t* spread_lds = grid_lds + G::GRID_BYTES;
  uint8_t* wave_base = spread_lds + G::SPREAD_BYTES;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, kg = lane >> 5;
  const int M = a.M, N = a.N, K = a.K;
  const int nsteps = (K + CK_STEP - 1) / CK_STEP;
  const size_t row_bytes = (size_t)(K / G::WPB) * G::BPB;
  const int n0 = blockIdx.x * TILE_N;
  const int ncols = N - n0 < TILE_N ? N - n0 : TILE_N;
  const int item = GMODE ? (int)blockIdx.y : 0;
  const uint32_t expert = GMODE ? a.rhs[item] : 0u;
  if (GMODE && expert >= (uint32_t)a.E) return;  // uniform over the workgroup, ahead of every barrier
  const uint8_t* wmat = a.w + (GMODE ? (size_t)expert * (size_t)a.w_expert_stride : 0);
  const uint8_t* wmat2 = GMODE == 2 ? a.w2 + (size_t)expert * (size_t)a.w_expert_stride : wmat;
  const uint8_t* w_last = wmat + (size_t)N * row_bytes - 16;    // the last 16 bytes of the matrix
  const uint8_t* w_last2 = wmat2 + (size_t)N * row_bytes - 16;

  uint8_t* b_lds = wave_base + wave * WAVE_LDS;                                    // [32][LROW] wire bytes of the step
  uint8_t* a_lds = b_lds + 32 * G::LROW;                                           // [MB][XA_STRIDE] f16 activations
  float* xs_lds = reinterpret_cast<float*>(a_lds + MB * XA_STRIDE);                // [8] activation scale per row
  float* xsum_lds = xs_lds + CK_MAXM;                                              // [8 blocks][8 rows] (HAS_MIN)

  // ---- tables (whole workgroup)
  build_tables<C, NTHREADS, false>(grid_lds, spread_lds, a.grids, tid);
  if constexpr (G::GRID_N > 0 || G::SPREAD_BYTES > 0 || G::PAIR_LUT) lds_barrier();
  const Tables tabs{grid_lds, spread_lds, 2};

  // ---- piece maps of this wave.  Wire: piece i = lane + 64 t -> (row i / PIECES, piece i % PIECES).
  // Activations: lane -> (row lane / 32 + 2 t, 16-byte piece lane % 32).
  const uint8_t* w_src[WPT];
  uint32_t w_loff[WPT];
  bool w_up[WPT];
#pragma unroll
  for (int t = 0; t < WPT; t++) {
    const int i = lane + 64 * t;
    const int r = i / G::PIECES, pc = i % G::PIECES;
    const int col = GMODE == 2 ? (r & 15) : r;  // GLU: LDS rows 0..15 gate, 16..31 up
    w_up[t] = GMODE == 2 && (r & 16);
    const bool ok = col < ncols;  // rows past N (and pieces past the tile) re-read the tile's first row
    w_src[t] = (w_up[t] ? wmat2 : wmat) + (size_t)(n0 + (ok ? col : 0)) * row_bytes + 16 * pc;
    w_loff[t] = r < 32 ? (uint32_t)r * G::LROW + 16 * pc : 0xffffffffu;
  }
  const int a_row0 = lane >> 5, a_pc = lane & 31;
  const uint16_t* a_src = static_cast<const uint16_t*>(a.x) + 8 * a_pc +
                          (GMODE ? (size_t)(a.lhs ? a.lhs[item] : (uint32_t)(item / a.x_div)) * (size_t)a.x_item_stride : 0);

  u32x4 areg[XPT], wreg[WPT];
  auto issue = [&](int st) {
    const int kvalid = K - CK_STEP * st;  // weights of this step that exist (>= 256 except in the last step)
#pragma unroll
    for (int t = 0; t < XPT; t++) {
      const int row = a_row0 + 2 * t;
      u32x4 av = {0, 0, 0, 0};
      if (row < M && row < MB && 8 * a_pc < kvalid)
        av = *reinterpret_cast<const u32x4*>(a_src + (size_t)row * K + (size_t)CK_STEP * st);
      areg[t] = av;
    }
#pragma unroll
    for (int t = 0; t < WPT; t++) {
      // Pieces past the step's valid bytes (last step of a ragged K, last piece of a row) carry bytes
      // that no MFMA reads; only the end of the matrix needs care: there the 16 bytes ending at the
      // matrix end are loaded instead and shifted down, so nothing past the end is ever read.
      const uint8_t* p = w_src[t] + (size_t)st * G::BYTES;
      const uint8_t* end = (GMODE == 2 && w_up[t]) ? w_last2 : w_last;
      const uint8_t* q = p <= end ? p : end;
      u32x4 v = *reinterpret_cast<const u32x4_a1*>(q);
      if (q != p) v = shr_bytes(v, (uint32_t)(p - q));
      wreg[t] = v;
    }
  };
  auto park = [&]() {
#pragma unroll
    for (int t = 0; t < XPT; t++) {
      const int row = a_row0 + 2 * t;
      if (MB == 1 && lane >= 32) break;
      // activations: f16 as given, bf16 scaled into f16 range by a power of two per (row, step)
      float xscale = 1.f;
      _Float16 h[8];
      if constexpr (DT == KQ_BF16) {
        float amax = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          amax = fmaxf(amax, fabsf(__builtin_bit_cast(float, areg[t][e] << 16)));
          amax = fmaxf(amax, fabsf(__builtin_bit_cast(float, areg[t][e] & 0xffff0000u)));
        }
#pragma unroll
        for (int off = 16; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));  // the row's 32 lanes
        float inv = 1.f;
        const uint32_t eb = (__builtin_bit_cast(uint32_t, amax) >> 23) & 0xff;
        if (eb != 0 && eb != 0xff) {
          int e = (int)eb - 127 - 14;  // the largest magnitude lands in [2^14, 2^15)
          if (e < -100) e = -100;
          xscale = __builtin_bit_cast(float, (uint32_t)(127 + e) << 23);
          inv = __builtin_bit_cast(float, (uint32_t)(127 - e) << 23);
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
          h[2 * e] = (_Float16)(__builtin_bit_cast(float, areg[t][e] << 16) * inv);
          h[2 * e + 1] = (_Float16)(__builtin_bit_cast(float, areg[t][e] & 0xffff0000u) * inv);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          h[2 * e] = __builtin_bit_cast(_Float16, (uint16_t)(areg[t][e] & 0xffff));
          h[2 * e + 1] = __builtin_bit_cast(_Float16, (uint16_t)(areg[t][e] >> 16));
        }
      }
      stage_group<G::PAIR_LUT>(a_lds + row * XA_STRIDE, a_pc, h);
      if (a_pc == 0) xs_lds[row] = xscale;
      if constexpr (G::HAS_MIN) {
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++) sum += (float)h[e];
        sum += __shfl_xor(sum, 1);
        sum += __shfl_xor(sum, 2);  // 4 lanes = one 32-weight block
        if ((a_pc & 3) == 0) xsum_lds[(a_pc >> 2) * CK_MAXM + row] = sum;
      }
    }
#pragma unroll
    for (int t = 0; t < WPT; t++)
      if (w_loff[t] != 0xffffffffu) *reinterpret_cast<u32x4*>(b_lds + w_loff[t]) = wreg[t];
  };

  float acc[4] = {0.f, 0.f, 0.f, 0.f};  // output rows 4 kg + i of weight row n0 + l32
  const uint8_t* b_lane = b_lds + l32 * G::LROW;
  const uint8_t* a_lane = a_lds + (l32 & (MB - 1)) * XA_STRIDE + 16 * kg;
  if (lane < CK_MAXM) xs_lds[lane] = 0.f;  // rows past MB keep a zero scale

  if (wave < nsteps) issue(wave);
  for (int st = wave; st < nsteps; st += NWAVES) {
    park();
    wave_sync();
    if (st + NWAVES < nsteps) issue(st + NWAVES);
    const int kvalid = K - CK_STEP * st;
    float sacc[4] = {0.f, 0.f, 0.f, 0.f};
    constexpr int MPS = G::SB / 16;  // MFMAs per scale block
    // FULL: all 16 MFMAs of the step, branch-free so that decode, MFMA and scaling of neighbouring
    // blocks overlap; otherwise (the last step of a K that is not a multiple of 256) MFMA by MFMA.
    auto run_step = [&](auto full_c) {
      constexpr bool FULL = decltype(full_c)::value;
      f32x16 part[2];
      RowRegs<4 * G::PIECES> row;
      StaticFor<G::PIECES>::run([&](auto pc) {
        constexpr int P = decltype(pc)::value;
        const u32x4 v = *reinterpret_cast<const u32x4*>(b_lane + 16 * P);
        row.d[4 * P] = v[0];
        row.d[4 * P + 1] = v[1];
        row.d[4 * P + 2] = v[2];
        row.d[4 * P + 3] = v[3];
      });
      StaticFor<16>::run([&](auto jc) {
        constexpr int J = decltype(jc)::value;
        if (FULL || 16 * J < kvalid) {  // uniform
          const f16x8 bv = codes<C, J>(row, kg, tabs);
          // activation rows past M hold zeros or another row's values: they only reach output rows that
          // are never stored
          const f16x8 av = *reinterpret_cast<const f16x8*>(a_lane + 32 * J);
          constexpr int sbi = J / MPS, slot = sbi & 1;
          if constexpr (J % MPS == 0)
            part[slot] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, f32x16{0}, 0, 0, 0);
          else
            part[slot] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, part[slot], 0, 0, 0);
          if constexpr (J % MPS == MPS - 1) {
            float mn;
            const float sc = block_scale<C, sbi>(row, mn);
#pragma unroll
            for (int i = 0; i < 4; i++) sacc[i] = fmaf(sc, part[slot][i], sacc[i]);
            if constexpr (G::HAS_MIN) {
              const float4 xm = *reinterpret_cast<const float4*>(xsum_lds + sbi * CK_MAXM + 4 * kg);
              sacc[0] = fmaf(mn, xm.x, sacc[0]);
              sacc[1] = fmaf(mn, xm.y, sacc[1]);
              sacc[2] = fmaf(mn, xm.z, sacc[2]);
              sacc[3] = fmaf(mn, xm.w, sacc[3]);
            }
          }
        }
      });
    };
    if (kvalid >= CK_STEP)
      run_step(std::true_type{});
    else
      run_step(std::false_type{});
    const float4 xs4 = *reinterpret_cast<const float4*>(xs_lds + 4 * kg);
    acc[0] = fmaf(xs4.x, sacc[0], acc[0]);
    acc[1] = fmaf(xs4.y, sacc[1], acc[1]);
    acc[2] = fmaf(xs4.z, sacc[2], acc[2]);
    acc[3] = fmaf(xs4.w, sacc[3], acc[3]);
    wave_sync();  // this wave's reads of the step are done before the next park overwrites it
  }

  // ---- the waves' partial sums meet in LDS (the step buffers are free now)
  lds_barrier();
  float* red = reinterpret_cast<float*>(wave_base);  // [NWAVES][4][64]
#pragma unroll
  for (int i = 0; i < 4; i++) red[(wave * 4 + i) * 64 + lane] = acc[i];
  lds_barrier();
  if (wave == 0) {
    const int n = n0 + l32;
    uint16_t* y = static_cast<uint16_t*>(a.y);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < NWAVES; w++) v += red[(w * 4 + i) * 64 + lane];
      const int m = 4 * kg + i;
      if constexpr (GMODE == 0) {
        if (m < M && n < N) {
          if (a.bias) v += DT == KQ_F16 ? kq::h2f(a.bias[n]) : kq::bf162f(a.bias[n]);
          y[(size_t)m * N + n] = DT == KQ_F16 ? kq::f2f16(v) : kq::f2bf16(v);
        }
      } else if constexpr (GMODE == 1) {
        if (m < M && n < N) {
          if (a.fbias) v += a.fbias[(size_t)expert * N + n];
          kq::store_result<DT>(a.y, a.om, ((size_t)kq::out_row(a.om, item) * M + m) * N + n, v);
        }
      } else {
        float u = 0.f;  // the up row of this column sits 16 lanes further on
#pragma unroll
        for (int w = 0; w < NWAVES; w++) u += red[(w * 4 + i) * 64 + (lane ^ 16)];
        if (l32 < 16 && m < M && l32 < ncols) {
          if (a.fbias) v += a.fbias[(size_t)expert * N + n];
          if (a.fbias2) u += a.fbias2[(size_t)expert * N + n];
          v = kq::glu_epilogue(a.act, v, u, a.limit, a.alpha);
          kq::store_result<DT>(a.y, a.om, ((size_t)kq::out_row(a.om, item) * M + m) * N + n, v);
        }
      }
    }
  }
}

template <int C, int DT, int MB, int GMODE, int NWAVES>
int launch_codes_wv(const CkArgs& a, hipStream_t s, int items) {
  using G = CodeGeom<C>;
  size_t lds = (size_t)G::GRID_BYTES + G::SPREAD_BYTES + (size_t)NWAVES * wave_lds_bytes<C>(MB);
  const size_t red = (size_t)G::GRID_BYTES + G::SPREAD_BYTES + NWAVES * 4 * 64 * 4;
  if (lds < red) lds = red;
  auto kern = codes_skinny_kernel<C, DT, MB, GMODE, NWAVES>;
  KQ_SET_MAX_LDS_ONCE((kern), lds);
  constexpr int TILE_N = GMODE == 2 ? 16 : 32;
  hipLaunchKernelGGL(kern, dim3((a.N + TILE_N - 1) / TILE_N, items), dim3(64 * NWAVES), lds, s, a);
  KQ_HIP_CHECK(hipGetLastError());
  return KQ_OK;
}

template <int C, int DT, int MB, int GMODE = 0>
int launch_codes(const CkArgs& a, hipStream_t s, int items = 1) {
  if constexpr (GMODE == 0 && MB == 1 && !ck_small<C>()) {
    if ((a.N + 31) / 32 > 256) return launch_codes_wv<C, DT, MB, GMODE, 4>(a, s, items);
  }
  return launch_codes_wv<C, DT, MB, GMODE, ck_waves<C, GMODE>()>(a, s, items);
}

template <int C>
int launch_codes_dt(const CkArgs& a, int dtype, hipStream_t s) {
  const int mb = a.M <= 1 ? 1 : a.M <= 2 ? 2 : a.M <= 4 ? 4 : 8;
#define KQ_MB(m)                                                                               \
  if (mb == m)                                                                                 \
    return dtype == KQ_F16 ? launch_codes<C, KQ_F16, m>(a, s) : launch_codes<C, KQ_BF16, m>(a, s);
  KQ_MB(1) KQ_MB(2) KQ_MB(4) KQ_MB(8)
#undef KQ_MB
  return KQ_ERR_UNSUPPORTED;
}

// ------------------------------------------------------------------ grouped kernel (batched MoE)
// Pairs sorted by expert and cut into segments of at most 32 pairs of one expert (codes_prepass_kernel).  A
// workgroup multiplies a segment's gathered activation rows (the MFMA's 32 rows) by a 128-row slab of that
// expert's wire: 4 waves x 32 weight rows, one 256-weight step at a time, wire bytes and activations
// fetched one step ahead and parked in LDS.  GLU: the slab is 64 gate rows + the same 64 up rows (waves
// 0 / 2 gate, 1 / 3 up); the up waves hand their sums to the gate waves through LDS and the epilogue runs
// before the single rounding.  Same code extraction and block-scale-after-the-MFMA numerics as above.
using kqsort::Segment;

struct CgArgs {
  const void* x;        // [rows][K], pair p reads row p / x_div
  const uint8_t* w;
  const uint8_t* w2;    // up stack (GLU) or null
  void* y;              // [P][N]
  const float* bias;    // f32 [E][N] or null
  const float* bias2;
  const int* order;     // pair ids sorted by expert
  const Segment* segs;
  const int* nseg;
  const uint8_t* grids;
  int N, K, x_div, act;
  int64_t w_expert_stride;
  float limit, alpha;
  KqOutMap om;
  // outputs of codes_prepass_kernel: per activation row and 256-wide step the f16 values in staging order (512 bytes),
  // their power-of-two scale and (codecs with a block minimum) the sums of the eight 32-wide blocks
  const uint8_t* xh;
  const float* xsc;
  const float* xsum;
};

constexpr int CG_THREADS = 256;

// Activation prepass of the grouped kernel: what every workgroup used to redo for its 32 slots at every step (bf16 ->
// f16 with an exact power-of-two scale per (row, step), staging order, block sums) is done once per row.  32 threads per
// (row, step), whatever row it belongs to: rows of three steps leave no thread idle.  Steps are zero-filled past K.
// The pair sort is workgroup 0 of the same launch, and rows are read where the call has them: 128 heads of 128 x 512 q8_0, four
// entries each, row gather + sort + prepass as three launches 9.9 us, as one 3.6.  THREADS: the sort keeps eight pairs per thread in
// registers and counts the others twice, so more than 2048 pairs take 1024 threads.  A pass of 8000 pairs over 128 experts of 2048 <-> 768,
// against a sort launch of its own and a workgroup per row: q8_0 440 -> 432 us, iq3_s 407 -> 398; 2056 pairs 203 -> 197, 180 -> 174; level
// below 2048.
template <int DT, bool PAIR, bool SUMS, int THREADS>
__global__ __launch_bounds__(THREADS) void codes_prepass_kernel(const uint16_t* __restrict__ x, uint8_t* __restrict__ xh,
                                                                float* __restrict__ xsc, float* __restrict__ xsum, int K, int rows,
                                                                int nsteps, KqRowSource src, const uint32_t* __restrict__ idx, int P,
                                                                int E, int* __restrict__ order, Segment* __restrict__ segs,
                                                                int* __restrict__ nseg_out) {
  __shared__ int cnt[kqsort::SORT_MAX_E];
  __shared__ int scan_p[THREADS / 64], scan_s[THREADS / 64];
  if (blockIdx.x == 0) {
    kqsort::moe_sort_body<THREADS>(idx, P, E, order, segs, nseg_out, cnt, scan_p, scan_s, kqsort::SEG_M,
                                   src.rows_per_entry ? src.rows_per_entry : 1);
    return;
  }
  const int tid = threadIdx.x, pc = tid & 31;
  const int64_t item = (int64_t)(blockIdx.x - 1) * (THREADS / 32) + (tid >> 5);
  const int row = (int)(item / nsteps), st = (int)(item - (int64_t)row * nsteps);
  if (row >= rows) return;
  const uint16_t* xi = src.row(x, row, K);
  const int k0 = CK_STEP * st + 8 * pc;
  u32x4 v = {0, 0, 0, 0};
  if (k0 < K) v = *reinterpret_cast<const u32x4*>(xi + k0);
  float xscale = 1.f;
  _Float16 h[8];
  if constexpr (DT == KQ_BF16) {
    float amax = 0.f;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      amax = fmaxf(amax, fabsf(__builtin_bit_cast(float, v[e] << 16)));
      amax = fmaxf(amax, fabsf(__builtin_bit_cast(float, v[e] & 0xffff0000u)));
    }
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));  // the step's 32 lanes
    float inv = 1.f;
    const uint32_t eb = (__builtin_bit_cast(uint32_t, amax) >> 23) & 0xff;
    if (eb != 0 && eb != 0xff) {
      int e = (int)eb - 127 - 14;  // the largest magnitude lands in [2^14, 2^15)
      if (e < -100) e = -100;
      xscale = __builtin_bit_cast(float, (uint32_t)(127 + e) << 23);
      inv = __builtin_bit_cast(float, (uint32_t)(127 - e) << 23);
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
      h[2 * e] = (_Float16)(__builtin_bit_cast(float, v[e] << 16) * inv);
      h[2 * e + 1] = (_Float16)(__builtin_bit_cast(float, v[e] & 0xffff0000u) * inv);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      h[2 * e] = __builtin_bit_cast(_Float16, (uint16_t)(v[e] & 0xffff));
      h[2 * e + 1] = __builtin_bit_cast(_Float16, (uint16_t)(v[e] >> 16));
    }
  }
  const size_t rs = (size_t)row * nsteps + st;
  stage_group<PAIR>(xh + rs * 512, pc, h);
  if (pc == 0) xsc[rs] = xscale;
  if constexpr (SUMS) {
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) sum += (float)h[e];
    sum += __shfl_xor(sum, 1);
    sum += __shfl_xor(sum, 2);  // 4 lanes = one 32-weight block
    if ((pc & 3) == 0) xsum[rs * 8 + (pc >> 2)] = sum;
  }
}

constexpr int CG_BN = 128;

template <int C>
constexpr int grouped_lds_bytes() {
  return 32 * XA_STRIDE + 32 * 4 + 8 * 32 * 4 + CG_BN * CodeGeom<C>::LROW + 32 * 4 + CodeGeom<C>::GROUPED_GRID_BYTES +
         CodeGeom<C>::SPREAD_BYTES;
}

template <int C, int DT, bool GLU>
__global__ __launch_bounds__(CG_THREADS, 2) void codes_grouped_kernel(CgArgs a) {
  using G = CodeGeom<C>;
  constexpr int WPT = (CG_BN * G::PIECES + CG_THREADS - 1) / CG_THREADS;
  constexpr int NCOLS = GLU ? CG_BN / 2 : CG_BN;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  uint8_t* a_lds = smem;                                                  // [32][XA_STRIDE] f16 activations of the step
  float* xs_lds = reinterpret_cast<float*>(a_lds + 32 * XA_STRIDE);       // [32] activation scale per slot
  float* xsum_lds = xs_lds + 32;                                          // [8 blocks][32 slots] (HAS_MIN)
  uint8_t* b_lds = reinterpret_cast<uint8_t*>(xsum_lds + 8 * 32);         // [128][LROW]
  int* pair_lds = reinterpret_cast<int*>(b_lds + CG_BN * G::LROW);        // [32] output row per slot, -1 = none
  uint8_t* grid_lds = reinterpret_cast<uint8_t*>(pair_lds + 32);
  uint8_t* spread_lds = grid_lds + G::GROUPED_GRID_BYTES;

  if ((int)blockIdx.y >= *a.nseg) return;  // uniform: the grid is sized for the worst case
  const Segment seg = a.segs[blockIdx.y];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, kg = lane >> 5;
  const int N = a.N, K = a.K;
  const int nsteps = (K + CK_STEP - 1) / CK_STEP;
  const size_t row_bytes = (size_t)(K / G::WPB) * G::BPB;
  const int n0 = blockIdx.x * NCOLS;
  const int ncols = N - n0 < NCOLS ? N - n0 : NCOLS;
  const uint8_t* wbase = a.w + (size_t)seg.expert * (size_t)a.w_expert_stride;
  const uint8_t* wbase2 = GLU ? a.w2 + (size_t)seg.expert * (size_t)a.w_expert_stride : wbase;
  const uint8_t* w_last = wbase + (size_t)N * row_bytes - 16;  // the last 16 bytes of the expert's matrix
  const uint8_t* w_last2 = wbase2 + (size_t)N * row_bytes - 16;

  // slab row rr (= wave * 32 + l32 in the compute phase) -> (matrix, column)
  auto slab_col = [&](int rr, bool& up) {
    if constexpr (GLU) {
      const int wv = rr >> 5;
      up = wv & 1;
      return (wv >> 1) * 32 + (rr & 31);
    } else {
      up = false;
      return rr;
    }
  };

  if (tid < 32) pair_lds[tid] = tid < seg.count ? a.order[seg.start + tid] : -1;

  // ---- tables
  build_tables<C, CG_THREADS, true>(grid_lds, spread_lds, a.grids, tid);
  const Tables tabs{G::PAIR_LUT ? grid_lds + 4 * (tid & 31) : grid_lds, spread_lds, 7};

  // ---- piece maps.  Activations: piece i = tid + 256 t -> (slot i / 32, 16-byte piece i % 32).
  const int a_slot0 = tid >> 5, a_pc = tid & 31;
  size_t a_rs[4];  // (row, step 0) index of the slot's activation row in the prepass outputs
  bool a_live[4];
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const int slot = a_slot0 + 8 * t;
    a_live[t] = slot < seg.count;
    a_rs[t] = (size_t)(a.order[seg.start + (a_live[t] ? slot : 0)] / a.x_div) * nsteps;
  }
  const uint8_t* w_src[WPT];
  uint32_t w_loff[WPT];
  bool w_up[WPT];
#pragma unroll
  for (int t = 0; t < WPT; t++) {
    const int i = tid + CG_THREADS * t;
    const int r = i / G::PIECES, pc = i % G::PIECES;
    bool up;
    const int col = slab_col(r < CG_BN ? r : 0, up);
    const bool ok = r < CG_BN && col < ncols;  // rows past N re-read the slab's first row
    w_up[t] = up;
    w_src[t] = (up ? wbase2 : wbase) + (size_t)(n0 + (ok ? col : 0)) * row_bytes + 16 * pc;
    w_loff[t] = r < CG_BN ? (uint32_t)r * G::LROW + 16 * pc : 0xffffffffu;
  }

  u32x4 areg[4], wreg[WPT];
  float sreg[4] = {0.f, 0.f, 0.f, 0.f};  // a_pc == 0: the slot's scale; a_pc 8 .. 15 (HAS_MIN): block sum a_pc - 8
  auto issue = [&](int st) {
#pragma unroll
    for (int t = 0; t < 4; t++) {
      u32x4 av = {0, 0, 0, 0};
      float sv = 0.f;
      if (a_live[t]) {
        av = *reinterpret_cast<const u32x4*>(a.xh + (a_rs[t] + st) * 512 + 16 * a_pc);
        if (a_pc == 0) sv = a.xsc[a_rs[t] + st];
        if constexpr (G::HAS_MIN) {
          if (a_pc >= 8 && a_pc < 16) sv = a.xsum[(a_rs[t] + st) * 8 + (a_pc - 8)];
        }
      }
      areg[t] = av;
      sreg[t] = sv;
    }
#pragma unroll
    for (int t = 0; t < WPT; t++) {
      const uint8_t* p = w_src[t] + (size_t)st * G::BYTES;
      const uint8_t* last = w_up[t] ? w_last2 : w_last;
      const uint8_t* q = p <= last ? p : last;  // never read past the end of the expert's matrix
      u32x4 v = *reinterpret_cast<const u32x4_a1*>(q);
      if (q != p) v = shr_bytes(v, (uint32_t)(p - q));
      wreg[t] = v;
    }
  };
  auto park = [&]() {
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const int slot = a_slot0 + 8 * t;
      *reinterpret_cast<u32x4*>(a_lds + slot * XA_STRIDE + 16 * a_pc) = areg[t];
      if (a_pc == 0) xs_lds[slot] = sreg[t];
      if constexpr (G::HAS_MIN) {
        if (a_pc >= 8 && a_pc < 16) xsum_lds[(a_pc - 8) * 32 + slot] = sreg[t];
      }
    }
#pragma unroll
    for (int t = 0; t < WPT; t++)
      if (w_loff[t] != 0xffffffffu) *reinterpret_cast<u32x4*>(b_lds + w_loff[t]) = wreg[t];
  };

  float acc[16];  // output slots 8 (i / 4) + 4 kg + i % 4 of slab row wave * 32 + l32
#pragma unroll
  for (int i = 0; i < 16; i++) acc[i] = 0.f;
  const uint8_t* b_lane = b_lds + (wave * 32 + l32) * G::LROW;
  const uint8_t* a_lane = a_lds + l32 * XA_STRIDE + 16 * kg;

  issue(0);
  for (int st = 0; st < nsteps; st++) {
    lds_barrier();  // tables built / everyone is done reading the previous step
    park();
    if (st + 1 < nsteps) issue(st + 1);
    lds_barrier();
    const int kvalid = K - CK_STEP * st;
    float sacc[16];
#pragma unroll
    for (int i = 0; i < 16; i++) sacc[i] = 0.f;
    constexpr int MPS = G::SB / 16;
    auto run_step = [&](auto full_c) {
      constexpr bool FULL = decltype(full_c)::value;
      f32x16 part[2];
      RowRegs<4 * G::PIECES> row;
      StaticFor<G::PIECES>::run([&](auto pc) {
        constexpr int P = decltype(pc)::value;
        const u32x4 v = *reinterpret_cast<const u32x4*>(b_lane + 16 * P);
        row.d[4 * P] = v[0];
        row.d[4 * P + 1] = v[1];
        row.d[4 * P + 2] = v[2];
        row.d[4 * P + 3] = v[3];
      });
      StaticFor<16>::run([&](auto jc) {
        constexpr int J = decltype(jc)::value;
        if (FULL || 16 * J < kvalid) {  // uniform
          const f16x8 bv = codes<C, J>(row, kg, tabs);
          const f16x8 av = *reinterpret_cast<const f16x8*>(a_lane + 32 * J);
          constexpr int sbi = J / MPS, slot = sbi & 1;
          if constexpr (J % MPS == 0)
            part[slot] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, f32x16{0}, 0, 0, 0);
          else
            part[slot] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, part[slot], 0, 0, 0);
          if constexpr (J % MPS == MPS - 1) {
            float mn;
            const float sc = block_scale<C, sbi>(row, mn);
#pragma unroll
            for (int i = 0; i < 16; i++) sacc[i] = fmaf(sc, part[slot][i], sacc[i]);
            if constexpr (G::HAS_MIN) {
#pragma unroll
              for (int q = 0; q < 4; q++) {
                const float4 xm = *reinterpret_cast<const float4*>(xsum_lds + sbi * 32 + 8 * q + 4 * kg);
                sacc[4 * q + 0] = fmaf(mn, xm.x, sacc[4 * q + 0]);
                sacc[4 * q + 1] = fmaf(mn, xm.y, sacc[4 * q + 1]);
                sacc[4 * q + 2] = fmaf(mn, xm.z, sacc[4 * q + 2]);
                sacc[4 * q + 3] = fmaf(mn, xm.w, sacc[4 * q + 3]);
              }
            }
          }
        }
      });
    };
    if (kvalid >= CK_STEP)
      run_step(std::true_type{});
    else
      run_step(std::false_type{});
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const float4 xs4 = *reinterpret_cast<const float4*>(xs_lds + 8 * q + 4 * kg);
      acc[4 * q + 0] = fmaf(xs4.x, sacc[4 * q + 0], acc[4 * q + 0]);
      acc[4 * q + 1] = fmaf(xs4.y, sacc[4 * q + 1], acc[4 * q + 1]);
      acc[4 * q + 2] = fmaf(xs4.z, sacc[4 * q + 2], acc[4 * q + 2]);
      acc[4 * q + 3] = fmaf(xs4.w, sacc[4 * q + 3], acc[4 * q + 3]);
    }
  }

  // ---- epilogue
  if constexpr (!GLU) {
    const int col = wave * 32 + l32;
    const float bv = (a.bias && col < ncols) ? a.bias[(size_t)seg.expert * N + n0 + col] : 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int pr = pair_lds[8 * (i >> 2) + 4 * kg + (i & 3)];
      if (pr >= 0 && col < ncols)
        kq::store_result<DT>(a.y, a.om, (size_t)kq::out_row(a.om, pr) * N + n0 + col, acc[i] + bv);
    }
  } else {
    lds_barrier();  // the step buffers are free: reuse them for the up sums
    float* ex = reinterpret_cast<float*>(smem);  // [2 column blocks][16][64]
    const int nb = wave >> 1;
    if (wave & 1) {
#pragma unroll
      for (int i = 0; i < 16; i++) ex[(nb * 16 + i) * 64 + lane] = acc[i];
    }
    lds_barrier();
    if (!(wave & 1)) {
      const int col = nb * 32 + l32;
      const bool live = col < ncols;
      const float gb = (a.bias && live) ? a.bias[(size_t)seg.expert * N + n0 + col] : 0.f;
      const float ub = (a.bias2 && live) ? a.bias2[(size_t)seg.expert * N + n0 + col] : 0.f;
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int pr = pair_lds[8 * (i >> 2) + 4 * kg + (i & 3)];
        if (pr >= 0 && live) {
          const float v = kq::glu_epilogue_fast(a.act, acc[i] + gb, ex[(nb * 16 + i) * 64 + lane] + ub, a.limit, a.alpha);
          kq::store_result<DT>(a.y, a.om, (size_t)kq::out_row(a.om, pr) * N + n0 + col, v);
        }
      }
    }
  }
}

template <int C, int DT, bool GLU>
int launch_grouped(const CgArgs& a, int P, int E, hipStream_t s) {
  constexpr int NCOLS = GLU ? CG_BN / 2 : CG_BN;
  int maxseg = E + P / 32;  // sum over experts of ceil(c_e / 32) <= E + P / 32
  if (maxseg > P) maxseg = P;
  const size_t lds = grouped_lds_bytes<C>();
  auto kern = codes_grouped_kernel<C, DT, GLU>;
  KQ_SET_MAX_LDS_ONCE((kern), lds);
  hipLaunchKernelGGL(kern, dim3((a.N + NCOLS - 1) / NCOLS, maxseg), dim3(CG_THREADS), lds, s, a);
  KQ_HIP_CHECK(hipGetLastError());
  return KQ_OK;
}

template <int C>
int launch_grouped_any(const CgArgs& a, int P, int E, int glu, int dtype, hipStream_t s) {
  if (glu) return dtype == KQ_F16 ? launch_grouped<C, KQ_F16, true>(a, P, E, s) : launch_grouped<C, KQ_BF16, true>(a, P, E, s);
  return dtype == KQ_F16 ? launch_grouped<C, KQ_F16, false>(a, P, E, s) : launch_grouped<C, KQ_BF16, false>(a, P, E, s);
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

}  // namespace

// The three launcher groups below can be compiled into separate objects (KQ_CODES_PART = 1 dense, 2 gathered,
// 3 grouped; unset = all) so that the build instantiates their kernels in parallel.
#if !defined(KQ_CODES_PART) || KQ_CODES_PART == 3

bool kq_codes_moe_supported(int P, int E, int N, int K, int codec) {
  // nvfp4 (a scale per 16 weights: 16 x 16 scalings per step) does not fit the register file here and
  // stays on the any-codec path
  if (codec < KQ_Q4_0 || codec >= KQ_NUM_CODECS || codec == KQ_NVFP4) return false;
  return P > 16 && E > 0 && E <= 4096 && (int64_t)E + P / 32 < 65535 && N > 0 && K > 0 && (K & 7) == 0 &&
         K % kq_geom(codec).wpb == 0;
}

// Workspace: sorted pair list, segment table, segment count, then the prepass outputs for `rows` activation rows:
// f16 steps (512 bytes each), step scales, block sums.
size_t kq_codes_moe_workspace_bytes(int P, int E, int rows, int K) {
  const size_t rs = (size_t)rows * ((K + CK_STEP - 1) / CK_STEP);
  return align256((size_t)P * 4) + align256(((size_t)E + P / 32 + 1) * sizeof(Segment)) + 256 + align256(rs * 512) +
         align256(rs * 4) + align256(rs * 32);
}

// x: [rows][K]; pair p reads row p / x_div and expert idx[p]; out [P][N].
int kq_launch_codes_moe(const void* x, const uint8_t* w, const uint8_t* w2, const uint32_t* idx, const float* bias,
                        const float* bias2, void* out, int P, int E, int N, int K, int x_div, int64_t w_expert_stride,
                        int glu, int act, float limit, float alpha, int codec, int dtype, void* ws, KqOutMap om,
                        hipStream_t s, KqRowSource src) {
  if (!kq_codes_moe_supported(P, E, N, K, codec) || (reinterpret_cast<uintptr_t>(x) & 15) ||
      (reinterpret_cast<uintptr_t>(ws) & 255))
    return KQ_ERR_UNSUPPORTED;
  uint8_t* p = static_cast<uint8_t*>(ws);
  int* order = reinterpret_cast<int*>(p);
  Segment* segs = reinterpret_cast<Segment*>(p + align256((size_t)P * 4));
  int* nseg = reinterpret_cast<int*>(p + align256((size_t)P * 4) + align256(((size_t)E + P / 32 + 1) * sizeof(Segment)));
  const int rows = glu ? P / (x_div < 1 ? 1 : x_div) : P, nsteps = (K + CK_STEP - 1) / CK_STEP;
  const size_t rs = (size_t)rows * nsteps;
  uint8_t* xh = reinterpret_cast<uint8_t*>(nseg) + 256;
  float* xsc = reinterpret_cast<float*>(xh + align256(rs * 512));
  float* xsum = reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(xsc) + align256(rs * 4));
  {
    const bool pair = codec == KQ_IQ4_NL || codec == KQ_IQ4_XS || codec == KQ_MXFP4, sums = codec == KQ_Q4_1 || codec == KQ_Q5_1;
    const uint16_t* xi = static_cast<const uint16_t*>(x);
#define KQ_PRE(DTV, PV, SV)                                                                                                       \
  do {                                                                                                                          \
    constexpr int narrow = 256, wide = 1024;                                                                                    \
    if (P <= 8 * narrow)                                                                                                        \
      hipLaunchKernelGGL((codes_prepass_kernel<DTV, PV, SV, narrow>), dim3((unsigned)((rs + 7) / 8 + 1)), dim3(narrow), 0, s, xi, xh, xsc,  \
                         xsum, K, rows, nsteps, src, idx, P, E, order, segs, nseg);                                             \
    else                                                                                                                        \
      hipLaunchKernelGGL((codes_prepass_kernel<DTV, PV, SV, wide>), dim3((unsigned)((rs + 31) / 32 + 1)), dim3(wide), 0, s, xi, xh, xsc,    \
                         xsum, K, rows, nsteps, src, idx, P, E, order, segs, nseg);                                             \
  } while (0)
    if (dtype == KQ_F16) {
      if (pair) KQ_PRE(KQ_F16, true, false);
      else if (sums) KQ_PRE(KQ_F16, false, true);
      else KQ_PRE(KQ_F16, false, false);
    } else {
      if (pair) KQ_PRE(KQ_BF16, true, false);
      else if (sums) KQ_PRE(KQ_BF16, false, true);
      else KQ_PRE(KQ_BF16, false, false);
    }
#undef KQ_PRE
    KQ_HIP_CHECK(hipGetLastError());
  }
  CgArgs a{};
  a.xh = xh;
  a.xsc = xsc;
  a.xsum = xsum;
  a.x = x;
  a.w = w;
  a.w2 = w2;
  a.y = out;
  a.bias = bias;
  a.bias2 = bias2;
  a.order = order;
  a.segs = segs;
  a.nseg = nseg;
  a.grids = kq_device_grids();
  if (!a.grids) return KQ_ERR_HIP;
  a.N = N;
  a.K = K;
  a.x_div = x_div < 1 ? 1 : x_div;
  a.act = act;
  a.w_expert_stride = w_expert_stride;
  a.limit = limit;
  a.alpha = alpha;
  a.om = om;
  switch (codec) {
#define KQ_CASE(c) \
  case c:          \
    return launch_grouped_any<c>(a, P, E, glu, dtype, s);
    KQ_CASE(KQ_Q4_0) KQ_CASE(KQ_Q4_1) KQ_CASE(KQ_Q5_0) KQ_CASE(KQ_Q5_1) KQ_CASE(KQ_Q8_0) KQ_CASE(KQ_IQ4_NL)
    KQ_CASE(KQ_IQ4_XS) KQ_CASE(KQ_IQ3_S) KQ_CASE(KQ_IQ3_XXS) KQ_CASE(KQ_IQ2_XXS) KQ_CASE(KQ_IQ2_XS) KQ_CASE(KQ_IQ2_S)
    KQ_CASE(KQ_IQ1_S) KQ_CASE(KQ_IQ1_M) KQ_CASE(KQ_MXFP4) KQ_CASE(KQ_NVFP4)
#undef KQ_CASE
  }
  return KQ_ERR_UNSUPPORTED;
}

#endif  // grouped

#if !defined(KQ_CODES_PART) || KQ_CODES_PART == 1
bool kq_codes_supported(int M, int N, int K, int codec) {
  if (codec < KQ_Q4_0 || codec >= KQ_NUM_CODECS) return false;  // the K-quants have their own kernels
  return M > 0 && M <= CK_MAXM && N > 0 && K > 0 && K % kq_geom(codec).wpb == 0;
}

int kq_launch_codes_skinny(const void* x, const uint8_t* w, const void* bias, void* y, int M, int N, int K, int codec,
                           int dtype, hipStream_t s) {
  if (!kq_codes_supported(M, N, K, codec) || (reinterpret_cast<uintptr_t>(x) & 15) || (K & 7)) return KQ_ERR_UNSUPPORTED;
  CkArgs a{};
  a.x = x;
  a.w = w;
  a.y = y;
  a.bias = static_cast<const uint16_t*>(bias);
  a.grids = kq_device_grids();
  if (!a.grids) return KQ_ERR_HIP;
  a.M = M;
  a.N = N;
  a.K = K;
  switch (codec) {
#define KQ_CASE(c) \
  case c:          \
    return launch_codes_dt<c>(a, dtype, s);
    KQ_CASE(KQ_Q4_0) KQ_CASE(KQ_Q4_1) KQ_CASE(KQ_Q5_0) KQ_CASE(KQ_Q5_1) KQ_CASE(KQ_Q8_0) KQ_CASE(KQ_IQ4_NL)
    KQ_CASE(KQ_IQ4_XS) KQ_CASE(KQ_IQ3_S) KQ_CASE(KQ_IQ3_XXS) KQ_CASE(KQ_IQ2_XXS) KQ_CASE(KQ_IQ2_XS) KQ_CASE(KQ_IQ2_S)
    KQ_CASE(KQ_IQ1_S) KQ_CASE(KQ_IQ1_M) KQ_CASE(KQ_MXFP4) KQ_CASE(KQ_NVFP4)
#undef KQ_CASE
  }
  return KQ_ERR_UNSUPPORTED;
}

#endif  // dense

#if !defined(KQ_CODES_PART) || KQ_CODES_PART == 2
// Gathered calls of up to a few entries (MoE decode): one activation row per entry (M = 1), the entry's expert
// matrix, optional f32 biases; glu != 0 runs gate and up stacks and the fused epilogue.
// (iq4_nl / q4_0 / mxfp4 / nvfp4 entries come here only when the streamed kernel declines them: a K that is no
// multiple of 256, more than 16 (32) superblocks.)
// (q8_0 entries are not taken here: the streamed kernel has a q8_0 unit, and where that declines - a K that is no
// multiple of 256 - the plain vector kernel measured 9.1 / 8.4 us against 12.7 / 9.0 us here for the GLU / down ops
// of 8 experts of 768 x 2048.)
bool kq_codes_gather_supported(int M, int N, int K, int codec) {
  return M == 1 && codec != KQ_Q8_0 && kq_codes_supported(M, N, K, codec);
}

int kq_launch_codes_gather(const void* x, const uint8_t* w, const uint8_t* w2, const uint32_t* lhs, const uint32_t* rhs,
                           const float* bias, const float* bias2, void* out, int B, int M, int N, int K, int x_div,
                           int64_t x_batch_stride, int64_t w_expert_stride, int glu, int act, float limit, float alpha,
                           int codec, int dtype, int E, KqOutMap om, hipStream_t s) {
  if (!kq_codes_gather_supported(M, N, K, codec) || !rhs || B <= 0 || B > 65535 || (reinterpret_cast<uintptr_t>(x) & 15) ||
      (K & 7) || (x_batch_stride & 7) || (glu && !w2))
    return KQ_ERR_UNSUPPORTED;
  CkArgs a{};
  a.x = x;
  a.w = w;
  a.w2 = w2;
  a.y = out;
  a.lhs = lhs;
  a.rhs = rhs;
  a.fbias = bias;
  a.fbias2 = bias2;
  a.grids = kq_device_grids();
  if (!a.grids) return KQ_ERR_HIP;
  a.M = M;
  a.N = N;
  a.K = K;
  a.x_div = x_div < 1 ? 1 : x_div;
  a.act = act;
  a.x_item_stride = x_batch_stride;
  a.w_expert_stride = w_expert_stride;
  a.limit = limit;
  a.alpha = alpha;
  a.om = om;
  a.E = E;
  switch (codec) {
#define KQ_CASE(c)                                                                                               \
  case c:                                                                                                        \
    if (glu) return dtype == KQ_F16 ? launch_codes<c, KQ_F16, 1, 2>(a, s, B) : launch_codes<c, KQ_BF16, 1, 2>(a, s, B); \
    return dtype == KQ_F16 ? launch_codes<c, KQ_F16, 1, 1>(a, s, B) : launch_codes<c, KQ_BF16, 1, 1>(a, s, B);
    KQ_CASE(KQ_Q4_0) KQ_CASE(KQ_Q4_1) KQ_CASE(KQ_Q5_0) KQ_CASE(KQ_Q5_1) KQ_CASE(KQ_Q8_0) KQ_CASE(KQ_IQ4_NL)
    KQ_CASE(KQ_IQ4_XS) KQ_CASE(KQ_IQ3_S) KQ_CASE(KQ_IQ3_XXS) KQ_CASE(KQ_IQ2_XXS) KQ_CASE(KQ_IQ2_XS) KQ_CASE(KQ_IQ2_S)
    KQ_CASE(KQ_IQ1_S) KQ_CASE(KQ_IQ1_M) KQ_CASE(KQ_MXFP4) KQ_CASE(KQ_NVFP4)
#undef KQ_CASE
  }
  return KQ_ERR_UNSUPPORTED;
}
#endif  // gathered
