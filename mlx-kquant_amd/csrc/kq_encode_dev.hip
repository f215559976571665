// Device-side wire encoder behind kq_quantize_dev: the legacy 32-weight codecs and the K-quant superblock codecs.
// The bytes equal kq_quantize's: every value is computed by the expressions of kq_encode_blocks.h, in its order of
// additions, unfused.  The reference's GPU encoders cover the same codecs (metal/.../kq_quantized_encode.h); its IQ
// encoders are CPU-only (src/kquant_ops.cpp:602-606), as here.
//
// What bounds it.  K-quants: the vector ALU.  A sub-block's fit tries 37 (scale, min) or 19 scale candidates, and the
// order of its sums is part of the result, so a candidate is one lane's serial work: 15 (8) instructions per weight and
// candidate that cannot be fused.  The (scale, min) codecs evaluate one or two of the 37 and rule the others out by a bound
// (fit_scale_min below): 210 instead of 660 instructions a weight, the SIMDs 95 % busy issuing them.  One lane per
// sub-block (8 or 16 per superblock) keeps all three arrays of a fit in registers.  4096 x 4096 f32, normally distributed,
// all candidates -> bounded: q4_k 225 -> 112 us, q5_k 254 -> 116, q2_k 296 -> 161 (q3_k 82, q6_k 78: 19 candidates, no
// bound); 300 x 4096 q4_k 41 -> 26; small matrices, where one wave's latency counts, share all candidates of a sub-block between four
// lanes (launch_k).  Blocks narrow and far above zero, whose least-squares systems are near singular, keep more candidates
// (50 + normal: q4_k 223 -> 215, q5_k 252 -> 275; 100 + normal 222 -> 157, 252 -> 320; 1000 + normal 222 -> 281, 251 -> 219).
// Legacy codecs: memory.  Eight lanes per block, 16-byte loads, wire bytes assembled in LDS and stored as dwords
// (4096 x 4096 f32 to q8_0: 20 us, 4.2 TB/s).
#include "kq_common.h"
#include "kq_decode.h"
#include "kq_encode_blocks.h"

namespace {

__device__ __forceinline__ float clamp_level(float v, float lo, float hi) {  // clampi(rne(v), lo, hi), kept as a float
  return __builtin_amdgcn_fmed3f(__builtin_rintf(v), lo, hi);
}
// The same where the levels go below zero and v may be a NaN: the integer conversion made that level 0, the median of three
// makes it the lower bound.  (With lo = 0 both are 0.)
__device__ __forceinline__ float clamp_level_signed(float v, float lo, float hi) {
  return v == v ? clamp_level(v, lo, hi) : 0.f;
}

// rint(a / b) for a quotient that is clamped to a few hundred levels afterwards, from v_rcp_f32 (1 ulp): the product is
// within 4e-7 of its size of the quotient, so it rounds like the quotient unless it lies that close to a half.  `sure` is
// cleared then, and for every quotient that is not finite; the caller divides instead.
__device__ __forceinline__ float rint_quotient(float a, float rcp_b, bool& sure) {
  const float q = a * rcp_b, l = __builtin_rintf(q);
  sure &= std::fabs(q - l) < 0.4999f;
  return l;
}

// four weights at element i (a multiple of four) of w, widened exactly
__device__ __forceinline__ float4 load4(const void* w, int dtype, int64_t i) {
  if (dtype == KQ_F32) return *reinterpret_cast<const float4*>(static_cast<const float*>(w) + i);
  const ushort4 h = *reinterpret_cast<const ushort4*>(static_cast<const uint16_t*>(w) + i);
  if (dtype == KQ_F16) return make_float4(kq::h2f(h.x), kq::h2f(h.y), kq::h2f(h.z), kq::h2f(h.w));
  auto up = [](uint16_t v) { return __builtin_bit_cast(float, (uint32_t)v << 16); };
  return make_float4(up(h.x), up(h.y), up(h.z), up(h.w));
}
// the same for a tensor whose address is not a multiple of four elements
__device__ __forceinline__ float4 load4_any(const void* w, int dtype, int64_t i, bool aligned) {
  if (aligned) return load4(w, dtype, i);
  float v[4];
  for (int t = 0; t < 4; t++) {
    if (dtype == KQ_F32) v[t] = static_cast<const float*>(w)[i + t];
    else {
      const uint16_t h = static_cast<const uint16_t*>(w)[i + t];
      v[t] = dtype == KQ_F16 ? kq::h2f(h) : __builtin_bit_cast(float, (uint32_t)h << 16);
    }
  }
  return make_float4(v[0], v[1], v[2], v[3]);
}

// `bytes` staged wire bytes to dst, by the workgroup's `nthreads` threads
__device__ __forceinline__ void store_wire(uint8_t* dst, const uint8_t* staged, int bytes, int tid, int nthreads) {
  if ((reinterpret_cast<uintptr_t>(dst) & 3) == 0) {
    for (int i = tid; i < bytes / 4; i += nthreads)
      reinterpret_cast<uint32_t*>(dst)[i] = reinterpret_cast<const uint32_t*>(staged)[i];
    for (int i = (bytes & ~3) + tid; i < bytes; i += nthreads) dst[i] = staged[i];
  } else {
    for (int i = tid; i < bytes; i += nthreads) dst[i] = staged[i];
  }
}

// ------------------------------------------------------------------ legacy 32-weight codecs
// Lane t of a block's eight holds weights 4t ... 4t+3.  The reductions keep the sequential code's choice among equal
// values (the earlier one), which for a minimum of zero decides the sign that is stored.
constexpr int LEG_THREADS = 256, LEG_BLOCKS = LEG_THREADS / 8;

template <int C>
__global__ __launch_bounds__(LEG_THREADS) void encode_legacy_kernel(const void* __restrict__ w, int dtype,
                                                                    uint8_t* __restrict__ wire, int64_t nblocks,
                                                                    bool aligned) {
  constexpr int BPB = kq_geom(C).bpb;
  __shared__ __attribute__((aligned(16))) uint8_t out[LEG_BLOCKS * BPB];
  const int64_t blk0 = (int64_t)blockIdx.x * LEG_BLOCKS;
  const int tid = threadIdx.x, b = tid >> 3, t = tid & 7;
  const int64_t blk = min(blk0 + b, nblocks - 1);  // lanes past the end redo the last block; their bytes are not stored
  const float4 v4 = load4_any(w, dtype, blk * 32 + 4 * t, aligned);
  const float v[4] = {v4.x, v4.y, v4.z, v4.w};
  // the block's first weight starts the minimum and the maximum (a NaN there stays); a later NaN is passed over
  float amax = 0.f, lo = t == 0 ? v[0] : INFINITY, hi = t == 0 ? v[0] : -INFINITY;
  for (int i = 0; i < 4; i++) {
    amax = std::max(amax, std::fabs(v[i]));
    lo = std::min(lo, v[i]);
    hi = std::max(hi, v[i]);
  }
  for (int m = 1; m < 8; m <<= 1) {
    amax = std::max(amax, __shfl_xor(amax, m));
    const float ol = __shfl_xor(lo, m), oh = __shfl_xor(hi, m);
    lo = (t & m) ? std::min(ol, lo) : std::min(lo, ol);
    hi = (t & m) ? std::max(oh, hi) : std::max(hi, oh);
  }
  uint8_t* p = out + b * BPB;
  if constexpr (C == KQ_Q8_0) {
    const float d = amax / 127.0f, id = d != 0.f ? 1.0f / d : 0.f;
    if (t == 0) kqenc::put_f16(p, d);
    for (int i = 0; i < 4; i++)
      p[2 + 4 * t + i] = (uint8_t)static_cast<int8_t>(std::clamp(std::round(v[i] * id), -127.0f, 127.0f));
  } else {
    constexpr bool has_min = C == KQ_Q4_1 || C == KQ_Q5_1;
    constexpr int bits = C == KQ_Q5_0 || C == KQ_Q5_1 ? 5 : 4;
    constexpr float top = (1 << bits) - 1, bias = has_min ? 0.f : float(1 << (bits - 1));
    const float d = has_min ? (hi - lo) / top : amax / float((1 << (bits - 1)) - 1);
    const float id = d != 0.f ? 1.0f / d : 0.f;
    if (t == 0) {
      kqenc::put_f16(p, d);
      if (has_min) kqenc::put_f16(p + 2, lo);
    }
    uint32_t nib = 0, fifth = 0;  // levels of the lane's four weights, a byte each; their fifth bits at 4t ... 4t+3
    for (int i = 0; i < 4; i++) {
      const float x = has_min ? (v[i] - lo) * id : v[i] * id;
      const uint32_t q = static_cast<uint8_t>(std::clamp(std::round(x) + bias, 0.0f, top));
      nib |= (q & 15) << (8 * i);
      fifth |= (q >> 4) << (4 * t + i);
    }
    const uint32_t other = __shfl_xor(nib, 4);  // weight 4t+16+i for the lower four lanes
    uint8_t* qs = p + (has_min ? 4 : 2) + (bits == 5 ? 4 : 0);
    if (t < 4)
      for (int i = 0; i < 4; i++) qs[4 * t + i] = (uint8_t)((nib | (other << 4)) >> (8 * i));
    if (bits == 5) {
      for (int m = 1; m < 8; m <<= 1) fifth |= __shfl_xor(fifth, m);
      if (t < 4) qs[t - 4] = (uint8_t)(fifth >> (8 * t));
    }
  }
  __syncthreads();
  const int64_t left = nblocks - blk0;
  store_wire(wire + blk0 * BPB, out, (int)(left < LEG_BLOCKS ? left : LEG_BLOCKS) * BPB, tid, LEG_THREADS);
}

// ------------------------------------------------------------------ K-quant superblocks
// One wave per workgroup, lane = (superblock, sub-block j).
template <int C>
struct KGeom {
  static constexpr int SUBS = C == KQ_Q4_K || C == KQ_Q5_K ? 8 : 16, N = 256 / SUBS;
  static constexpr int NMAX = C == KQ_Q2_K ? 3 : C == KQ_Q4_K ? 15 : 31;  // of the (scale, min) codecs
};

// kqenc::fit_scale_min, with most of its 37 candidates ruled out before they are evaluated.  A candidate's levels decide
// everything about it, and from one candidate to the next few levels change: level i is the rounded product of an inverse
// scale that grows with the step and a distance d_i >= 0 from the minimum, so it climbs by less than two over all steps.
//   1. For each weight the steps at which its level climbs are found (estimated, then settled by the level's own rounded
//      expression at the estimate), and what the climb adds to the sums of w l, w l^2 and w l d is added to that step's
//      bins.  The weights of the bins are 16-bit whole numbers w' <= w: the first two sums are exact, the third to 2^-53.
//   2. Running sums over the steps give each candidate's least possible error E = min over (s, m <= 0) of
//      sum w' (s l + m - x)^2 in closed form.  The rounded error of the candidate cannot be below
//      (sqrt(E) - r X sqrt(sum w))^2 (1 - 1e-5), r = 2^-24 (10 + 2.2 cond): rounding moves each of its terms s l + m - x by
//      at most 2^-24 (2 X + 3 |term| + |m|) and d by 2^-24 2 X, X the largest |x|, and |m| <= 2.2 cond X where
//      sum w sum w l^2 <= cond det and cond <= 8000 (the rounded determinant is then within 7 % of det).
//      The grid from minimum to maximum has the levels of step 18 and a known (s, m): its error follows the same way, with
//      |m| <= X and 2^-24 3 X for the rounding of s.
//   3. The candidate of least E is evaluated as the sequential code does it, then what else has a bound that does not
//      exceed the best error so far, except candidates with the levels of the step before (the same result, tried earlier).
// What wins is the earliest candidate of least rounded error, as in the sequential scan.  Sub-blocks outside the ranges
// for which the bound is derived (negative, huge or vanishing weights, not-finite values, errors near underflow) evaluate
// every candidate, the others those whose system is too near singular.  On normally distributed weights a lane evaluates 1.0 - 1.1 candidates, the
// slowest of 64 about two.
// The steps are taken in two halves, each of which a level climbs in at most once (0.9 of a level where the distance is the
// whole range): half the bins, so that two waves share a SIMD.
constexpr int STEPS = 37, HALF = 18;

struct FitBins {  // [step of the half][lane], eight bytes a lane: conflict-free
  unsigned long long wl[HALF][64];  // low half: sum of w' and, from bit 24, the number of climbs; high half: growth of w' l^2
  double wld[HALF][64];             // of w' d
};

__device__ __forceinline__ float step_numerator(float step, int nmax) { return -0.9f + 0.05f * step + float(nmax); }

template <int N, int NMAX, int S>
__device__ __forceinline__ float fit_scale_min(float (&x)[N], float (&wt)[N], FitBins* bins_lds, int lane, int part,
                                               float& neg_min) {
  float vmin = x[0], vmax = x[0], sw = wt[0], swx = sw * x[0], wmin = wt[0], wmax = wt[0];
#pragma unroll
  for (int i = 1; i < N; i++) {
    if (x[i] < vmin) vmin = x[i];
    if (x[i] > vmax) vmax = x[i];
    sw += wt[i];
    swx += wt[i] * x[i];
    wmin = fminf(wmin, wt[i]);
    wmax = fmaxf(wmax, wt[i]);
  }
  // Blocks this narrow and far above zero have all levels alike at most steps and no bound there: a wave of them does not look for
  // one (1000 + normal, 4096 x 4096: q4_k 341 -> 281 us, q2_k 402 -> 262; 222 and 289 before there was a bound).
  const bool alike = __builtin_amdgcn_ballot_w64(!((vmax - vmin) * float(NMAX) < 0.1f * vmax)) == 0;
  if (vmin > 0.f) vmin = 0.f;
  const bool flat = vmax <= vmin;
  const float range = vmax - vmin;
  float scale = 0.f, best_min = vmin, best_err = INFINITY;
  int best_step = STEPS;
  auto evaluate = [&](int step) {
    const float inv_s = step_numerator(float(step), NMAX) / range;
    float lv[N], sl = 0.f, sl2 = 0.f, sxl = 0.f;
#pragma unroll
    for (int i = 0; i < N; i++) {
      lv[i] = clamp_level(inv_s * (x[i] - vmin), 0.f, float(NMAX));
      const float wl = wt[i] * lv[i];
      sl += wl;
      sl2 += wl * lv[i];
      sxl += wl * x[i];
    }
    const float det = sw * sl2 - sl * sl;
    float s = (sw * sxl - swx * sl) / det, m = (sl2 * swx - sl * sxl) / det;
    if (m > 0.f) {
      m = 0.f;
      s = sxl / sl2;
    }
    float err = 0.f;
#pragma unroll
    for (int i = 0; i < N; i++) {
      const float e = s * lv[i] + m - x[i];
      err += wt[i] * e * e;
    }
    if (det > 0.f && (err < best_err || (err == best_err && step < best_step))) {
      best_err = err;
      scale = s;
      best_min = m;
      best_step = step;
    }
  };

  unsigned long long todo = flat ? 0 : (1ull << STEPS) - 1;
  bool grid = true;
  if constexpr (S > 1) {
    unsigned long long every = 0;
    for (int step = 0; step < STEPS; step += S) every |= 1ull << step;
    todo &= every << part;
  } else if (range >= 1e-9f && range <= 1e9f && vmax <= 1e9f && vmin >= -1e9f && wmin >= 0.f && wmax >= 1e-9f && wmax <= 1e9f &&
      sw == sw && swx == swx && !alike) {
    FitBins& bins = *bins_lds;
    const float ws = 65535.0f / wmax, inv0 = step_numerator(0.f, NMAX) / range;
    const float rr = 1.0f / range;  // correctly rounded: two corrections of n * rr give n / range so
    const float per_step = 20.f * range, zero_step = -(float(NMAX) - 0.9f) * 20.f - 1e-3f;
    auto over_range = [&](float num) {  // num / range
      float v = num * rr;
      v = __builtin_fmaf(__builtin_fmaf(-v, range, num), rr, v);
      return __builtin_fmaf(__builtin_fmaf(-v, range, num), rr, v);
    };
    uint32_t W = 0, sl = 0, sl2 = 0;
    double sd = 0.0, sdd = 0.0, sdl = 0.0;
#pragma unroll
    for (int i = 0; i < N; i++) {
      const float d = x[i] - vmin, l0 = __builtin_rintf(inv0 * d);
      const uint32_t w = (uint32_t)(wt[i] * ws), l = (uint32_t)l0, wl = __umul24(w, l);
      const double wd = double(w) * double(d);
      W += w;
      sl += wl;
      sl2 += __umul24(wl, l);
      sd += wd;
      sdd = __builtin_fma(wd, double(d), sdd);
      sdl = __builtin_fma(wd, double(l0), sdl);
    }
    // The distances of the closed form are taken in units of 2^k next to the range: its numerators, about W^4 times the square
    // of a distance, leave the floats otherwise (from a range of 1e7 on).  A power of two: the same digits.
    const uint32_t rexp = __builtin_bit_cast(uint32_t, range) >> 23;
    const double dunit = double(__builtin_bit_cast(float, (254u - rexp) << 23)), range_unit2 = 1.0 / (dunit * dunit);
    const double Wd = double(W), sddc = __builtin_fma(Wd, sdd, -sd * sd) * (dunit * dunit), Wu = Wd * dunit, sdu = sd * dunit;
    const float unit = float(range_unit2 / (double(ws) * Wd));
    float least = INFINITY, det_least = INFINITY;
    const float reach = fmaxf(vmax, -vmin) * std::sqrt(sw);
    int first = 0;
    auto bound_of = [&](auto at_zero, int c, bool same) {
      const double sld = double(sl), sl2d = double(sl2);
      const double det = __builtin_fma(Wd, sl2d, -sld * sld), cross = __builtin_fma(Wu, sdl, -sdu * sld);
      const float detf = float(det);
      float e = float(__builtin_fma(sddc, det, -cross * cross)) * __builtin_amdgcn_rcpf(detf) * unit;
      if constexpr (decltype(at_zero)::value) {  // the minimum may be held at zero: where m would be positive, it is zero
        const float e0 = float(__builtin_fma(sdd, sl2d, -sdl * sdl)) * __builtin_amdgcn_rcpf(float(sl2) * ws);
        e = vmin == 0.f && sl2d * sd > sld * sdl ? e0 : e;
        // such lanes may have levels almost all alike at some steps (narrow blocks far from zero): cond by the step, and no
        // bound where it is too large
        const float cond = float(W) * (float(sl2) + float(N * NMAX * NMAX)) * __builtin_amdgcn_rcpf(detf);
        if (!(cond <= 8000.f)) return same ? INFINITY : -INFINITY;
        const float root = fmaxf(std::sqrt(e) - (2.2f * 5.98e-8f) * cond * reach, 0.f);
        e = root * root;
      } else {
        det_least = fminf(det_least, detf);
      }
      e = same ? INFINITY : e;
      if (e < least) {
        least = e;
        first = c;
      }
      return e;
    };
    float bound0 = bound_of(std::true_type{}, 0, false), bound[HALF], bound_lo[HALF], grid_bound = 0.f;
#pragma unroll 1
    for (int base = 0; base < 2 * HALF; base += HALF) {
#pragma unroll
      for (int c = 0; c < HALF; c++) {
        bins.wl[c][lane] = 0;
        bins.wld[c][lane] = 0.0;
      }
      // what the loop below derives from x and wt is not to be kept from one half to the next: that would be 150 registers
#pragma unroll
      for (int i = 0; i < N; i++) asm volatile("" : "+v"(x[i]), "+v"(wt[i]));
      const float inv_b = over_range(step_numerator(float(base), NMAX));
#pragma unroll
      for (int g = 0; g < N; g += 8) {
        unsigned at[8], l[8];
#pragma unroll
        for (int t = 0; t < 8; t++) {
          const float d = x[g + t] - vmin, lb = __builtin_rintf(inv_b * d);
          // The real step at which the product passes lb + 1/2, off by less than 1e-3: every rounding on the way, here and in
          // the level's own expression, is 2^-24 of at most 20 (NMAX + 1) steps.  d = 0: no step.
          const float q = __builtin_amdgcn_rcpf(std::fabs(d)) * per_step;
          const float n = fminf(__builtin_ceilf(__builtin_fmaf(lb + 0.5f, q, zero_step)), 64.f);
          const float inv_s = over_range(step_numerator(n, NMAX));
          at[t] = unsigned(int(n)) - unsigned(base) - (__builtin_rintf(inv_s * d) > lb ? 1u : 0u);
          l[t] = (uint32_t)lb;
        }
#pragma unroll
        for (int t = 0; t < 8; t++)
          if (at[t] < unsigned(HALF) && l[t] < unsigned(NMAX)) {
            const uint32_t w = (uint32_t)(wt[g + t] * ws);
            __builtin_assume(w < 1u << 16);
            const unsigned long long v = (unsigned long long)__umul24(w, 2 * l[t] + 1) << 32 | w | 1u << 24;
            const double wd = double(w) * double(x[g + t] - vmin);
            __hip_atomic_fetch_add(&bins.wl[at[t]][lane], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_fetch_add(&bins.wld[at[t]][lane], wd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          }
      }
      auto steps = [&](auto at_zero) {
#pragma unroll
        for (int c = 0; c < HALF; c++) {
          const unsigned long long v = bins.wl[c][lane];
          sl += (uint32_t)v & 0xffffff;
          sl2 += (uint32_t)(v >> 32);
          sdl += bins.wld[c][lane];
          bound[c] = bound_of(at_zero, base + c + 1, (uint32_t)v == 0);
        }
      };
      if (__builtin_amdgcn_ballot_w64(vmin == 0.f)) steps(std::true_type{});
      else steps(std::false_type{});
      if (base == 0) {
        const float s = range / float(NMAX);  // the grid's levels are those of step 18
        grid_bound = float(__builtin_fma(double(s), __builtin_fma(double(s), double(sl2), -2.0 * sdl), sdd)) / ws;
#pragma unroll
        for (int c = 0; c < HALF; c++) bound_lo[c] = bound[c];
      }
    }
    evaluate(first);
    const float cond = float(W) * (float(sl2) + float(N * NMAX * NMAX)) / det_least;
    if (cond <= 8000.f && det_least > 0.f && best_err >= 1e-28f) {
      const float r = (10.f + 2.2f * cond) * 5.97e-8f;
      const float root = std::sqrt(best_err) * 1.00001f + r * reach, lim = root * root * 1.00001f;
      uint32_t lo = 0, hi = 0;
#pragma unroll
      for (int c = 0; c < HALF; c++) {
        lo |= bound_lo[c] > lim ? 0 : 2u << c;
        hi |= bound[c] > lim ? 0 : 2u << c;
      }
      todo = ((unsigned long long)hi << HALF | lo | (bound0 > lim ? 0 : 1)) & ~(1ull << first);
      grid = !(grid_bound > lim);
    } else {
      best_err = INFINITY;
    }
  }
  if (grid && !flat) {
    const float inv = float(NMAX) / range, s = 1.0f / inv;
    float err = 0.f;
#pragma unroll
    for (int i = 0; i < N; i++) {
      const float l = clamp_level(inv * (x[i] - vmin), 0.f, float(NMAX));
      const float e = s * l + vmin - x[i];
      err += wt[i] * e * e;
    }
    if (!(err > best_err)) {  // first of all in the sequential order (where a NaN stays)
      best_err = err;
      scale = s;
      best_min = vmin;
      best_step = -1;
    }
  }
  while (todo) {
    const int step = __builtin_ctzll(todo);
    todo &= todo - 1;
    evaluate(step);
  }
#pragma unroll
  for (int m = 1; m < S; m <<= 1) {  // of equal errors the earliest
    const float oe = __shfl_xor(best_err, m), os = __shfl_xor(scale, m), om = __shfl_xor(best_min, m);
    const int ost = __shfl_xor(best_step, m);
    if (oe < best_err || (oe == best_err && ost < best_step)) {
      best_err = oe;
      scale = os;
      best_min = om;
      best_step = ost;
    }
  }
  neg_min = flat ? -vmin : -best_min;
  return flat ? 0.f : scale;
}

// kqenc::fit_signed16 (the acceptance test compares against a rounded running best, so the candidates stay in order).
// FINITE: no weight of the wave is infinite or a NaN, so no level is a NaN either (the factors are finite: peaks below 1e-30
// return 0 whatever the scan did).
template <int NMAX, bool FINITE>
__device__ __forceinline__ float fit_signed16(const float (&x)[16], const float (&wt)[16]) {
  float peak = 0.f, apeak = 0.f;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const float a = std::fabs(x[i]);
    if (a > apeak) {
      apeak = a;
      peak = x[i];
    }
  }
  float wx[16];
#pragma unroll
  for (int i = 0; i < 16; i++) wx[i] = wt[i] * x[i];
  auto sums = [&](float inv, float& slx, float& sl2) {
    slx = sl2 = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const float l = FINITE ? clamp_level(inv * x[i], -float(NMAX), float(NMAX - 1))
                             : clamp_level_signed(inv * x[i], -float(NMAX), float(NMAX - 1));
      slx += wx[i] * l;
      sl2 += wt[i] * l * l;
    }
  };
  float slx, sl2;
  sums(-float(NMAX) / peak, slx, sl2);
  float scale = sl2 > 0.f ? slx / sl2 : 0.f, best = scale * slx;
#pragma unroll 1
  for (int k = -9; k <= 9; k++) {
    if (k == 0) continue;
    sums(-(float(NMAX) + 0.1f * float(k)) / peak, slx, sl2);
    if (sl2 > 0.f && slx * slx > best * sl2) {
      scale = slx / sl2;
      best = scale * slx;
    }
  }
  return apeak < 1e-30f ? 0.f : scale;
}

// kqenc::fit_positive of the sub-block scales (even lanes) and of the minima (odd ones): both arrays lie in LDS.  The four
// lanes of an octet that share an array take two candidates each of the nine-point scan (again the earliest of least error
// wins) and all do the refinement, whose steps depend on each other.  Returns the factor of the lane's array and leaves its
// levels in lv.
template <int N, int NMAX>
__device__ __forceinline__ float fit_positive_pair(const float* sc, const float* mn, const float* sw, int lane,
                                                   int (&lv)[N]) {
  const float* src = lane & 1 ? mn : sc;
  float wt[N], x[N], vmax = 0.f;
#pragma unroll
  for (int i = 0; i < N; i++) {
    wt[i] = sw[i];
    x[i] = src[i];
    if (x[i] > vmax) vmax = x[i];
  }
  float inv = float(NMAX) / vmax, best = 0.f;
  {
    const float s = 1.0f / inv;
#pragma unroll
    for (int i = 0; i < N; i++) {
      const int l = (uint8_t)kqenc::clampi(kqenc::rne(inv * x[i]), 0, NMAX);
      const float e = x[i] - s * float(l);
      best += wt[i] * e * e;
    }
  }
  float err = NAN, inv_k = 0.f;
  int order = 0;
#pragma unroll
  for (int half = 0; half < 2; half++) {
    const int c = ((lane >> 1) & 3) + 4 * half, k = half ? c - 3 : c - 4;
    const float inv_c = (0.1f * float(k) + float(NMAX)) / vmax, s_c = 1.0f / inv_c;
    float err_c = 0.f;
#pragma unroll
    for (int i = 0; i < N; i++) {
      const int l = min(NMAX, kqenc::rne(inv_c * x[i]));
      const float e = x[i] - s_c * float(l);
      err_c += wt[i] * e * e;
    }
    if (err_c < err || !(err == err)) {
      err = err_c;
      inv_k = inv_c;
      order = c;
    }
  }
#pragma unroll
  for (int m = 2; m < 8; m <<= 1) {
    const float oe = __shfl_xor(err, m), oi = __shfl_xor(inv_k, m);
    const int oo = __shfl_xor(order, m);
    if (oe < err || (oe == err && oo < order) || !(err == err)) {
      err = oe;
      inv_k = oi;
      order = oo;
    }
  }
  inv = vmax < 1e-30f ? -1.f : err < best ? inv_k : inv;
  float slx = 0.f, sl2 = 0.f;
#pragma unroll
  for (int i = 0; i < N; i++) {
    const int l = min(NMAX, kqenc::rne(inv * x[i]));
    lv[i] = (uint8_t)l;
    slx += wt[i] * x[i] * float(l);
    sl2 += wt[i] * float(l) * float(l);
  }
#pragma unroll 1
  for (int round = 0; round < 5; round++) {
    bool changed = false;
#pragma unroll
    for (int i = 0; i < N; i++) {
      const float w = wt[i];
      float a = slx - w * x[i] * float(lv[i]);
      float b = sl2 - w * float(lv[i]) * float(lv[i]);
      const float xb = x[i] * b;
      bool sure = true;
      float r = rint_quotient(xb, __builtin_amdgcn_rcpf(a), sure);
      if (!sure) r = std::rint(xb / a);
      const int nl = min(NMAX, int(r));
      if (a > 0.f && b > 0.f && nl != lv[i]) {
        a += w * x[i] * float(nl);
        b += w * float(nl) * float(nl);
        if (a * a * sl2 > slx * slx * b) {
          lv[i] = (uint8_t)nl;
          slx = a;
          sl2 = b;
          changed = true;
        }
      }
    }
    if (!changed) break;
  }
  if (inv < 0.f) {
#pragma unroll
    for (int i = 0; i < N; i++) lv[i] = 0;
    return 0.f;
  }
  return sl2 > 0.f ? slx / sl2 : 0.f;
}

template <int C, int S>
__global__ __launch_bounds__(64, 2) void encode_k_kernel(const void* __restrict__ w, int dtype,
                                                      const float* __restrict__ imatrix, uint8_t* __restrict__ wire,
                                                      int64_t nblocks, int64_t blocks_per_row, bool aligned) {
  constexpr int BPB = kq_geom(C).bpb, SUBS = KGeom<C>::SUBS, N = KGeom<C>::N;
  constexpr int GROUP = SUBS * S, NSB = 64 / GROUP;  // lanes per superblock, superblocks per wave
  constexpr int XS = 256 + 4;                        // floats between superblocks in LDS: eight of them in eight banks
  constexpr bool kMin = C == KQ_Q2_K || C == KQ_Q4_K || C == KQ_Q5_K;
  // One buffer for what lives one after the other: the staged weights, the bins of the (scale, min) fit, and the levels and
  // wire bytes (a workgroup of less than 20 KiB lets a CU hold eight, two per SIMD).
  constexpr size_t BUF = NSB * XS * sizeof(float);
  __shared__ __attribute__((aligned(16))) uint8_t buf[kMin && S == 1 ? sizeof(FitBins) : BUF];
  static_assert(BUF >= NSB * 256 + NSB * BPB && sizeof(FitBins) >= BUF, "buffer");
  float* xs = reinterpret_cast<float*>(buf);
  auto* s_lv = reinterpret_cast<uint8_t(*)[256]>(buf);
  uint8_t* out = buf + NSB * 256;
  __shared__ float s_sc[NSB][SUBS], s_mn[NSB][SUBS], s_sw[NSB][SUBS];
  __shared__ int s_ls[NSB][SUBS], s_lm[NSB][SUBS];
  const int lane = threadIdx.x, sb = lane / GROUP, gl = lane % GROUP, j = gl / S, part = gl % S;
  // superblocks past the end redo the last one; their bytes are not stored
  const int64_t blk0 = (int64_t)blockIdx.x * NSB, last = min(blk0 + NSB, nblocks) - 1;
  auto stage = [&](int dt, bool al) {  // all loads first: few waves are there to cover their latency
    float4 v[NSB];
#pragma unroll
    for (int i = 0; i < NSB; i++) v[i] = load4_any(w, dt, min(blk0 + i, last) * 256 + 4 * lane, al);
#pragma unroll
    for (int i = 0; i < NSB; i++) *reinterpret_cast<float4*>(xs + i * XS + 4 * lane) = v[i];
  };
  if (!aligned) stage(dtype, false);
  else if (dtype == KQ_F32) stage(KQ_F32, true);
  else if (dtype == KQ_F16) stage(KQ_F16, true);
  else stage(KQ_BF16, true);
  __syncthreads();
  const float* xb = xs + sb * XS;
  float x[N], wt[N];
#pragma unroll
  for (int i = 0; i < N; i++) x[i] = xb[N * j + i];

  // importance weights (kqenc::importance; q6_k weights by the matrix itself, q3_k and q6_k by x^2 without one)
  const float* im = nullptr;
  if (imatrix) im = imatrix + (min(blk0 + sb, last) % blocks_per_row) * 256 + N * j;
  if (C == KQ_Q6_K || (C == KQ_Q3_K && !im)) {
#pragma unroll
    for (int i = 0; i < N; i++) wt[i] = im ? im[i] : x[i] * x[i];
  } else {
    __syncthreads();
    float* sq = xs + sb * XS;
#pragma unroll
    for (int i = 0; i < N; i++) sq[N * j + i] = x[i] * x[i];
    __syncthreads();
    float total = 0.f;
#pragma unroll 32
    for (int i = 0; i < 256; i++) total += sq[i];
    const float sigma2 = (C == KQ_Q2_K ? 1.0f : 2.0f) * total / 256.0f, av = std::sqrt(sigma2);
    if (im) {
#pragma unroll
      for (int i = 0; i < N; i++) wt[i] = im[i] * std::sqrt(sigma2 + x[i] * x[i]);
    } else {
#pragma unroll
      for (int i = 0; i < N; i++) wt[i] = av + std::fabs(x[i]);
    }
  }

  __syncthreads();  // the weights have been read from buf
  uint8_t* b = out + sb * BPB;
  // levels of the lane's weights, four to a word: level(i, rint((x + add) / by)).  (A sum with a zero changes no quotient.)
  auto store_levels = [&](auto level, float add, float by) {
    const float rcp = __builtin_amdgcn_rcpf(by);
    bool sure = true;
    uint32_t packed[N / 4];
#pragma unroll
    for (int i = 0; i < N; i++) {
      const uint32_t l = level(i, rint_quotient(x[i] + add, rcp, sure));
      packed[i / 4] = i % 4 ? packed[i / 4] | l << (8 * (i % 4)) : l;
    }
    if (!sure) {
#pragma unroll
      for (int i = 0; i < N; i++) {
        const uint32_t l = level(i, __builtin_rintf((x[i] + add) / by));
        packed[i / 4] = i % 4 ? packed[i / 4] | l << (8 * (i % 4)) : l;
      }
    }
#pragma unroll
    for (int i = 0; i < N / 4; i++)
      if (i % S == part) reinterpret_cast<uint32_t*>(s_lv[sb])[N / 4 * j + i] = packed[i];
  };
  if constexpr (kMin) {
    float sw = 0.f, neg_min;
#pragma unroll
    for (int i = 0; i < N; i++) sw += wt[i];
    const float sc = fit_scale_min<N, KGeom<C>::NMAX, S>(x, wt, reinterpret_cast<FitBins*>(buf), lane, part, neg_min);
    if (part == 0) {
      s_sc[sb][j] = sc;
      s_mn[sb][j] = neg_min;
      s_sw[sb][j] = sw;
    }
    __syncthreads();
    constexpr int LMAX = C == KQ_Q2_K ? 15 : 63, DOFF = C == KQ_Q2_K ? 80 : 0;
    int lv[SUBS];
    const float f = fit_positive_pair<SUBS, LMAX>(s_sc[sb], s_mn[sb], s_sw[sb], lane, lv);
    if (gl < 2) {
      kqenc::put_f16(b + DOFF + 2 * gl, f);
#pragma unroll
      for (int i = 0; i < SUBS; i++) (gl ? s_lm : s_ls)[sb][i] = lv[i];
    }
    __syncthreads();
    const float ds = kqenc::get_f16(b + DOFF) * float(s_ls[sb][j]), dm = kqenc::get_f16(b + DOFF + 2) * float(s_lm[sb][j]);
    store_levels([&](int i, float q) { return ds == 0.f ? 0 : (uint8_t)(int)__builtin_amdgcn_fmed3f(q, 0.f, float(KGeom<C>::NMAX)); },
                 dm, ds);
  } else {
    constexpr int NMAX = C == KQ_Q6_K ? 32 : 4;
    bool finite = true;
#pragma unroll
    for (int i = 0; i < N; i++) finite &= std::fabs(x[i]) < INFINITY;
    s_sc[sb][j] = __builtin_amdgcn_ballot_w64(!finite) == 0 ? fit_signed16<NMAX, true>(x, wt) : fit_signed16<NMAX, false>(x, wt);
    __syncthreads();
    float peak = 0.f, apeak = 0.f;
    for (int i = 0; i < 16; i++) {
      const float v = s_sc[sb][i];
      if (std::fabs(v) > apeak) {
        apeak = std::fabs(v);
        peak = v;
      }
    }
    float de;
    if constexpr (C == KQ_Q6_K) {
      const float inv = -128.0f / peak;
      const bool dead = apeak < 1e-30f;
      const int8_t so = dead ? 0 : int8_t(min(127, kqenc::rne(inv * s_sc[sb][j])));
      b[192 + j] = (uint8_t)so;
      if (j == 0) kqenc::put_f16(b + 208, dead ? 0.f : 1.0f / inv);
      s_ls[sb][j] = dead;
      __syncthreads();
      de = kqenc::get_f16(b + 208) * float(so);
    } else {
      const float inv = -32.0f / peak;
      const int l = peak != 0.f ? kqenc::clampi(kqenc::rne(inv * s_sc[sb][j]), -32, 31) + 32 : 0;
      s_ls[sb][j] = l;
      if (j == 0) kqenc::put_f16(b + 108, peak != 0.f ? 1.0f / inv : 0.f);
      __syncthreads();
      de = kqenc::get_f16(b + 108) * float(l - 32);
    }
    store_levels([&](int i, float q) {
      return de == 0.f ? NMAX : (uint8_t)((q == q ? (int)__builtin_amdgcn_fmed3f(q, -float(NMAX), float(NMAX - 1)) : 0) + NMAX);
    }, 0.f, de);
  }
  __syncthreads();

  // block layout (kq_encode_blocks.h), the superblock's lanes taking its bytes in turn
  const uint8_t* lv = s_lv[sb];
  const int* ls = s_ls[sb];
  if constexpr (C == KQ_Q4_K || C == KQ_Q5_K) {
    const int* lm = s_lm[sb];
    if (gl < 4) {
      b[4 + gl] = (uint8_t)(ls[gl] | ((ls[gl + 4] >> 4) << 6));
      b[8 + gl] = (uint8_t)(lm[gl] | ((lm[gl + 4] >> 4) << 6));
      b[12 + gl] = (uint8_t)((ls[gl + 4] & 15) | ((lm[gl + 4] & 15) << 4));
    }
    constexpr int QS = C == KQ_Q4_K ? 16 : 48;
    for (int i = gl; i < 128; i += GROUP) {
      const int g = i >> 5, l = i & 31;
      b[QS + i] = (lv[64 * g + l] & 15) | ((lv[64 * g + 32 + l] & 15) << 4);
    }
    if (C == KQ_Q5_K)
      for (int l = gl; l < 32; l += GROUP) {
        uint8_t bits = 0;
        for (int t = 0; t < 8; t++) bits |= uint8_t((lv[32 * t + l] > 15) << t);
        b[16 + l] = bits;
      }
  } else if constexpr (C == KQ_Q2_K || C == KQ_Q3_K) {
    constexpr int QS = C == KQ_Q2_K ? 16 : 32;
    for (int i = gl; i < 64; i += GROUP) {
      const int h = i >> 5, l = i & 31;
      uint8_t byte = 0;
      for (int t = 0; t < 4; t++) byte |= uint8_t((lv[128 * h + 32 * t + l] & 3) << (2 * t));
      b[QS + i] = byte;
    }
    if constexpr (C == KQ_Q2_K) {
      if (gl < 16) b[gl] = (uint8_t)((ls[gl] & 15) | ((s_lm[sb][gl] & 15) << 4));
    } else {
      for (int l = gl; l < 32; l += GROUP) {
        uint8_t byte = 0;
        for (int t = 0; t < 8; t++) byte |= uint8_t(((lv[128 * (t >> 2) + 32 * (t & 3) + l] >> 2) & 1) << t);
        b[l] = byte;
      }
      if (gl < 8) b[96 + gl] = (uint8_t)((ls[gl] & 15) | ((ls[gl + 8] & 15) << 4));
      if (gl < 4) {
        uint8_t byte = 0;
        for (int t = 0; t < 4; t++) byte |= uint8_t(((ls[4 * t + gl] >> 4) & 3) << (2 * t));
        b[104 + gl] = byte;
      }
    }
  } else {
    const bool dead = ls[0];  // an empty block is all zero bytes
    for (int i = gl; i < 64; i += GROUP) {
      const int h = i >> 5, l = i & 31;
      const uint8_t a = lv[128 * h + l], bb = lv[128 * h + l + 32], c = lv[128 * h + l + 64], e = lv[128 * h + l + 96];
      b[64 * h + l] = dead ? 0 : (a & 15) | ((c & 15) << 4);
      b[64 * h + l + 32] = dead ? 0 : (bb & 15) | ((e & 15) << 4);
      b[128 + 32 * h + l] = dead ? 0 : (a >> 4) | ((bb >> 4) << 2) | ((c >> 4) << 4) | ((e >> 4) << 6);
    }
  }
  __syncthreads();
  store_wire(wire + blk0 * BPB, out, (int)(last + 1 - blk0) * BPB, lane, 64);
}

// four elements per load need the tensor's address to be a multiple of them
bool four_aligned(const void* w, int dtype) {
  return (reinterpret_cast<uintptr_t>(w) & (dtype == KQ_F32 ? 15 : 7)) == 0;
}

template <int C>
int launch_legacy(const void* w, int dtype, uint8_t* wire, int64_t nblocks, hipStream_t s) {
  const int64_t wgs = (nblocks + LEG_BLOCKS - 1) / LEG_BLOCKS;
  if (wgs > 0x7fffffff) return kq_set_error(KQ_ERR_INVALID, "quantize: tensor too large for one launch");
  hipLaunchKernelGGL(encode_legacy_kernel<C>, dim3((unsigned)wgs), dim3(LEG_THREADS), 0, s, w, dtype, wire, nblocks,
                     four_aligned(w, dtype));
  KQ_HIP_CHECK(hipGetLastError());
  return KQ_OK;
}

template <int C, int S>
int launch_k_shared(const void* w, int dtype, const float* im, uint8_t* wire, int64_t nblocks, int64_t bpr, hipStream_t s) {
  constexpr int NSB = 64 / (KGeom<C>::SUBS * S);
  const int64_t wgs = (nblocks + NSB - 1) / NSB;
  if (wgs > 0x7fffffff) return kq_set_error(KQ_ERR_INVALID, "quantize: tensor too large for one launch");
  hipLaunchKernelGGL((encode_k_kernel<C, S>), dim3((unsigned)wgs), dim3(64), 0, s, w, dtype, im, wire, nblocks, bpr,
                     four_aligned(w, dtype));
  KQ_HIP_CHECK(hipGetLastError());
  return KQ_OK;
}

// Up to this many waves of four lanes to a sub-block (one per SIMD) they share its candidates: latency counts, and it hardly depends
// on the weights.  us, four lanes / one and the bound, normally distributed, in [0, 1), 1000 + normal: q4_k 512 superblocks 22, 22,
// 20 / 24, 30, 70; 2048 22, 22, 20 / 25, 32, 84; 4096 30, 30, 29 / 25, 32, 84; q2_k 1024 21, 21, 17 / 22, 27, 41.
constexpr int64_t SHARED_WAVES = 1024;

template <int C>
int launch_k(const void* w, int dtype, const float* im, uint8_t* wire, int64_t nblocks, int64_t bpr, hipStream_t s) {
  if constexpr (C == KQ_Q2_K || C == KQ_Q4_K || C == KQ_Q5_K)
    if (nblocks * KGeom<C>::SUBS * 4 <= 64 * SHARED_WAVES) return launch_k_shared<C, 4>(w, dtype, im, wire, nblocks, bpr, s);
  return launch_k_shared<C, 1>(w, dtype, im, wire, nblocks, bpr, s);
}

}  // namespace

bool kq_encode_dev_supported(int codec) {
  switch (codec) {
    case KQ_Q8_0: case KQ_Q4_0: case KQ_Q4_1: case KQ_Q5_0: case KQ_Q5_1:
    case KQ_Q2_K: case KQ_Q3_K: case KQ_Q4_K: case KQ_Q5_K: case KQ_Q6_K:
      return true;
  }
  return false;
}

int kq_launch_encode(const void* w, int dtype, const float* im, uint8_t* wire, int64_t rows, int64_t K, int codec,
                     hipStream_t s) {
  const KqGeom g = kq_geom(codec);
  const int64_t bpr = K / g.wpb, nblocks = rows * bpr;
  switch (codec) {
    case KQ_Q8_0: return launch_legacy<KQ_Q8_0>(w, dtype, wire, nblocks, s);
    case KQ_Q4_0: return launch_legacy<KQ_Q4_0>(w, dtype, wire, nblocks, s);
    case KQ_Q4_1: return launch_legacy<KQ_Q4_1>(w, dtype, wire, nblocks, s);
    case KQ_Q5_0: return launch_legacy<KQ_Q5_0>(w, dtype, wire, nblocks, s);
    case KQ_Q5_1: return launch_legacy<KQ_Q5_1>(w, dtype, wire, nblocks, s);
    case KQ_Q2_K: return launch_k<KQ_Q2_K>(w, dtype, im, wire, nblocks, bpr, s);
    case KQ_Q3_K: return launch_k<KQ_Q3_K>(w, dtype, im, wire, nblocks, bpr, s);
    case KQ_Q4_K: return launch_k<KQ_Q4_K>(w, dtype, im, wire, nblocks, bpr, s);
    case KQ_Q5_K: return launch_k<KQ_Q5_K>(w, dtype, im, wire, nblocks, bpr, s);
    case KQ_Q6_K: return launch_k<KQ_Q6_K>(w, dtype, im, wire, nblocks, bpr, s);
  }
  return KQ_ERR_UNSUPPORTED;
}
