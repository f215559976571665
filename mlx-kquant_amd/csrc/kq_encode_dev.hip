// Device-side wire encoder behind kq_quantize_dev: the legacy 32-weight codecs and the K-quant superblock codecs.
// The bytes equal kq_quantize's: every value is computed by the expressions of kq_encode_blocks.h, in its order of
// additions, unfused.  The reference's GPU encoders cover the same codecs (metal/.../kq_quantized_encode.h); its IQ
// encoders are CPU-only (src/kquant_ops.cpp:602-606), as here.
//
// What bounds it.  K-quants: the vector ALU.  A sub-block's fit tries 37 (scale, min) or 19 scale candidates, and the
// order of its sums is part of the result, so a candidate is one lane's serial work: 15 (8) instructions per weight and
// candidate that cannot be fused.  16.8 M weights of q4_k are 1.5e8 wave instructions = 240 us at the chip's issue rate,
// against 32 us of memory traffic.  One lane per sub-block (8 or 16 per superblock) keeps all three arrays of a fit in
// registers; one thread per superblock, the form this replaced, kept them in 2.4 KB of scratch per lane.  4096 x 4096
// f32: q4_k 3527 -> 222 us (q5_k 261, q2_k 338, q3_k 82, q6_k 78).
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
// One wave per workgroup.  Lane = (superblock, sub-block j, part s): S lanes share a sub-block's candidates.  S > 1 is
// for matrices whose sub-blocks are too few to fill the chip; the lanes of a sub-block redo everything outside the
// candidate scan, so it costs instructions where they are not short of waves.
template <int C>
struct KGeom {
  static constexpr int SUBS = C == KQ_Q4_K || C == KQ_Q5_K ? 8 : 16, N = 256 / SUBS;
  static constexpr int NMAX = C == KQ_Q2_K ? 3 : C == KQ_Q4_K ? 15 : 31;  // of the (scale, min) codecs
};

// kqenc::fit_scale_min.  A candidate replaces the best one if its error is strictly smaller, so the scan's result is the
// earliest candidate of least error whatever order they are tried in: part s tries steps s, s + S, ... and the parts
// are compared afterwards.
template <int N, int NMAX, int S>
__device__ __forceinline__ float fit_scale_min(const float (&x)[N], const float (&wt)[N], int part, float& neg_min) {
  float vmin = x[0], vmax = x[0], sw = wt[0], swx = sw * x[0];
#pragma unroll
  for (int i = 1; i < N; i++) {
    if (x[i] < vmin) vmin = x[i];
    if (x[i] > vmax) vmax = x[i];
    sw += wt[i];
    swx += wt[i] * x[i];
  }
  if (vmin > 0.f) vmin = 0.f;
  const bool flat = vmax <= vmin;
  const float range = vmax - vmin;
  float scale, best_min = vmin, best_err = 0.f;
  {
    const float inv = float(NMAX) / range;
    scale = 1.0f / inv;
#pragma unroll
    for (int i = 0; i < N; i++) {
      const float l = clamp_level(inv * (x[i] - vmin), 0.f, float(NMAX));
      const float e = scale * l + vmin - x[i];
      best_err += wt[i] * e * e;
    }
  }
  int best_step = -1;
#pragma unroll 1
  for (int step = part; step <= 36; step += S) {
    const float inv_s = (-0.9f + 0.05f * float(step) + float(NMAX)) / range;
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
    if (det > 0.f && err < best_err) {
      best_err = err;
      scale = s;
      best_min = m;
      best_step = step;
    }
  }
#pragma unroll
  for (int m = 1; m < S; m <<= 1) {
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

// kqenc::fit_positive of the sub-block scales (which = 0) and of the minima (1): both arrays lie in LDS.  The nine-point
// scan takes one candidate per lane of an octet (again the earliest of least error wins); the refinement, whose steps
// depend on each other, runs on the even lanes for the scales and on the odd ones for the minima.  Returns the factor
// of the lane's array and leaves its levels in lv.
template <int N, int NMAX>
__device__ __forceinline__ float fit_positive_pair(const float* sc, const float* mn, const float* sw, int lane,
                                                   int (&lv)[N]) {
  float wt[N], inv_of[2];
#pragma unroll
  for (int i = 0; i < N; i++) wt[i] = sw[i];
  float x[N];
#pragma unroll
  for (int which = 0; which < 2; which++) {
    const float* src = which ? mn : sc;
    float vmax = 0.f;
#pragma unroll
    for (int i = 0; i < N; i++) {
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
    const int c = lane & 7, k = c < 4 ? c - 4 : c - 3;
    float inv_k = (0.1f * float(k) + float(NMAX)) / vmax, err = 0.f;
    const float s_k = 1.0f / inv_k;
#pragma unroll
    for (int i = 0; i < N; i++) {
      const int l = min(NMAX, kqenc::rne(inv_k * x[i]));
      const float e = x[i] - s_k * float(l);
      err += wt[i] * e * e;
    }
    int order = c;
#pragma unroll
    for (int m = 1; m < 8; m <<= 1) {
      const float oe = __shfl_xor(err, m), oi = __shfl_xor(inv_k, m);
      const int oo = __shfl_xor(order, m);
      if (oe < err || (oe == err && oo < order) || !(err == err)) {
        err = oe;
        inv_k = oi;
        order = oo;
      }
    }
    inv_of[which] = vmax < 1e-30f ? -1.f : err < best ? inv_k : inv;
  }
  const bool odd = lane & 1;
  const float inv = odd ? inv_of[1] : inv_of[0];
  const float* src = odd ? mn : sc;
  float slx = 0.f, sl2 = 0.f;
#pragma unroll
  for (int i = 0; i < N; i++) {
    x[i] = src[i];
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
      const int nl = min(NMAX, kqenc::rne(x[i] * b / a));
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
__global__ __launch_bounds__(64) void encode_k_kernel(const void* __restrict__ w, int dtype,
                                                      const float* __restrict__ imatrix, uint8_t* __restrict__ wire,
                                                      int64_t nblocks, int64_t blocks_per_row, bool aligned) {
  constexpr int BPB = kq_geom(C).bpb, SUBS = KGeom<C>::SUBS, N = KGeom<C>::N;
  constexpr int GROUP = SUBS * S, NSB = 64 / GROUP;  // lanes per superblock, superblocks per wave
  constexpr int XS = 256 + 4;                        // floats between superblocks in LDS: eight of them in eight banks
  constexpr bool kMin = C == KQ_Q2_K || C == KQ_Q4_K || C == KQ_Q5_K;
  __shared__ __attribute__((aligned(16))) float xs[NSB * XS];
  __shared__ float s_sc[NSB][SUBS], s_mn[NSB][SUBS], s_sw[NSB][SUBS];
  __shared__ __attribute__((aligned(16))) uint8_t s_lv[NSB][256];
  __shared__ int s_ls[NSB][SUBS], s_lm[NSB][SUBS];
  __shared__ __attribute__((aligned(16))) uint8_t out[NSB * BPB];
  const int lane = threadIdx.x, sb = lane / GROUP, gl = lane % GROUP, j = gl / S, part = gl % S;
  const int64_t blk0 = (int64_t)blockIdx.x * NSB;
  for (int i = lane; i < NSB * 64; i += 64) {
    // superblocks past the end redo the last one; their bytes are not stored
    const int64_t blk = min(blk0 + (i >> 6), nblocks - 1);
    *reinterpret_cast<float4*>(xs + (i >> 6) * XS + 4 * (i & 63)) = load4_any(w, dtype, blk * 256 + 4 * (i & 63), aligned);
  }
  __syncthreads();
  const float* xb = xs + sb * XS;
  float x[N], wt[N];
#pragma unroll
  for (int i = 0; i < N; i++) x[i] = xb[N * j + i];

  // importance weights (kqenc::importance; q6_k weights by the matrix itself, q3_k and q6_k by x^2 without one)
  const float* im = nullptr;
  if (imatrix) im = imatrix + (min(blk0 + sb, nblocks - 1) % blocks_per_row) * 256 + N * j;
  if (C == KQ_Q6_K || (C == KQ_Q3_K && !im)) {
#pragma unroll
    for (int i = 0; i < N; i++) wt[i] = im ? im[i] : x[i] * x[i];
  } else {
    float total = 0.f;
#pragma unroll 16
    for (int i = 0; i < 256; i++) total += xb[i] * xb[i];
    const float sigma2 = (C == KQ_Q2_K ? 1.0f : 2.0f) * total / 256.0f, av = std::sqrt(sigma2);
    if (im) {
#pragma unroll
      for (int i = 0; i < N; i++) wt[i] = im[i] * std::sqrt(sigma2 + x[i] * x[i]);
    } else {
#pragma unroll
      for (int i = 0; i < N; i++) wt[i] = av + std::fabs(x[i]);
    }
  }

  uint8_t* b = out + sb * BPB;
  if constexpr (kMin) {
    float sw = 0.f, neg_min;
#pragma unroll
    for (int i = 0; i < N; i++) sw += wt[i];
    const float sc = fit_scale_min<N, KGeom<C>::NMAX, S>(x, wt, part, neg_min);
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
#pragma unroll
    for (int i = 0; i < N; i++)
      if (i % S == part)
        s_lv[sb][N * j + i] = ds == 0.f ? 0 : (uint8_t)(int)clamp_level((x[i] + dm) / ds, 0.f, float(KGeom<C>::NMAX));
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
#pragma unroll
    for (int i = 0; i < N; i++)
      s_lv[sb][N * j + i] =
          de == 0.f ? NMAX : (uint8_t)((int)clamp_level_signed(x[i] / de, -float(NMAX), float(NMAX - 1)) + NMAX);
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
  const int64_t left = nblocks - blk0;
  store_wire(wire + blk0 * BPB, out, (int)(left < NSB ? left : NSB) * BPB, lane, 64);
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
int launch_k_split(const void* w, int dtype, const float* im, uint8_t* wire, int64_t nblocks, int64_t bpr, hipStream_t s) {
  constexpr int NSB = 64 / (KGeom<C>::SUBS * S);
  const int64_t wgs = (nblocks + NSB - 1) / NSB;
  if (wgs > 0x7fffffff) return kq_set_error(KQ_ERR_INVALID, "quantize: tensor too large for one launch");
  hipLaunchKernelGGL((encode_k_kernel<C, S>), dim3((unsigned)wgs), dim3(64), 0, s, w, dtype, im, wire, nblocks, bpr,
                     four_aligned(w, dtype));
  KQ_HIP_CHECK(hipGetLastError());
  return KQ_OK;
}

// Below this many waves of whole sub-blocks (one per SIMD) four lanes share one's candidates.  One lane / four lanes,
// us: q4_k 16384 superblocks 70 / 87, 8192 (1024 waves) 50 / 49, 4096 49 / 30, 2048 49 / 23; q2_k 8192 (2048 waves)
// 53 / 65, 4096 37 / 40, 2048 37 / 27.
constexpr int64_t SPLIT_WAVES = 1024;

template <int C>
int launch_k(const void* w, int dtype, const float* im, uint8_t* wire, int64_t nblocks, int64_t bpr, hipStream_t s) {
  if constexpr (C == KQ_Q2_K || C == KQ_Q4_K || C == KQ_Q5_K)
    if (nblocks * KGeom<C>::SUBS < 64 * SPLIT_WAVES) return launch_k_split<C, 4>(w, dtype, im, wire, nblocks, bpr, s);
  return launch_k_split<C, 1>(w, dtype, im, wire, nblocks, bpr, s);
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
