// The entries of one expert in the id list of a gathered call, found by a workgroup of 256 threads: for the kernels whose
// workgroups belong to an expert and look for their rows themselves (a list of at most 1024 ids, read by all of them at once).
// An expert's rows are done in rounds of so many rows, and the grid has `cap` workgroups for each expert (and column tile), at
// least for the rounds of an average expert.  Experts with more leave rounds over, which the workgroups of smaller experts take
// (share_rounds): in series on their own workgroups they made 1024 entries on one expert up to 70 times as long as even shares.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace kqentries {

constexpr int THREADS = 256, WAVES = THREADS / 64, MAX_ENTRIES = 1024, PER_THREAD = MAX_ENTRIES / THREADS;

// In LDS; place p of the expert's entries, in the order of the list (the same in every workgroup of the expert)
struct Places {
  int4 counts[PER_THREAD];  // hits of the four waves, by 256 ids of the list
  int entry_of[MAX_ENTRIES];
  uint32_t lhs_of[MAX_ENTRIES];
};

struct Ids {
  uint32_t id[PER_THREAD], lhs[PER_THREAD];

  __device__ __forceinline__ void load(const uint32_t* rhs, const uint32_t* lhs_list, int B, int tid) {
#pragma unroll
    for (int u = 0; u < PER_THREAD; u++) {
      if (THREADS * u >= B) break;  // uniform
      const int j = tid + THREADS * u;
      id[u] = j < B ? rhs[j] : ~0u;
      lhs[u] = j < B ? lhs_list[j] : 0u;
    }
  }

  // The number of entries; their places are in LDS after the caller's next barrier.
  template <class Barrier>
  __device__ __forceinline__ int find(uint32_t expert, int B, int tid, int wave, Places& p, Barrier barrier) const {
    const int lane = tid & 63;
    uint64_t hit[PER_THREAD];
#pragma unroll
    for (int u = 0; u < PER_THREAD; u++) {
      if (THREADS * u >= B) break;
      hit[u] = __builtin_amdgcn_ballot_w64(id[u] == expert);
      if (lane == 0) reinterpret_cast<int*>(&p.counts[u])[wave] = __builtin_popcountll(hit[u]);
    }
    barrier();
    int count = 0;
#pragma unroll
    for (int u = 0; u < PER_THREAD; u++) {
      if (THREADS * u >= B) break;
      const int4 n = p.counts[u];
      const int before = (wave > 0 ? n.x : 0) + (wave > 1 ? n.y : 0) + (wave > 2 ? n.z : 0);
      if ((hit[u] >> lane) & 1) {
        const int place = count + before + __builtin_popcountll(hit[u] & ((1ull << lane) - 1));
        p.entry_of[place] = tid + THREADS * u;
        p.lhs_of[place] = lhs[u];
      }
      count += n.x + n.y + n.z + n.w;
    }
    return __builtin_amdgcn_readfirstlane(count);
  }
};

constexpr int MAX_EXPERTS = 4096, EXPERT_BITS = 12;
constexpr uint32_t NO_ROUND = ~0u;
static_assert(MAX_EXPERTS <= 1 << EXPERT_BITS);

struct Share {
  uint32_t sums[WAVES], own, round, left;  // left: some expert has more rounds than workgroups
};

// Entries per expert, sixteen bits each, in LDS: experts 2 i and 2 i + 1 in word i.  Counted beside the search (four LDS atomics
// a thread), so that a call without rounds left over, which is most, ends where it did.
constexpr size_t count_bytes(int E) { return (size_t)(E + 1) / 2 * 4; }
__device__ __forceinline__ int count_of(const uint32_t* cnt, int e) { return (int)((cnt[e >> 1] >> (16 * (e & 1))) & 0xffffu); }

// Ids::find for the workgroup's own expert, and the counts of all, complete after the caller's next barrier.
template <class Barrier>
__device__ __forceinline__ int find_and_count(const Ids& ids, uint32_t expert, int B, int E, int tid, int wave, Places& p,
                                              uint32_t* cnt, Share& share, Barrier barrier) {
#pragma unroll 1
  for (int i = tid; i < (E + 1) / 2; i += THREADS) cnt[i] = 0;
  if (tid == 0) {
    share.left = 0;
    share.round = NO_ROUND;
  }
  const int count = ids.find(expert, B, tid, wave, p, barrier);
#pragma unroll
  for (int u = 0; u < PER_THREAD; u++) {
    if (THREADS * u >= B) break;
    if (ids.id[u] < (uint32_t)E) atomicAdd(&cnt[ids.id[u] >> 1], 1u << (16 * (ids.id[u] & 1)));
  }
  return count;
}

// share.left, known after the caller's next barrier: where the workgroup waits for loads
template <int ROWS>
__device__ __forceinline__ void note_left(int M, int E, int cap, int tid, const uint32_t* cnt, Share& share) {
  bool left = false;
#pragma unroll 1
  for (int e = tid; e < E; e += THREADS) left |= count_of(cnt, e) * M > ROWS * cap;
  if (left) share.left = 1;
}

// Whether a workgroup that has done its own round takes one of those left over: its expert leaves some, or has fewer rows than
// the average.  B M <= 2^20.
template <int ROWS>
__device__ __forceinline__ bool shares_rounds(int rows, int B, int M, int E, int cap) {
  return rows > ROWS * cap || (uint32_t)rows * (uint32_t)E < (uint32_t)B * (uint32_t)M;
}

// The rounds left over, one each to the workgroups that take some: all of an expert for which shares_rounds holds, those
// without a round of their own of the others; every one comes to the same numbering.  For workgroup y of expert `own`:
// round << EXPERT_BITS | expert, or NO_ROUND.
// cap >= B M / E / ROWS, so one each is enough: an expert above the average leaves less than (its rows - average) / ROWS + 1
// over, and what is above the average in all is missing below it, where `cap` workgroups of each expert are free.
// E <= MAX_EXPERTS; rounds and workgroups of all experts below 2^16 (B M / ROWS and E cap).
template <int ROWS, class Barrier>
__device__ __forceinline__ uint32_t share_rounds(int B, int M, int E, int cap, uint32_t own, int y, int tid, const uint32_t* cnt,
                                                 Share& share, Barrier barrier) {
  // nothing of this is computed ahead of the round that comes before
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63, wave = tid >> 6;
  // thread t owns experts e0 ... e1 - 1; rounds left over in the low half, workgroups that take some in the high half
  const int chunk = (E + THREADS - 1) / THREADS, e0 = min(tid * chunk, E), e1 = min(e0 + chunk, E);
  auto shares = [&](int e, int& rounds) {
    const int rows = count_of(cnt, e) * M;
    rounds = (rows + ROWS - 1) / ROWS;
    const uint32_t over = (uint32_t)(rounds > cap ? rounds - cap : 0);
    return over | (uint32_t)(shares_rounds<ROWS>(rows, B, M, E, cap) ? cap : rounds < cap ? cap - rounds : 0) << 16;
  };
  uint32_t sum = 0;
  int rounds;
#pragma unroll 1
  for (int e = e0; e < e1; e++) sum += shares(e, rounds);
  uint32_t incl = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t v = (uint32_t)__shfl_up((int)incl, off);
    if (lane >= off) incl += v;
  }
  if (lane == 63) share.sums[wave] = incl;
  barrier();
  uint32_t before = incl - sum;
#pragma unroll
  for (int w = 0; w < WAVES; w++)
    if (w < wave) before += share.sums[w];
  uint32_t me = 0;
#pragma unroll 1
  for (int pass = 0; pass < 2; pass++) {  // this workgroup's number; the round of that number
    uint32_t run = before;
#pragma unroll 1
    for (int e = e0; e < e1; e++) {
      const uint32_t v = shares(e, rounds), s = run & 0xffffu;
      if (pass == 0) {
        if ((uint32_t)e == own) share.own = (run >> 16) + (uint32_t)((int)(v >> 16) == cap ? y : y - rounds);
      } else if (me - s < (v & 0xffffu)) {
        share.round = (uint32_t)e | ((uint32_t)cap + me - s) << EXPERT_BITS;
      }
      run += v;
    }
    barrier();
    me = share.own;
  }
  return __builtin_amdgcn_readfirstlane(share.round);
}

}  // namespace kqentries
