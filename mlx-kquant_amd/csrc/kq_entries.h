// The entries of one expert in the id list of a gathered call, found by a workgroup of 256 threads: for the kernels whose
// workgroups belong to an expert and look for their rows themselves (a list of at most 1024 ids, read by all of them at once).
#pragma once

#include <hip/hip_runtime.h>
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
    return count;
  }
};

}  // namespace kqentries
