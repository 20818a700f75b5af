// rlk_normalize.hpp -- the second half of a normalised GAE: from the scan's per-workgroup
// statistics to the normalised advantages.
#pragma once
#include "rlk_launch.hpp"
#include "rlk_time_major.h"

namespace rlk {

// First launches of more workgroups than this have their partials summed by a tree of
// reduce_partials_kernel levels (kReduceSlice triples into one per level) until at most
// this many remain, which normalize_kernel's workgroups then each read.  The crossover,
// measured on MI355X (float32, µs per call): 2048 triples read directly 24.1, through one
// level 24.7 ([32768,128]); 4096 triples 44.9 directly, 42.5 through a level ([65536,128]).
// Against every normalising workgroup reading every triple, the tree takes [2^20,128]
// (65536 triples) from 761 to 630 µs and [16384,2048] from 167 to 139 µs.
constexpr int64_t kDirectParts = 2048;

// Triples of the partials buffer for a first launch of `nparts` workgroups: its own, then
// each tree level's.
inline int64_t partials_triples(int64_t nparts) {
  int64_t total = nparts;
  for (int64_t n = nparts; n > kDirectParts;) {
    n = (n + kReduceSlice - 1) / kReduceSlice;
    total += n;
  }
  return total;
}

inline bool partials_fit(const void* partials, size_t bytes, int64_t nparts) {
  return partials != nullptr && (reinterpret_cast<uintptr_t>(partials) & 7u) == 0 && nparts <= 0x7fffffffLL &&
         bytes >= (size_t)partials_triples(nparts) * kStatWords * sizeof(double);
}

// The one-launch form a call asks for (c.sync != nullptr).
inline OneLaunch one_launch(const rlk_time_major_call& c) {
  return {static_cast<uint64_t*>(c.sync), c.epoch, g_fallback_polls.load(std::memory_order_relaxed), c.eps};
}

// Rewrites the n advantages as (A - mean) / (std + eps), from the first launch's nparts triples
// at the start of the partials buffer.
template <class E>
int normalize(E* advantages, double* parts, int64_t nparts, int64_t n, float eps, hipStream_t s) {
  int np = (int)nparts;
  while (np > kDirectParts) {
    const int next = (np + kReduceSlice - 1) / kReduceSlice;
    double* up = parts + kStatWords * (int64_t)np;
    void* rargs[] = {&parts, &np, &up};
    if (hipLaunchKernel(reinterpret_cast<const void*>(&reduce_partials_kernel<kReduceNT>),
                        dim3((unsigned)next), dim3(kReduceNT), rargs, 0, s) != hipSuccess)
      return RLK_ERR_LAUNCH;
    parts = up;
    np = next;
  }
  constexpr int kNormNT = 256;
  const bool nvec = n % 4 == 0 && quad_aligned(advantages);
  const int64_t units = nvec ? n / 4 : n;
  int64_t grid = (units + kNormNT - 1) / kNormNT;
  if (grid > 2048) grid = 2048;
  void* args[] = {&advantages, &parts, &np, &n, &eps};
  const void* kernel = nvec ? reinterpret_cast<const void*>(&normalize_kernel<kNormNT, true, E>)
                            : reinterpret_cast<const void*>(&normalize_kernel<kNormNT, false, E>);
  const hipError_t e = hipLaunchKernel(kernel, dim3((unsigned)grid), dim3(kNormNT), args, 0, s);
  return e == hipSuccess ? RLK_OK : RLK_ERR_LAUNCH;
}

}  // namespace rlk
