// rlk_gae_normalized.hip -- normalised GAE entry points (include/rl_triton_amd.h).
#include "rlk_launch.hpp"

namespace rlk {
namespace {

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
int64_t partials_triples(int64_t nparts) {
  int64_t total = nparts;
  for (int64_t n = nparts; n > kDirectParts;) {
    n = (n + kReduceSlice - 1) / kReduceSlice;
    total += n;
  }
  return total;
}

// Partials of compute_gae_normalized: kStatWords doubles per workgroup of the first launch
// and per tree level, for the larger of the two ops' grids (the masked op uses narrower
// long-row tiles).
size_t gae_normalized_partials(int64_t num_envs, int64_t seq_len) {
  if (num_envs <= 0 || seq_len <= 0) return 0;
  const int64_t a = call_blocks<GaeStatsOp<true>>(num_envs, seq_len);
  const int64_t b = call_blocks<MaskedGaeStatsOp<true>>(num_envs, seq_len);
  return (size_t)partials_triples(a > b ? a : b) * kStatWords * sizeof(double);
}

// The two launches of a normalised GAE: `op` (GaeStatsOp or MaskedGaeStatsOp, partials not
// yet set) writes A, the returns and the per-workgroup statistics; normalize_kernel then
// rewrites A as (A - mean) / (std + eps).
template <class StatsOp, class E>
int normalized_launch(StatsOp op, E* advantages, int64_t num_envs, int64_t seq_len, bool vec,
                      float eps, void* workspace, size_t workspace_bytes, void* partials,
                      size_t partials_bytes, void* stream) {
  if (num_envs < 0 || seq_len < 0 || seq_len > (int64_t{1} << 30)) return RLK_ERR_INVALID_ARGUMENT;
  double* parts = reinterpret_cast<double*>(partials);
  const int64_t nparts = call_blocks<StatsOp>(num_envs, seq_len);
  if (parts == nullptr || (reinterpret_cast<uintptr_t>(parts) & 7u) != 0 ||
      partials_bytes < (size_t)partials_triples(nparts) * kStatWords * sizeof(double) ||
      nparts > 0x7fffffffLL)
    return RLK_ERR_WORKSPACE;
  op.partials = parts;
  const int st = launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream);
  if (st != RLK_OK) return st;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
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
  int64_t n = num_envs * seq_len;
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

// mask == nullptr: every step counts (GaeStatsOp); otherwise the masked op
template <class E>
int gae_normalized_impl(const E* rewards, const E* values, const E* terminateds,
                        const E* truncateds, const E* bootstrap, int boot_mode, const E* mask,
                        E* advantages, E* returns, int64_t num_envs, int64_t seq_len, float gamma,
                        float lambda_, float eps, void* workspace, size_t workspace_bytes,
                        void* partials, size_t partials_bytes, void* stream) {
  if (is_empty(num_envs, seq_len)) return RLK_OK;
  if (!rewards || !values || !terminateds || !advantages || !returns ||
      !valid_boot(bootstrap, boot_mode))
    return RLK_ERR_INVALID_ARGUMENT;
  const E* boot = boot_mode == RLK_BOOT_NONE ? nullptr : bootstrap;
  const bool vec = seq_len % 4 == 0 &&
                   quad_aligned(rewards, values, terminateds, truncateds, mask, advantages,
                                returns) &&
                   (boot_mode != RLK_BOOT_FULL || quad_aligned(bootstrap));
  const float gl = gamma * lambda_;
  auto run = [&](auto op) {
    return normalized_launch(op, advantages, num_envs, seq_len, vec, eps, workspace,
                             workspace_bytes, partials, partials_bytes, stream);
  };
  if (mask) {
    if (truncateds)
      return run(MaskedGaeStatsOp<true, E>{{rewards, values, terminateds, truncateds, boot, mask,
                                             advantages, boot_mode, gamma, gl},
                                            returns, nullptr});
    return run(MaskedGaeStatsOp<false, E>{{rewards, values, terminateds, nullptr, boot, mask,
                                            advantages, boot_mode, gamma, gl},
                                           returns, nullptr});
  }
  if (truncateds)
    return run(GaeStatsOp<true, E>{{rewards, values, terminateds, truncateds, boot, advantages,
                                     boot_mode, gamma, gl},
                                    returns, nullptr});
  return run(GaeStatsOp<false, E>{{rewards, values, terminateds, nullptr, boot, advantages,
                                    boot_mode, gamma, gl},
                                   returns, nullptr});
}

}  // namespace
}  // namespace rlk

using namespace rlk;

extern "C" {

size_t rlk_gae_normalized_partials_bytes(int64_t num_envs, int64_t seq_len) {
  return gae_normalized_partials(num_envs, seq_len);
}

int rlk_gae_normalized(const float* rewards, const float* values, const float* terminateds,
                       const float* truncateds, const float* bootstrap, int boot_mode,
                       float* advantages, float* returns, int64_t num_envs, int64_t seq_len,
                       float gamma, float lambda_, float eps, void* workspace,
                       size_t workspace_bytes, void* partials, size_t partials_bytes,
                       void* stream) {
  return gae_normalized_impl<float>(rewards, values, terminateds, truncateds, bootstrap,
                                    boot_mode, nullptr, advantages, returns, num_envs, seq_len,
                                    gamma, lambda_, eps, workspace, workspace_bytes, partials,
                                    partials_bytes, stream);
}

int rlk_gae_normalized_bf16(const rlk_bf16* rewards, const rlk_bf16* values,
                            const rlk_bf16* terminateds, const rlk_bf16* truncateds,
                            const rlk_bf16* bootstrap, int boot_mode, rlk_bf16* advantages,
                            rlk_bf16* returns, int64_t num_envs, int64_t seq_len, float gamma,
                            float lambda_, float eps, void* workspace, size_t workspace_bytes,
                            void* partials, size_t partials_bytes, void* stream) {
  return gae_normalized_impl<bf16>(B(rewards), B(values), B(terminateds), B(truncateds),
                                   B(bootstrap), boot_mode, nullptr, B(advantages), B(returns),
                                   num_envs, seq_len, gamma, lambda_, eps, workspace,
                                   workspace_bytes, partials, partials_bytes, stream);
}

int rlk_gae_normalized_masked(const float* rewards, const float* values,
                              const float* terminateds, const float* truncateds,
                              const float* bootstrap, int boot_mode, const float* mask,
                              float* advantages, float* returns, int64_t num_envs,
                              int64_t seq_len, float gamma, float lambda_, float eps,
                              void* workspace, size_t workspace_bytes, void* partials,
                              size_t partials_bytes, void* stream) {
  if (!is_empty(num_envs, seq_len) && !mask) return RLK_ERR_INVALID_ARGUMENT;
  return gae_normalized_impl<float>(rewards, values, terminateds, truncateds, bootstrap,
                                    boot_mode, mask, advantages, returns, num_envs, seq_len,
                                    gamma, lambda_, eps, workspace, workspace_bytes, partials,
                                    partials_bytes, stream);
}

int rlk_gae_normalized_masked_bf16(const rlk_bf16* rewards, const rlk_bf16* values,
                                   const rlk_bf16* terminateds, const rlk_bf16* truncateds,
                                   const rlk_bf16* bootstrap, int boot_mode, const rlk_bf16* mask,
                                   rlk_bf16* advantages, rlk_bf16* returns, int64_t num_envs,
                                   int64_t seq_len, float gamma, float lambda_, float eps,
                                   void* workspace, size_t workspace_bytes, void* partials,
                                   size_t partials_bytes, void* stream) {
  if (!is_empty(num_envs, seq_len) && !mask) return RLK_ERR_INVALID_ARGUMENT;
  return gae_normalized_impl<bf16>(B(rewards), B(values), B(terminateds), B(truncateds),
                                   B(bootstrap), boot_mode, B(mask), B(advantages), B(returns),
                                   num_envs, seq_len, gamma, lambda_, eps, workspace,
                                   workspace_bytes, partials, partials_bytes, stream);
}

}  // extern "C"
