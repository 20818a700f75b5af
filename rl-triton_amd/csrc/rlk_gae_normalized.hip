// rlk_gae_normalized.hip -- normalised GAE entry points (include/rl_triton_amd.h).
#include "rlk_launch.hpp"
#include "rlk_normalize.hpp"

namespace rlk {
namespace {

// Partials of compute_gae_normalized: kStatWords doubles per workgroup of the first launch
// and per tree level, for the larger of the two ops' grids (the masked op uses narrower
// long-row tiles).
size_t gae_normalized_partials(int64_t num_envs, int64_t seq_len) {
  if (num_envs <= 0 || seq_len <= 0) return 0;
  const CusScope cus;
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
  const CusScope cus;
  const int64_t nparts = call_blocks<StatsOp>(num_envs, seq_len);
  if (!partials_fit(partials, partials_bytes, nparts)) return RLK_ERR_WORKSPACE;
  op.partials = reinterpret_cast<double*>(partials);
  const int st = launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream);
  if (st != RLK_OK) return st;
  return normalize(advantages, op.partials, nparts, num_envs * seq_len, eps, reinterpret_cast<hipStream_t>(stream));
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

static_assert(RLK_NORM_SYNC_BYTES == kNormSyncWords * sizeof(uint64_t) && RLK_NORM_MAX_EPOCH == kNormMaxEpoch,
              "the sync buffer's layout");

// One launch, or kNotTaken.
template <class E>
int one_launch_impl(const rlk_time_major_call& c, void* stream) {
  auto in = [&](int i) { return static_cast<const E*>(c.in[i]); };
  E *adv = static_cast<E*>(c.out[0]), *ret = static_cast<E*>(c.out[1]);
  if (!in(0) || !in(1) || !in(2) || !adv || !ret || !c.sync || c.epoch == 0 || c.epoch > kNormMaxEpoch ||
      !valid_boot(c.bootstrap, c.boot_mode))
    return RLK_ERR_INVALID_ARGUMENT;
  const E* boot = c.boot_mode == RLK_BOOT_NONE ? nullptr : static_cast<const E*>(c.bootstrap);
  const bool vec = c.seq_len % 4 == 0 && quad_aligned(in(0), in(1), in(2), in(3), in(4), adv, ret) &&
                   (c.boot_mode != RLK_BOOT_FULL || quad_aligned(boot));
  const float gl = c.gamma * c.lambda_;
  auto run = [&](auto op) {
    return launch(OneLaunchOp<decltype(op)>{op, one_launch(c)}, c.num_envs, c.seq_len, vec, nullptr, 0, stream);
  };
  if (in(4)) {
    if (in(3))
      return run(MaskedGaeStatsOp<true, E>{{in(0), in(1), in(2), in(3), boot, in(4), adv, c.boot_mode, c.gamma, gl},
                                           ret, nullptr});
    return run(MaskedGaeStatsOp<false, E>{{in(0), in(1), in(2), nullptr, boot, in(4), adv, c.boot_mode, c.gamma, gl},
                                          ret, nullptr});
  }
  if (in(3))
    return run(GaeStatsOp<true, E>{{in(0), in(1), in(2), in(3), boot, adv, c.boot_mode, c.gamma, gl}, ret, nullptr});
  return run(GaeStatsOp<false, E>{{in(0), in(1), in(2), nullptr, boot, adv, c.boot_mode, c.gamma, gl}, ret, nullptr});
}

}  // namespace
}  // namespace rlk

using namespace rlk;

extern "C" {

int rlk_gae_normalized_one_launch_takes(int64_t num_envs, int64_t seq_len, int masked) {
  // Asked ahead of every call: one that launch() then refused would pay for both forms on the host
  // ([1000,500] 8.1 us per call, 7.8 so).
  const int64_t E = num_envs, T = seq_len;
  if (E <= 0 || T <= 0 || T > 4 * kWholeRowThreads * kSeg) return 0;
  const int64_t most = T > kShortMaxT || T % 4 == 0 ? one_launch_blocks(T, masked != 0) : kNormPollers;
  if (T > kShortMaxT / 2)  // a workgroup per row
    return E <= most && (T <= kShortMaxT || whole_row_segments<GaeStatsOp<true>>(E, T, true) > 0) ? 1 : 0;
  // the finest grid, the coarsest, else the one it is
  if (rows_grid(E, T, rows_seg(T), kNT) <= most) return 1;
  if (rows_grid(E, T, rows_seg(T), kNTWide) > most) return 0;
  return launch_grid<GaeStatsOp<true>>(E, T) <= most ? 1 : 0;
}

int rlk_gae_normalized_one_launch(const rlk_time_major_call* call, void* stream) {
  if (is_empty(call->num_envs, call->seq_len)) return kNotTaken;
  return call->bf16 ? one_launch_impl<bf16>(*call, stream) : one_launch_impl<float>(*call, stream);
}

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
