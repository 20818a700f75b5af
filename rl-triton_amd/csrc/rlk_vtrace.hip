// rlk_vtrace.hip -- V-trace entry points (include/rl_triton_amd.h).
#include "rlk_launch.hpp"

namespace rlk {
namespace {

template <class E>
int vtrace_impl(const E* log_pi_target, const E* log_pi_behavior, const E* values,
                const E* rewards, const E* terminateds, const E* truncateds, const E* bootstrap,
                int boot_mode, E* targets, E* advantages, int64_t num_envs, int64_t seq_len,
                float gamma, float rho_bar, float c_bar, void* workspace, size_t workspace_bytes,
                void* stream) {
  if (is_empty(num_envs, seq_len)) return RLK_OK;
  if (!log_pi_target || !log_pi_behavior || !values || !rewards || !terminateds || !targets ||
      !advantages || !valid_boot(bootstrap, boot_mode))
    return RLK_ERR_INVALID_ARGUMENT;
  const E* boot = boot_mode == RLK_BOOT_NONE ? nullptr : bootstrap;
  const bool vec = seq_len % 4 == 0 &&
                   quad_aligned(log_pi_target, log_pi_behavior, values, rewards, terminateds,
                                truncateds, targets, advantages) &&
                   (boot_mode != RLK_BOOT_FULL || quad_aligned(bootstrap));
  const int ph = common_phase<E>(log_pi_target, log_pi_behavior, values, rewards, terminateds,
                                 truncateds, targets, advantages,
                                 boot_mode == RLK_BOOT_FULL ? bootstrap : nullptr);
  if (truncateds) {
    VtraceOp<true, E> op{log_pi_target, log_pi_behavior, values, rewards, terminateds, truncateds,
                         boot, targets, advantages, boot_mode, gamma, rho_bar, c_bar};
    return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream, ph);
  }
  VtraceOp<false, E> op{log_pi_target, log_pi_behavior, values, rewards, terminateds, nullptr,
                        boot, targets, advantages, boot_mode, gamma, rho_bar, c_bar};
  return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream, ph);
}

}  // namespace
}  // namespace rlk

using namespace rlk;

extern "C" {

int rlk_vtrace(const float* log_pi_target, const float* log_pi_behavior, const float* values,
               const float* rewards, const float* terminateds, const float* truncateds,
               const float* bootstrap, int boot_mode, float* targets, float* advantages,
               int64_t num_envs, int64_t seq_len, float gamma, float rho_bar, float c_bar,
               void* workspace, size_t workspace_bytes, void* stream) {
  return vtrace_impl(log_pi_target, log_pi_behavior, values, rewards, terminateds, truncateds,
                     bootstrap, boot_mode, targets, advantages, num_envs, seq_len, gamma, rho_bar,
                     c_bar, workspace, workspace_bytes, stream);
}

int rlk_vtrace_bf16(const rlk_bf16* log_pi_target, const rlk_bf16* log_pi_behavior,
                    const rlk_bf16* values, const rlk_bf16* rewards, const rlk_bf16* terminateds,
                    const rlk_bf16* truncateds, const rlk_bf16* bootstrap, int boot_mode,
                    rlk_bf16* targets, rlk_bf16* advantages, int64_t num_envs, int64_t seq_len,
                    float gamma, float rho_bar, float c_bar, void* workspace,
                    size_t workspace_bytes, void* stream) {
  return vtrace_impl(B(log_pi_target), B(log_pi_behavior), B(values), B(rewards), B(terminateds),
                     B(truncateds), B(bootstrap), boot_mode, B(targets), B(advantages), num_envs,
                     seq_len, gamma, rho_bar, c_bar, workspace, workspace_bytes, stream);
}

}  // extern "C"
