// rlk_returns.hip -- TD(lambda) and discounted returns entry points (include/rl_triton_amd.h).
#include "rlk_launch.hpp"

namespace rlk {
namespace {

template <class E>
int lambda_returns_impl(const E* rewards, const E* next_values, const E* terminateds,
                        const E* truncateds, const E* bootstrap, int boot_mode, E* returns,
                        int64_t num_envs, int64_t seq_len, float gamma, float lambda_,
                        void* workspace, size_t workspace_bytes, void* stream) {
  if (is_empty(num_envs, seq_len)) return RLK_OK;
  if (!rewards || !next_values || !terminateds || !returns || !valid_boot(bootstrap, boot_mode))
    return RLK_ERR_INVALID_ARGUMENT;
  const E* boot = boot_mode == RLK_BOOT_NONE ? nullptr : bootstrap;
  const bool vec = seq_len % 4 == 0 &&
                   quad_aligned(rewards, next_values, terminateds, truncateds, returns) &&
                   (boot_mode != RLK_BOOT_FULL || quad_aligned(bootstrap));
  const int ph = common_phase<E>(rewards, next_values, terminateds, truncateds, returns,
                                 boot_mode == RLK_BOOT_FULL ? bootstrap : nullptr);
  if (truncateds) {
    ReturnsOp<true, true, E> op{rewards, next_values, terminateds, truncateds, boot, returns,
                                boot_mode, gamma, gamma * (1.f - lambda_), gamma * lambda_};
    return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream, ph);
  }
  ReturnsOp<true, false, E> op{rewards, next_values, terminateds, nullptr, boot, returns,
                               boot_mode, gamma, gamma * (1.f - lambda_), gamma * lambda_};
  return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream, ph);
}

template <class E>
int discounted_returns_impl(const E* rewards, const E* terminateds, const E* truncateds,
                            const E* bootstrap, int boot_mode, E* returns, int64_t num_envs,
                            int64_t seq_len, float gamma, void* workspace,
                            size_t workspace_bytes, void* stream) {
  if (is_empty(num_envs, seq_len)) return RLK_OK;
  if (!rewards || !terminateds || !returns || !valid_boot(bootstrap, boot_mode))
    return RLK_ERR_INVALID_ARGUMENT;
  const E* boot = boot_mode == RLK_BOOT_NONE ? nullptr : bootstrap;
  const bool vec = seq_len % 4 == 0 && quad_aligned(rewards, terminateds, truncateds, returns) &&
                   (boot_mode != RLK_BOOT_FULL || quad_aligned(bootstrap));
  const int ph = common_phase<E>(rewards, terminateds, truncateds, returns,
                                 boot_mode == RLK_BOOT_FULL ? bootstrap : nullptr);
  if (truncateds) {
    ReturnsOp<false, true, E> op{rewards, nullptr, terminateds, truncateds, boot, returns,
                                 boot_mode, gamma, 0.f, gamma};
    return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream, ph);
  }
  ReturnsOp<false, false, E> op{rewards, nullptr, terminateds, nullptr, boot, returns, boot_mode,
                                gamma, 0.f, gamma};
  return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream, ph);
}

}  // namespace
}  // namespace rlk

using namespace rlk;

extern "C" {

int rlk_lambda_returns(const float* rewards, const float* next_values, const float* terminateds,
                       const float* truncateds, const float* bootstrap, int boot_mode,
                       float* returns, int64_t num_envs, int64_t seq_len, float gamma,
                       float lambda_, void* workspace, size_t workspace_bytes, void* stream) {
  return lambda_returns_impl(rewards, next_values, terminateds, truncateds, bootstrap, boot_mode,
                             returns, num_envs, seq_len, gamma, lambda_, workspace,
                             workspace_bytes, stream);
}

int rlk_lambda_returns_bf16(const rlk_bf16* rewards, const rlk_bf16* next_values,
                            const rlk_bf16* terminateds, const rlk_bf16* truncateds,
                            const rlk_bf16* bootstrap, int boot_mode, rlk_bf16* returns,
                            int64_t num_envs, int64_t seq_len, float gamma, float lambda_,
                            void* workspace, size_t workspace_bytes, void* stream) {
  return lambda_returns_impl(B(rewards), B(next_values), B(terminateds), B(truncateds),
                             B(bootstrap), boot_mode, B(returns), num_envs, seq_len, gamma,
                             lambda_, workspace, workspace_bytes, stream);
}

int rlk_discounted_returns(const float* rewards, const float* terminateds,
                           const float* truncateds, const float* bootstrap, int boot_mode,
                           float* returns, int64_t num_envs, int64_t seq_len, float gamma,
                           void* workspace, size_t workspace_bytes, void* stream) {
  return discounted_returns_impl(rewards, terminateds, truncateds, bootstrap, boot_mode, returns,
                                 num_envs, seq_len, gamma, workspace, workspace_bytes, stream);
}

int rlk_discounted_returns_bf16(const rlk_bf16* rewards, const rlk_bf16* terminateds,
                                const rlk_bf16* truncateds, const rlk_bf16* bootstrap,
                                int boot_mode, rlk_bf16* returns, int64_t num_envs,
                                int64_t seq_len, float gamma, void* workspace,
                                size_t workspace_bytes, void* stream) {
  return discounted_returns_impl(B(rewards), B(terminateds), B(truncateds), B(bootstrap),
                                 boot_mode, B(returns), num_envs, seq_len, gamma, workspace,
                                 workspace_bytes, stream);
}

}  // extern "C"
