// rlk_retrace.hip -- Retrace(lambda) entry points (include/rl_triton_amd.h).
#include "rlk_launch.hpp"

namespace rlk {
namespace {

template <class E>
int retrace_impl(const E* action_probs_target, const E* action_probs_behavior, const E* q_values,
                 const E* next_q_values_all, const int64_t* actions, const E* rewards,
                 const E* terminateds, const E* truncateds, E* targets, E* advantages,
                 int64_t num_envs, int64_t seq_len, int64_t num_actions, float gamma,
                 float lambda_, float c_bar, float rho_bar, void* workspace,
                 size_t workspace_bytes, void* stream) {
  if (is_empty(num_envs, seq_len)) return RLK_OK;
  if (!action_probs_target || !action_probs_behavior || !q_values || !next_q_values_all ||
      !actions || !rewards || !terminateds || !targets || !advantages || num_actions <= 0 ||
      num_actions > (1 << 20))
    return RLK_ERR_INVALID_ARGUMENT;
  const bool vec = seq_len % 4 == 0 &&
                   quad_aligned(action_probs_target, action_probs_behavior, q_values,
                                next_q_values_all, rewards, terminateds, truncateds, targets,
                                advantages) &&
                   aligned16(actions);
  const int A = (int)num_actions;
#define RLK_RETRACE(NA)                                                                          \
  {                                                                                              \
    if (truncateds) {                                                                            \
      RetraceOp<NA, true, E> op{action_probs_target, action_probs_behavior, q_values,            \
                                next_q_values_all, actions, rewards, terminateds, truncateds,    \
                                targets, advantages, A, gamma, lambda_, c_bar, rho_bar};         \
      return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream);             \
    }                                                                                            \
    RetraceOp<NA, false, E> op{action_probs_target, action_probs_behavior, q_values,             \
                               next_q_values_all, actions, rewards, terminateds, nullptr,        \
                               targets, advantages, A, gamma, lambda_, c_bar, rho_bar};          \
    return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream);               \
  }
  switch (A) {
    case 1: RLK_RETRACE(1)
    case 2: RLK_RETRACE(2)
    case 3: RLK_RETRACE(3)
    case 4: RLK_RETRACE(4)
    default: RLK_RETRACE(0)
  }
#undef RLK_RETRACE
}

}  // namespace
}  // namespace rlk

using namespace rlk;

extern "C" {

int rlk_retrace(const float* action_probs_target, const float* action_probs_behavior,
                const float* q_values, const float* next_q_values_all, const int64_t* actions,
                const float* rewards, const float* terminateds, const float* truncateds,
                float* targets, float* advantages, int64_t num_envs, int64_t seq_len,
                int64_t num_actions, float gamma, float lambda_, float c_bar, float rho_bar,
                void* workspace, size_t workspace_bytes, void* stream) {
  return retrace_impl(action_probs_target, action_probs_behavior, q_values, next_q_values_all,
                      actions, rewards, terminateds, truncateds, targets, advantages, num_envs,
                      seq_len, num_actions, gamma, lambda_, c_bar, rho_bar, workspace,
                      workspace_bytes, stream);
}

int rlk_retrace_bf16(const rlk_bf16* action_probs_target, const rlk_bf16* action_probs_behavior,
                     const rlk_bf16* q_values, const rlk_bf16* next_q_values_all,
                     const int64_t* actions, const rlk_bf16* rewards,
                     const rlk_bf16* terminateds, const rlk_bf16* truncateds, rlk_bf16* targets,
                     rlk_bf16* advantages, int64_t num_envs, int64_t seq_len,
                     int64_t num_actions, float gamma, float lambda_, float c_bar, float rho_bar,
                     void* workspace, size_t workspace_bytes, void* stream) {
  return retrace_impl(B(action_probs_target), B(action_probs_behavior), B(q_values),
                      B(next_q_values_all), actions, B(rewards), B(terminateds), B(truncateds),
                      B(targets), B(advantages), num_envs, seq_len, num_actions, gamma, lambda_,
                      c_bar, rho_bar, workspace, workspace_bytes, stream);
}

}  // extern "C"
