// rlk_gae.hip -- GAE entry points (include/rl_triton_amd.h), with and without a mask.
#include "rlk_launch.hpp"

namespace rlk {
namespace {

// ---------------------------------------------------------------------------------------
// Entry points, one template per estimator over the storage type E (float or bf16); the
// extern "C" functions below instantiate them.
// ---------------------------------------------------------------------------------------
template <class E>
int gae_impl(const E* rewards, const E* values, const E* terminateds, const E* truncateds,
             const E* bootstrap, int boot_mode, E* advantages, int64_t num_envs, int64_t seq_len,
             float gamma, float lambda_, void* workspace, size_t workspace_bytes, void* stream) {
  if (is_empty(num_envs, seq_len)) return RLK_OK;
  if (!rewards || !values || !terminateds || !advantages || !valid_boot(bootstrap, boot_mode))
    return RLK_ERR_INVALID_ARGUMENT;
  const E* boot = boot_mode == RLK_BOOT_NONE ? nullptr : bootstrap;
  const bool vec = seq_len % 4 == 0 &&
                   quad_aligned(rewards, values, terminateds, truncateds, advantages) &&
                   (boot_mode != RLK_BOOT_FULL || quad_aligned(bootstrap));
  const int ph = common_phase<E>(rewards, values, terminateds, truncateds, advantages,
                                 boot_mode == RLK_BOOT_FULL ? bootstrap : nullptr);
  if (truncateds) {
    GaeOp<true, E> op{rewards, values, terminateds, truncateds, boot, advantages, boot_mode, gamma,
                      gamma * lambda_};
    return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream, ph);
  }
  GaeOp<false, E> op{rewards, values, terminateds, nullptr, boot, advantages, boot_mode, gamma,
                     gamma * lambda_};
  return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream, ph);
}

template <class E>
int gae_masked_impl(const E* rewards, const E* values, const E* terminateds, const E* truncateds,
                    const E* bootstrap, int boot_mode, const E* mask, E* advantages,
                    int64_t num_envs, int64_t seq_len, float gamma, float lambda_,
                    void* workspace, size_t workspace_bytes, void* stream) {
  if (is_empty(num_envs, seq_len)) return RLK_OK;
  if (!rewards || !values || !terminateds || !mask || !advantages ||
      !valid_boot(bootstrap, boot_mode))
    return RLK_ERR_INVALID_ARGUMENT;
  const E* boot = boot_mode == RLK_BOOT_NONE ? nullptr : bootstrap;
  const bool vec = seq_len % 4 == 0 &&
                   quad_aligned(rewards, values, terminateds, truncateds, mask, advantages) &&
                   (boot_mode != RLK_BOOT_FULL || quad_aligned(bootstrap));
  const int ph = common_phase<E>(rewards, values, terminateds, truncateds, mask, advantages,
                                 boot_mode == RLK_BOOT_FULL ? bootstrap : nullptr);
  if (truncateds) {
    MaskedGaeOp<true, E> op{rewards, values, terminateds, truncateds, boot, mask, advantages,
                            boot_mode, gamma, gamma * lambda_};
    return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream, ph);
  }
  MaskedGaeOp<false, E> op{rewards, values, terminateds, nullptr, boot, mask, advantages,
                           boot_mode, gamma, gamma * lambda_};
  return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream, ph);
}

}  // namespace
}  // namespace rlk

using namespace rlk;

extern "C" {

int rlk_gae(const float* rewards, const float* values, const float* terminateds,
            const float* truncateds, const float* bootstrap, int boot_mode, float* advantages,
            int64_t num_envs, int64_t seq_len, float gamma, float lambda_, void* workspace,
            size_t workspace_bytes, void* stream) {
  return gae_impl(rewards, values, terminateds, truncateds, bootstrap, boot_mode, advantages,
                  num_envs, seq_len, gamma, lambda_, workspace, workspace_bytes, stream);
}

int rlk_gae_bf16(const rlk_bf16* rewards, const rlk_bf16* values, const rlk_bf16* terminateds,
                 const rlk_bf16* truncateds, const rlk_bf16* bootstrap, int boot_mode,
                 rlk_bf16* advantages, int64_t num_envs, int64_t seq_len, float gamma,
                 float lambda_, void* workspace, size_t workspace_bytes, void* stream) {
  return gae_impl(B(rewards), B(values), B(terminateds), B(truncateds), B(bootstrap), boot_mode,
                  B(advantages), num_envs, seq_len, gamma, lambda_, workspace, workspace_bytes,
                  stream);
}

int rlk_gae_masked(const float* rewards, const float* values, const float* terminateds,
                   const float* truncateds, const float* bootstrap, int boot_mode,
                   const float* mask, float* advantages, int64_t num_envs, int64_t seq_len,
                   float gamma, float lambda_, void* workspace, size_t workspace_bytes,
                   void* stream) {
  return gae_masked_impl(rewards, values, terminateds, truncateds, bootstrap, boot_mode, mask,
                         advantages, num_envs, seq_len, gamma, lambda_, workspace,
                         workspace_bytes, stream);
}

int rlk_gae_masked_bf16(const rlk_bf16* rewards, const rlk_bf16* values,
                        const rlk_bf16* terminateds, const rlk_bf16* truncateds,
                        const rlk_bf16* bootstrap, int boot_mode, const rlk_bf16* mask,
                        rlk_bf16* advantages, int64_t num_envs, int64_t seq_len, float gamma,
                        float lambda_, void* workspace, size_t workspace_bytes, void* stream) {
  return gae_masked_impl(B(rewards), B(values), B(terminateds), B(truncateds), B(bootstrap),
                         boot_mode, B(mask), B(advantages), num_envs, seq_len, gamma, lambda_,
                         workspace, workspace_bytes, stream);
}

}  // extern "C"
