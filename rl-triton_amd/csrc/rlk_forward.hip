// rlk_forward.hip -- entry points of the done-gated forward scans (eligibility traces, episodic
// prefix sum) and of the generic affine scans (include/rl_triton_amd.h).
#include "rlk_launch.hpp"

namespace rlk {
namespace {

// eligibility traces (decay = gamma * lambda, gated on done[t-1]) and the episodic prefix
// sum (decay 1, ends_at or starts_at) share one op
template <class E>
int done_gated_impl(const E* x, const E* dones, const E* seed, E* out, int64_t num_envs,
                    int64_t seq_len, float decay, int ends_at, void* workspace,
                    size_t workspace_bytes, void* stream) {
  if (is_empty(num_envs, seq_len)) return RLK_OK;
  if (!x || !dones || !out) return RLK_ERR_INVALID_ARGUMENT;
  DoneGatedForwardOp<E> op{x, dones, seed, out, decay, ends_at};
  const bool vec = seq_len % 4 == 0 && quad_aligned(x, dones, out);
  return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream,
                common_phase<E>(x, dones, out));
}

template <class E>
int affine_scan_impl(const E* u, const E* v, const E* carry, E* out, int64_t num_envs,
                     int64_t seq_len, int direction, void* workspace, size_t workspace_bytes,
                     void* stream) {
  if (is_empty(num_envs, seq_len)) return RLK_OK;
  if (!u || !v || !out || (direction != RLK_BACKWARD && direction != RLK_FORWARD))
    return RLK_ERR_INVALID_ARGUMENT;
  const bool vec = seq_len % 4 == 0 && quad_aligned(u, v, out);
  const int ph = common_phase<E>(u, v, out);
  if (direction == RLK_FORWARD) {
    AffineScanOp<true, E> op{u, v, carry, out};
    return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream, ph);
  }
  AffineScanOp<false, E> op{u, v, carry, out};
  return launch(op, num_envs, seq_len, vec, workspace, workspace_bytes, stream, ph);
}

}  // namespace
}  // namespace rlk

using namespace rlk;

extern "C" {

int rlk_eligibility_traces(const float* gradients, const float* dones, const float* seed_values,
                           float* traces, int64_t num_envs, int64_t seq_len, float gamma,
                           float lambda_, void* workspace, size_t workspace_bytes, void* stream) {
  return done_gated_impl(gradients, dones, seed_values, traces, num_envs, seq_len,
                         gamma * lambda_, 1, workspace, workspace_bytes, stream);
}

int rlk_eligibility_traces_bf16(const rlk_bf16* gradients, const rlk_bf16* dones,
                                const rlk_bf16* seed_values, rlk_bf16* traces, int64_t num_envs,
                                int64_t seq_len, float gamma, float lambda_, void* workspace,
                                size_t workspace_bytes, void* stream) {
  return done_gated_impl(B(gradients), B(dones), B(seed_values), B(traces), num_envs, seq_len,
                         gamma * lambda_, 1, workspace, workspace_bytes, stream);
}

int rlk_prefix_sum(const float* inputs, const float* dones, const float* seed_values,
                   float* prefix_sums, int64_t num_envs, int64_t seq_len, int ends_at,
                   void* workspace, size_t workspace_bytes, void* stream) {
  return done_gated_impl(inputs, dones, seed_values, prefix_sums, num_envs, seq_len, 1.f,
                         ends_at ? 1 : 0, workspace, workspace_bytes, stream);
}

int rlk_prefix_sum_bf16(const rlk_bf16* inputs, const rlk_bf16* dones,
                        const rlk_bf16* seed_values, rlk_bf16* prefix_sums, int64_t num_envs,
                        int64_t seq_len, int ends_at, void* workspace, size_t workspace_bytes,
                        void* stream) {
  return done_gated_impl(B(inputs), B(dones), B(seed_values), B(prefix_sums), num_envs, seq_len,
                         1.f, ends_at ? 1 : 0, workspace, workspace_bytes, stream);
}

int rlk_affine_scan(const float* u, const float* v, const float* carry, float* out,
                    int64_t num_envs, int64_t seq_len, int direction, void* workspace,
                    size_t workspace_bytes, void* stream) {
  return affine_scan_impl(u, v, carry, out, num_envs, seq_len, direction, workspace,
                          workspace_bytes, stream);
}

int rlk_affine_scan_bf16(const rlk_bf16* u, const rlk_bf16* v, const rlk_bf16* carry,
                         rlk_bf16* out, int64_t num_envs, int64_t seq_len, int direction,
                         void* workspace, size_t workspace_bytes, void* stream) {
  return affine_scan_impl(B(u), B(v), B(carry), B(out), num_envs, seq_len, direction, workspace,
                          workspace_bytes, stream);
}

}  // extern "C"
