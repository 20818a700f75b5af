/*
 * rlk_time_major.h -- calls on time-major arrays, and normalised GAE in one launch, between the
 * PyTorch extension and librl_triton_amd.so (not part of the C ABI of rl_triton_amd.h).
 *
 * A call's [num_envs, seq_len] inputs are transposed views of [seq_len, num_envs] buffers:
 * element (env, t) at env + t * step_stride of every array (Retrace's action rows at
 * (env + t * step_stride) * num_actions).  One kernel reads them in place; the outputs are
 * contiguous [num_envs, seq_len] arrays.  Results are those of the op's rl_triton_amd.h entry
 * point on contiguous copies, up to the order of float32 sums; no workspace.
 */
#ifndef RLK_TIME_MAJOR_H
#define RLK_TIME_MAJOR_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

enum rlk_op {
  RLK_OP_GAE,                /* in: rewards, values, terminateds, truncateds, mask */
  RLK_OP_GAE_NORMALIZED,     /* the same; out: advantages, returns */
  RLK_OP_VTRACE,             /* in: log_pi_target, log_pi_behavior, values, rewards,
                                terminateds, truncateds; out: targets, advantages */
  RLK_OP_RETRACE,            /* in: action_probs_target, action_probs_behavior, q_values,
                                next_q_values_all, actions, rewards, terminateds, truncateds;
                                out: targets, advantages */
  RLK_OP_LAMBDA_RETURNS,     /* in: rewards, next_values, terminateds, truncateds */
  RLK_OP_DISCOUNTED_RETURNS, /* in: rewards, terminateds, truncateds */
  RLK_OP_FORWARD             /* traces and prefix sum; in: x, dones; bootstrap: seed_values */
};

typedef struct rlk_time_major_call {
  int op;
  int bf16;             /* 0: float32 arrays, 1: bfloat16 */
  const void *in[8];    /* as listed above, NULL where absent */
  const void *bootstrap;
  int boot_mode;        /* RLK_BOOT_* (RLK_OP_FORWARD: ignored) */
  int ends_at;          /* RLK_OP_FORWARD */
  void *out[2];
  int64_t num_envs, seq_len, step_stride, num_actions;
  float gamma, lambda_; /* RLK_OP_FORWARD: gamma is the decay */
  float rho_bar, c_bar, eps;
  void *partials;       /* RLK_OP_GAE_NORMALIZED: rlk_time_major_partials_bytes bytes */
  size_t partials_bytes;
  void *sync;           /* RLK_OP_GAE_NORMALIZED in one launch, or NULL: see below */
  uint32_t epoch;
} rlk_time_major_call;

/* 1 if calls of this shape are taken (rlk_time_major returns RLK_ERR_INVALID_ARGUMENT for
 * others): rows of up to 2048 steps, and for Retrace (num_actions > 0) with more than four
 * actions up to 512 steps or at least 1024 environments.  Other calls are faster through
 * contiguous copies. */
int rlk_time_major_takes(int64_t num_envs, int64_t seq_len, int64_t step_stride, int64_t num_actions);
/* 1 if a taken call is also faster on the device than copying its `arrays` [num_envs, seq_len] arrays
 * to rows, without the host's launches: what counts while a graph is captured. */
int rlk_time_major_beats_copies(int op, int arrays, int64_t num_envs, int64_t seq_len, int64_t num_actions);
size_t rlk_time_major_partials_bytes(int64_t num_envs, int64_t seq_len);
int rlk_time_major(const rlk_time_major_call *call, void *stream);

/* Normalised GAE in one launch (step_stride ignored: contiguous rows; rlk_time_major takes the
 * same two fields).  sync: RLK_NORM_SYNC_BYTES of device memory, zero-filled once, for calls
 * ordered on one stream; epoch: 1 to RLK_NORM_MAX_EPOCH and different from every earlier call's on
 * it since it was zeroed (so not for graph capture, whose replays would repeat it).  Returns 1,
 * with nothing launched, for calls whose workgroups do not all fit the GPU at once, rows split
 * into tiles and time-major rows of more than one pass: those take two launches. */
#define RLK_NORM_SYNC_BYTES (8 * (8 + 4 * 512 + 512))
#define RLK_NORM_MAX_EPOCH 0xffff
int rlk_gae_normalized_one_launch(const rlk_time_major_call *call, void *stream);
/* 0: no call of this shape takes one launch (contiguous rows; time-major). */
int rlk_gae_normalized_one_launch_takes(int64_t num_envs, int64_t seq_len, int masked);
int rlk_time_major_one_launch_takes(int64_t num_envs, int64_t seq_len);

#ifdef __cplusplus
}
#endif

#endif /* RLK_TIME_MAJOR_H */
