// rlk_columns.hip -- launches of the time-major kernels (include/rlk_time_major.h).
#include "rlk_columns.hpp"
#include "rlk_launch.hpp"
#include "rlk_normalize.hpp"
#include "rlk_time_major.h"

namespace rlk {
namespace {

// Waves per column group (the fewest that cover T in the fewest passes), column groups per
// workgroup (so that a workgroup has four waves at least) and workgroups.
struct ColumnShape {
  int waves, groups;
  int64_t blocks;
};
ColumnShape column_shape(int64_t num_envs, int64_t T, int max_waves) {
  constexpr int wave_steps = 4 * kWave / kCols;
  const int64_t passes = (T + max_waves * wave_steps - 1) / (max_waves * wave_steps);
  const int waves = (int)((T + passes * wave_steps - 1) / (passes * wave_steps));
  const int groups = (4 + waves - 1) / waves;
  const int64_t col_groups = (num_envs + kCols - 1) / kCols;
  return {waves, groups, (col_groups + groups - 1) / groups};
}

template <class Op>
int64_t column_blocks(int64_t num_envs, int64_t T) {
  return column_shape(num_envs, T, column_waves<Op>::value).blocks;
}

template <class Op>
int launch_columns(const Op& op, const rlk_time_major_call& c, hipStream_t stream) {
  const ColumnShape sh = column_shape(c.num_envs, c.seq_len, column_waves<Op>::value);
  const int threads = kWave * sh.waves * sh.groups;
  int64_t n = c.num_envs, ld = c.step_stride;
  int T = (int)c.seq_len, waves = sh.waves;
  void* args[] = {const_cast<Op*>(&op), &n, &T, &ld, &waves};
  return status_of(launch_kernel(reinterpret_cast<const void*>(&columns_kernel<Op>), op, sh.blocks, threads, args, stream));
}

// Rows above 2048 steps are few and are split over workgroups, which the row kernels do.  Retrace
// with any action count waits for its action rows in every pass of 128 steps (8.7 us at A = 18):
// more than four passes of few environments lose to copying the arrays to rows.  Per call, copies
// against this, us: A = 18 [64,1000] 63, 69, [64,2048] 61, 141, [256,2048] 80, 142; A = 6 [64,2048]
// 64, 93; and [1000,500] 211, 41, [1000,1000] 171, 74.  (The line is on the copies' side of the
// crossover: calls that this would serve faster lie beyond it, A = 18 [64,600] 61, 43, A = 6
// [64,1000] 61, 44.)
bool takes(int64_t num_envs, int64_t T, int64_t ld, int64_t num_actions) {
  return num_envs > 0 && T > 0 && T <= kShortMaxT && ld >= num_envs &&
         (num_envs + kCols - 1) / kCols <= kMaxLaunchBlocks && (num_actions <= 4 || T <= 512 || num_envs >= 1024);
}

// Whether the kernel takes less time on the device than a copy of each of the call's `arrays`
// [E, T] arrays and the row kernel.  A call made eagerly waits for the host's launches first, and
// one launch is faster at every shape taken (few environments, 2048 steps: prefix sum 16.7 us
// against 20.0, GAE 20 against 40, Retrace 36 against 61); in a graph the device's time is all.
// A pass over 256 steps costs about a copy of a small array, 2 us (quarters of it by op below),
// whatever the environments until they fill the GPU; copies grow with the elements.  Replayed from
// a graph on MI355X, copies against this, us: prefix sum [16,512] 7.1, 5.7, [16,1024] 7.3, 9.3,
// [64,2048] 8.1, 17.0, [512,2048] 19.2, 17.5; GAE with truncations [16,1280] 14.4, 13.7, [16,2048]
// 14.2, 19.9, [128,2048] 21.3, 20.1; V-trace [16,2048] 14.5, 23.1, [256,2048] 27.5, 23.6; Retrace
// A = 4 [16,1536] 23.6, 28.3, [64,1536] 30.5, 27.3; normalised GAE [64,2048] 13.6, 25.5.  Of 800
// calls of 2 to 2000 environments the rule is wrong by more than 10% at four (V-trace with
// truncations [64,2048] 21.1, 25.6; masked GAE [2,1024] 10.6, 12.4).
bool beats_copies(int op, int arrays, int64_t num_envs, int64_t T, int64_t num_actions) {
  if (op == RLK_OP_RETRACE && num_actions > 4) return true;  // (takes has a rule of its own)
  const int64_t passes = (T + 255) / 256;
  const int quarters = op == RLK_OP_RETRACE ? 7 : op == RLK_OP_GAE_NORMALIZED ? 6
                       : op == RLK_OP_GAE || op == RLK_OP_VTRACE ? 5 : 4;
  return quarters * passes <= 4 * (arrays + 1) + 4 * arrays * num_envs * T / 350000;
}

template <class E>
const E* in_of(const rlk_time_major_call& c, int i) { return static_cast<const E*>(c.in[i]); }
template <class E>
E* out_of(const rlk_time_major_call& c, int i) { return static_cast<E*>(c.out[i]); }

template <class StatsOp>
int launch_normalized(StatsOp op, const rlk_time_major_call& c, hipStream_t stream) {
  using E = typename StatsOp::Elem;
  if (c.sync != nullptr) {
    const ColumnShape sh = column_shape(c.num_envs, c.seq_len, column_waves<StatsOp>::value);
    if (c.seq_len > 4 * kWave / kCols * sh.waves) return kNotTaken;  // more than one pass
    return launch_columns(OneLaunchOp<StatsOp>{op, one_launch(c)}, c, stream);
  }
  const int64_t blocks = column_blocks<StatsOp>(c.num_envs, c.seq_len);
  op.partials = static_cast<double*>(c.partials);
  if (!partials_fit(c.partials, c.partials_bytes, blocks)) return RLK_ERR_WORKSPACE;
  const int st = launch_columns(op, c, stream);
  if (st != RLK_OK) return st;
  return normalize(out_of<E>(c, 0), op.partials, blocks, c.num_envs * c.seq_len, c.eps, stream);
}

template <class E, bool TRUNC>
int run(const rlk_time_major_call& c, hipStream_t s) {
  const E* boot = c.boot_mode == RLK_BOOT_NONE ? nullptr : static_cast<const E*>(c.bootstrap);
  const float gl = c.gamma * c.lambda_;
  auto in = [&](int i) { return in_of<E>(c, i); };
  E *o0 = out_of<E>(c, 0), *o1 = out_of<E>(c, 1);
  switch (c.op) {
    case RLK_OP_GAE: {
      const E *r = in(0), *v = in(1), *te = in(2), *tr = in(3), *mask = in(4);
      if (!r || !v || !te) return RLK_ERR_INVALID_ARGUMENT;
      if (mask)
        return launch_columns(MaskedGaeOp<TRUNC, E>{r, v, te, tr, boot, mask, o0, c.boot_mode, c.gamma, gl}, c, s);
      return launch_columns(GaeOp<TRUNC, E>{r, v, te, tr, boot, o0, c.boot_mode, c.gamma, gl}, c, s);
    }
    case RLK_OP_GAE_NORMALIZED: {
      const E *r = in(0), *v = in(1), *te = in(2), *tr = in(3), *mask = in(4);
      if (!r || !v || !te || !o1) return RLK_ERR_INVALID_ARGUMENT;
      if (mask)
        return launch_normalized(MaskedGaeStatsOp<TRUNC, E>{{r, v, te, tr, boot, mask, o0, c.boot_mode, c.gamma, gl},
                                                            o1, nullptr}, c, s);
      return launch_normalized(GaeStatsOp<TRUNC, E>{{r, v, te, tr, boot, o0, c.boot_mode, c.gamma, gl}, o1, nullptr}, c, s);
    }
    case RLK_OP_VTRACE: {
      if (!in(0) || !in(1) || !in(2) || !in(3) || !in(4) || !o1) return RLK_ERR_INVALID_ARGUMENT;
      return launch_columns(VtraceOp<TRUNC, E>{in(0), in(1), in(2), in(3), in(4), in(5), boot, o0, o1, c.boot_mode,
                                               c.gamma, c.rho_bar, c.c_bar}, c, s);
    }
    case RLK_OP_RETRACE: {
      const int64_t* act = static_cast<const int64_t*>(c.in[4]);
      if (!in(0) || !in(1) || !in(2) || !in(3) || !act || !in(5) || !in(6) || !o1 || c.num_actions <= 0 ||
          c.num_actions > (1 << 20))
        return RLK_ERR_INVALID_ARGUMENT;
      auto go = [&](auto na) {
        return launch_columns(RetraceOp<decltype(na)::value, TRUNC, E>{in(0), in(1), in(2), in(3), act, in(5), in(6),
                                                                       in(7), o0, o1, (int)c.num_actions, c.gamma,
                                                                       c.lambda_, c.c_bar, c.rho_bar}, c, s);
      };
      switch (c.num_actions) {
        case 1: return go(std::integral_constant<int, 1>{});
        case 2: return go(std::integral_constant<int, 2>{});
        case 3: return go(std::integral_constant<int, 3>{});
        case 4: return go(std::integral_constant<int, 4>{});
        default: return go(std::integral_constant<int, 0>{});
      }
    }
    case RLK_OP_LAMBDA_RETURNS:
      if (!in(0) || !in(1) || !in(2)) return RLK_ERR_INVALID_ARGUMENT;
      return launch_columns(ReturnsOp<true, TRUNC, E>{in(0), in(1), in(2), in(3), boot, o0, c.boot_mode, c.gamma,
                                                      c.gamma * (1.f - c.lambda_), gl}, c, s);
    case RLK_OP_DISCOUNTED_RETURNS:
      if (!in(0) || !in(1)) return RLK_ERR_INVALID_ARGUMENT;
      return launch_columns(ReturnsOp<false, TRUNC, E>{in(0), nullptr, in(1), in(2), boot, o0, c.boot_mode, c.gamma,
                                                       0.f, c.gamma}, c, s);
    case RLK_OP_FORWARD:
      if constexpr (!TRUNC) {
        if (!in(0) || !in(1)) return RLK_ERR_INVALID_ARGUMENT;
        return launch_columns(DoneGatedForwardOp<E>{in(0), in(1), static_cast<const E*>(c.bootstrap), o0, c.gamma,
                                                    c.ends_at}, c, s);
      }
  }
  return RLK_ERR_INVALID_ARGUMENT;
}

template <class E>
int run(const rlk_time_major_call& c, hipStream_t s) {
  // the truncation array's place among the inputs
  const int at = c.op == RLK_OP_GAE || c.op == RLK_OP_GAE_NORMALIZED || c.op == RLK_OP_LAMBDA_RETURNS ? 3
                 : c.op == RLK_OP_VTRACE ? 5 : c.op == RLK_OP_RETRACE ? 7 : c.op == RLK_OP_DISCOUNTED_RETURNS ? 2 : -1;
  return at >= 0 && c.in[at] != nullptr ? run<E, true>(c, s) : run<E, false>(c, s);
}

}  // namespace
}  // namespace rlk

using namespace rlk;

extern "C" {

int rlk_time_major_takes(int64_t num_envs, int64_t seq_len, int64_t step_stride, int64_t num_actions) {
  return takes(num_envs, seq_len, step_stride, num_actions) ? 1 : 0;
}

int rlk_time_major_beats_copies(int op, int arrays, int64_t num_envs, int64_t seq_len, int64_t num_actions) {
  return beats_copies(op, arrays, num_envs, seq_len, num_actions) ? 1 : 0;
}

int rlk_time_major_one_launch_takes(int64_t num_envs, int64_t seq_len) {
  if (num_envs <= 0 || seq_len <= 0 || seq_len > 4 * kWave / kCols * column_waves<GaeStatsOp<true>>::value) return 0;
  return column_blocks<GaeStatsOp<true>>(num_envs, seq_len) <= kNormPollers ? 1 : 0;
}

size_t rlk_time_major_partials_bytes(int64_t num_envs, int64_t seq_len) {
  if (num_envs <= 0 || seq_len <= 0) return 0;
  return (size_t)partials_triples(column_blocks<GaeStatsOp<true>>(num_envs, seq_len)) * kStatWords * sizeof(double);
}

int rlk_time_major(const rlk_time_major_call* call, void* stream) {
  const rlk_time_major_call& c = *call;
  if (!takes(c.num_envs, c.seq_len, c.step_stride, c.op == RLK_OP_RETRACE ? c.num_actions : 0) || !c.out[0] || !valid_boot(c.bootstrap, c.boot_mode))
    return RLK_ERR_INVALID_ARGUMENT;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  return c.bf16 ? run<bf16>(c, s) : run<float>(c, s);
}

}  // extern "C"
