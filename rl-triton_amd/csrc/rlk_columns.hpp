// rlk_columns.hpp -- scans of time-major arrays: [T, E] in memory, as rollout buffers filled one
// time step at a time are, read in place; outputs are [E, T] rows.
//
// Work decomposition.  A wave holds 16 consecutive environments (columns) of four consecutive
// 4-step chunks each, environments along the lanes: a load of one step is 16 consecutive
// elements (float32: 64 bytes) per chunk, a store of one chunk 16 bytes (bfloat16: 8) per
// environment, the wave's chunks beside each other (64 bytes of each output row).  Waves follow
// each other along time; `waves` of them (a column group) cover a pass of waves * 16 steps, and
// the passes run one after another in scan order.  Chunks are taken in scan order (reversed in
// time for backward scans), so every scan runs towards higher chunks:
//   * across a wave's chunks by lane swaps (v_permlane16_swap, v_permlane32_swap);
//   * across the group's waves, and from pass to pass, through LDS.
// The layout is one for both storage types, so that a bfloat16 result is the float32 result
// rounded; 32 bfloat16 environments (64 bytes) per wave were slower on most shapes (GAE
// [4096,128] 3.81 -> 4.28 us, [1024,256] 4.36 -> 6.31).
//
// Bound by HBM for many environments (GAE [16384,128] 10.6 us, 50 MB), by the passes' latency
// for few: 2.0-2.9 us each.  (Two register sets in turn instead of a copy, and all of a pass's
// LDS reads at once, were no faster, or spilled.)  On MI355X, us on the GPU, copying each input
// to rows first -> this:
//   GAE with truncations [4096,128] 34.6 -> 3.8, [1000,500] 32.6 -> 7.9, [16384,128] 82.7 -> 10.6
//   V-trace [4096,128] 35.1 -> 4.3;  prefix sum [4096,128] 15.6 -> 3.1, [8192,600] 69.4 -> 12.9
//   Retrace [4096,128] A = 4 71.5 -> 8.0, A = 18 164 -> 18.6
//   few environments: GAE [64,1000] 19.0 -> 10.2, [32,2048] 17.0 -> 20.2 (40.0 -> 10.5 and
//   37.2 -> 20.4 per call in a loop: the copies are launches of their own)
#pragma once
#include "rlk_ops.hpp"

namespace rlk {

constexpr int kCols = 16;  // environments side by side in a wave

// ---------------------------------------------------------------------------------------
// Moves between the lane groups of a wave (chunks), lanes of equal position in their group.
// ---------------------------------------------------------------------------------------
// Of the four rows of 16 lanes (x0 x1 x2 x3): {x0 x0 x2 x2} and {x1 x1 x3 x3}.
struct Swapped {
  uint32_t even, odd;
};
__device__ __forceinline__ Swapped swap16(uint32_t x) {
  const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  return Swapped{(uint32_t)r[0], (uint32_t)r[1]};
}
// The lower half's values in both halves.
__device__ __forceinline__ uint32_t lower_half(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_permlane32_swap(x, x, false, false)[0];
}

// The value 16 lanes below (the first chunk keeps its own).
__device__ __forceinline__ float chunk_prev(float v) {
  const uint32_t x = __float_as_uint(v);
  const Swapped s = swap16(x);
  const uint32_t second = lower_half(s.odd);  // x1 everywhere
  const int c = __lane_id() / kCols;
  return __uint_as_float(c == 0 ? x : c == 2 ? second : s.even);
}
__device__ __forceinline__ Halo2 chunk_prev(Halo2 h) { return Halo2{chunk_prev(h.a), chunk_prev(h.b)}; }
__device__ __forceinline__ NoHalo chunk_prev(NoHalo h) { return h; }
__device__ __forceinline__ NvX chunk_prev(NvX s) { return NvX{chunk_prev(s.nv), chunk_prev(s.x)}; }

// A map with every word moved by f.
template <class F>
__device__ __forceinline__ Affine move_map(Affine m, F f) { return Affine{f(m.mul), f(m.add)}; }
template <class F>
__device__ __forceinline__ SkipAffine move_map(SkipAffine m, F f) {
  return SkipAffine{f(m.a), f(m.c), f(m.p), f(m.q), f(m.d)};
}

// Inclusive scan over the wave's four chunks: the map of the first one up to this one.
template <class M>
__device__ __forceinline__ M chunk_scan(M m) {
  const int c = __lane_id() / kCols;
  const M even = move_map(m, [](float v) { return __uint_as_float(swap16(__float_as_uint(v)).even); });
  m = (c & 1) ? compose(m, even) : m;
  const M second = move_map(m, [](float v) { return __uint_as_float(lower_half(swap16(__float_as_uint(v)).odd)); });
  return c >= 2 ? compose(m, second) : m;
}

// Most waves of a column group: a workgroup of at most 1024 threads; Retrace with any action
// count holds more registers than 1024 threads have.
template <class Op>
struct column_waves : std::integral_constant<int, 16> {};
template <bool TRUNC, class E>
struct column_waves<RetraceOp<0, TRUNC, E>> : std::integral_constant<int, 8> {};

// waves: per column group; blockDim.x = kWave * waves * (groups per workgroup).
template <class Op>
__global__ __launch_bounds__(column_waves<Op>::value* kWave) void columns_kernel(const Op op, int64_t E, int T,
                                                                                 int64_t ld, int waves) {
  constexpr bool FWD = Op::kForward;
  constexpr int S = 4, COLS = kCols, CHUNKS = kWave / COLS, MAXW = column_waves<Op>::value;
  using At = ColumnAt<S>;
  using Regs = typename Op::template Regs<S>;
  using Halo = typename Op::Halo;
  using Map = typename Op::Map;
  using State = typename Map::State;
  constexpr bool HAS_HALO = !std::is_same<Halo, NoHalo>::value;
  __shared__ Map s_map[2][MAXW][COLS];

  const int lane = __lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int group = wave / waves, w = wave - group * waves;  // w: position in scan order
  const int groups = (int)(blockDim.x / kWave) / waves;
  // Workgroups go to the 8 XCDs in turn; an XCD takes consecutive column groups, so that the
  // halves of a 128-byte line are read through one L2.
  auto block_of = [](unsigned b) {
    const unsigned xcd = b & 7u, per = gridDim.x >> 3, rest = gridDim.x & 7u;
    return xcd * per + (xcd < rest ? xcd : rest) + (b >> 3);
  };
  const unsigned block = block_of(blockIdx.x);
  const int64_t col0 = ((int64_t)block * groups + group) * COLS;
  const bool active = col0 + (lane & (COLS - 1)) < E;
  const int64_t row = active ? col0 + (lane & (COLS - 1)) : E - 1;  // idle lanes read the last column
  const int64_t first_col = col0 < E ? col0 : E - 1;
  const int cols = E - first_col < COLS ? (int)(E - first_col) : COLS;
  const int c = lane / COLS;
  const int li = w * CHUNKS + c;  // chunk, in scan order
  const int pass_steps = waves * CHUNKS * S;
  const int passes = (T + pass_steps - 1) / pass_steps;
  auto seg_at = [&](int p) {
    const int base = (FWD ? p : passes - 1 - p) * pass_steps;
    return At{row, base + (FWD ? li : waves * CHUNKS - 1 - li) * S, T, ld, first_col, cols};
  };

  // Retrace with any action count waits inside its load: nothing to issue ahead
  constexpr bool AHEAD = MAXW == 16;
  Stats st;
  Regs R;
  if constexpr (AHEAD) op.load(seg_at(0), R);
  State carry = row_carry(op, seg_at(0));
  for (int p = 0; p < passes; ++p) {
    const At at = seg_at(p);
    const int t0 = at.t0;
    if constexpr (!AHEAD) op.load(at, R);
    // the first chunk of a wave that is not the row's first reads the neighbour step
    Halo edge{};
    if constexpr (HAS_HALO) {
      if (c == 0 && (p > 0 || li > 0)) edge = op.halo_load(at, clamp_step(FWD ? t0 - 1 : t0 + S, T), R);
    }
    op.template prepare<S, kElementAligned>(R, row, t0, T);
    Halo h{};
    if constexpr (HAS_HALO) {
      h = chunk_prev(scan_export<Op, S>(op, R));
      if (c == 0) h = edge;
    }
    Map steps[S];
    op.template coef<S, kElementAligned>(R, h, row, t0, T, steps);
    const Map m = chunk_scan(fold_segment<FWD, S>(steps));
    // the next pass's loads go out before this one's carry is waited for
    [[maybe_unused]] Regs next;
    const bool more = p + 1 < passes;
    if constexpr (AHEAD) {
      if (more) op.load(seg_at(p + 1), next);
    }
    State x = carry;
    if (waves > 1 || passes > 1) {
      Map(*maps)[COLS] = &s_map[p & 1][group * waves];
      if (c == CHUNKS - 1) maps[w][lane & (COLS - 1)] = m;
      __syncthreads();
      for (int v = 0; v < w; ++v) x = maps[v][lane & (COLS - 1)].apply(x);
      carry = x;
      if (more)
        for (int v = w; v < waves; ++v) carry = maps[v][lane & (COLS - 1)].apply(carry);
    }
    // state entering the chunk: the previous chunk's outgoing state, or the wave's carry
    State x_in = chunk_prev(m.apply(x));
    if (c == 0) x_in = x;
    State xs[S];
    replay<FWD, S>(steps, x_in, xs);
    if constexpr (in_one_launch<Op>::value) {  // (the launcher: one pass)
      if (active) {
        op.template emit_returns<S, kElementAligned, 0>(R, xs, row, t0, T);
        op.template stats<S>(R, xs, t0, T, st);
      }
      finish_normalized<MAXW * kWave>(
          op.one, st, op.out, (int)(blockDim.x / kWave),
          [&](auto f) {
            if (active) op.template emit_advantages<S, kElementAligned, 0>(f, xs, row, t0, T);
          },
          [&](int j, int64_t& first, int64_t& count) {
            const int64_t rows = (int64_t)groups * COLS, r0 = block_of(j) * rows;
            first = r0 * T;
            count = r0 >= E ? 0 : (E - r0 < rows ? E - r0 : rows) * T;
          });
      return;
    }
    if (active) {
      op.template emit<S, kElementAligned>(R, h, xs, x_in, row, t0, T);
      if constexpr (Op::kBlockStats) op.template stats<S>(R, xs, t0, T, st);
    }
    if constexpr (AHEAD) {
      if (more) R = next;
    }
  }
  if constexpr (Op::kBlockStats) block_stats<MAXW * kWave>(st, op.partials, (int)(blockDim.x / kWave));
}

}  // namespace rlk

