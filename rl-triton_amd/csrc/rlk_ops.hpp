// rlk_ops.hpp -- the rl_triton estimators as producers/epilogues of the scan engine.
//
// Each struct turns its inputs into per-step affine coefficients (truncation and
// bootstrap handling folded in, so there is no extra pass) and turns the scanned
// values into the estimator's outputs.  Semantics follow the reference's fused Triton
// kernels (simonsays1980/rl-triton v0.1.3, src/rl_triton/kernels/*.py); each struct
// cites the lines it reproduces.  Padding steps (t >= T) are the identity map.
//
// Optional operands that change which arrays are read (truncations, TD(lambda)'s next
// values) are template parameters; loads are clamped into the row and absent per-row
// values are read from g_zero.
#pragma once
#include "rlk_engine.hpp"

namespace rlk {

template <int S>
__device__ __forceinline__ void fill_regs(float (&v)[S], float x) {
#pragma unroll
  for (int i = 0; i < S; ++i) v[i] = x;
}

// ------------------------------------------------------------------------------------------
// GAE: kernels/gae.py:121-180 (gae_fused_kernel), both HAS_TRUNCATIONS branches.
//   v_next = boot(t)  if t == T-1 or trunc[t] == 1,  values[t+1] otherwise
//   add = r + gamma*v_next*(1-term) - v,   mul = gamma*lambda*(1 - done)
//   done = min(term + trunc, 1) with truncations, term without;   x[T] = 0
// ------------------------------------------------------------------------------------------
template <bool TRUNC, class E = float>
struct GaeOp {
  using Elem = E;  // storage type of the float arrays
  static constexpr bool kForward = false;
  static constexpr bool kBlockStats = false;  // no per-workgroup output statistics
  // long-row tiles: threads per workgroup and most 4-step segments per thread that stay
  // in registers (no spills at 1024 threads, whose cap is 128 VGPRs)
  static constexpr int kLongThreads = 1024, kLongMaxSegments = 4;
  using Halo = float;  // values[t+1]
  using Map = Affine;  // one carried value
  const E* r;
  const E* v;
  const E* term;
  const E* trunc;  // read iff TRUNC
  const E* boot;   // nullable, per boot_mode
  E* out;
  int boot_mode;
  float gamma, gl;  // gl = gamma*lambda


  template <int S>
  struct Regs {
    float r[S], v[S], te[S], tr[S], bt[S];
    float blast;
  };

  template <class At>
  __device__ void load(const At& at, Regs<At::S>& R) const {
    at.seg(r, R.r);
    at.seg(v, R.v);
    at.seg(term, R.te);
    if constexpr (TRUNC) at.seg(trunc, R.tr);
    else fill_regs(R.tr, 0.f);
    boot_load<TRUNC>(at, boot, boot_mode, R.bt, R.blast, r);
  }
  template <int S, int VEC>
  __device__ void prepare(Regs<S>& R, int64_t, int t0, int T) const {
    boot_prepare<S, TRUNC>(boot_mode, t0, T, R.bt, R.blast);
  }
  template <int S>
  __device__ float export_first(const Regs<S>& R) const { return R.v[0]; }
  template <class At>
  __device__ float halo_load(const At& at, int t, const Regs<At::S>&) const { return to_f32(v[at.index(t)]); }

  template <int S, int VEC = kElementAligned>
  __device__ void coef(const Regs<S>& R, float vh, int64_t, int t0, int T, Affine (&m)[S]) const {
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int t = t0 + i;
      const float raw = (i + 1 < S) ? R.v[i + 1] : vh;
      // kAligned: T % 4 == 0 and t0 % 4 == 0, so a segment is all in or all padding, and
      // only its last step can be T - 1 (one comparison per segment instead of one per step)
      const bool at_end = VEC == kAligned ? (i == S - 1 && t0 + S == T) : (t == T - 1);
      // `|`, not `||`: the short circuit compiled to a divergent branch on the path after
      // the loads (C2 [4096,128] 3.82 -> 3.80 us, bfloat16 3.28 -> 3.18 us on MI355X)
      const bool use_boot = at_end | (R.tr[i] == 1.f);
      const float vn = use_boot ? R.bt[i] : raw;
      const float done = TRUNC ? fminf(R.te[i] + R.tr[i], 1.f) : R.te[i];
      const float a = fmaf(gamma * vn, 1.f - R.te[i], R.r[i]) - R.v[i];
      const bool in = step_in<VEC>(t0, t, T);  // padding steps are the identity map
      m[i].add = in ? a : 0.f;
      m[i].mul = in ? gl * (1.f - done) : 1.f;
    }
  }
  template <class At>
  __device__ const E* row_carry_src(const At&) const { return nullptr; }

  template <int S, int VEC, int SP = 0>
  __device__ void emit(const Regs<S>&, float, const float (&xs)[S], float, int64_t row, int t0,
                       int T) const {
    store_seg<S, VEC>(out + row * (int64_t)T, t0, T, xs, SP != 0);
  }
};

// ------------------------------------------------------------------------------------------
// GAE with returns and batch statistics: the first half of compute_gae_normalized (no
// counterpart in the reference, which has none of this; it is the "fused GAE + advantage
// normalisation" item of its ROADMAP.md:75-81).  The scan is GaeOp's; the epilogue writes
// the raw advantages A and the returns A + values, and each workgroup reduces the count,
// sum and sum of squares of its A in float64 into partials[3*blockIdx.x .. +2] (see
// block_stats in rlk_engine.hpp).  normalize_kernel then turns A into
// (A - mean) / (std + eps) in place.
// ------------------------------------------------------------------------------------------
template <bool TRUNC, class E = float>
struct GaeStatsOp : GaeOp<TRUNC, E> {
  static constexpr bool kBlockStats = true;
  E* returns;
  double* partials;
  template <int S>
  using Regs = typename GaeOp<TRUNC, E>::template Regs<S>;

  // the two outputs by themselves, advantages mapped by f (OneLaunchOp)
  template <int S, int VEC, int SP>
  __device__ void emit_returns(const Regs<S>& R, const float (&xs)[S], int64_t row, int t0, int T) const {
    float rt[S];
#pragma unroll
    for (int i = 0; i < S; ++i) rt[i] = xs[i] + R.v[i];
    store_seg<S, VEC>(returns + row * (int64_t)T, t0, T, rt, SP != 0);
  }
  template <int S, int VEC, int SP, class F>
  __device__ void emit_advantages(F f, const float (&xs)[S], int64_t row, int t0, int T) const {
    float a[S];
#pragma unroll
    for (int i = 0; i < S; ++i) a[i] = f(xs[i]);
    store_seg<S, VEC>(this->out + row * (int64_t)T, t0, T, a, SP != 0);
  }

  template <int S, int VEC, int SP = 0>
  __device__ void emit(const Regs<S>& R, float, const float (&xs)[S], float, int64_t row, int t0,
                       int T) const {
    static_assert(VEC != kPhased, "stats() does not see the steps ahead of a phased row's tiles");
    float rt[S];
#pragma unroll
    for (int i = 0; i < S; ++i) rt[i] = xs[i] + R.v[i];
    const int64_t o = row * (int64_t)T;
    store_seg<S, VEC>(this->out + o, t0, T, xs, SP != 0);
    store_seg<S, VEC>(returns + o, t0, T, rt, SP != 0);
  }
  // every step of the row counts
  template <int S>
  __device__ void stats(const Regs<S>&, const float (&xs)[S], int t0, int T, Stats& st) const {
#pragma unroll
    for (int i = 0; i < S; ++i)
      if (t0 + i < T) st.add(xs[i]);
  }
};

// ------------------------------------------------------------------------------------------
// GAE with skipped steps: the "verl-style" masking of the reference's ROADMAP.md:131-140
// (not implemented in the reference).  Steps with mask == 0 leave the advantage and the
// next value unchanged, so credit and the continuation value pass across them (multi-turn
// rollouts whose observation tokens are not actions).  With nv = the value of the nearest
// kept step after t (boot(T-1) if there is none):
//   kept t:     v_next = boot(t) if trunc[t] == 1, nv otherwise
//               A[t] = r + gamma*v_next*(1-term) - v + gamma*lambda*(1-done)*A(after t)
//               nv <- v[t]
//   skipped t:  A[t] = A(after t) (0 if no kept step follows), nv unchanged
// With every step kept this is GaeOp.  The state {nv, A} is carried by SkipAffine maps:
// a kept step is (a, c, p, q, d) = (0, v, gamma*(1-term) [0 if truncated], gamma*lambda*
// (1-done), r - v [+ gamma*boot*(1-term) if truncated]); a skipped step is the identity.
// No halo: the next value arrives through the scan itself.
// ------------------------------------------------------------------------------------------
template <bool TRUNC, class E = float>
struct MaskedGaeOp {
  using Elem = E;  // storage type of the float arrays
  static constexpr bool kForward = false;
  static constexpr bool kBlockStats = false;
  static constexpr int kLongThreads = 512, kLongMaxSegments = 4;  // five-word maps
  using Halo = NoHalo;
  using Map = SkipAffine;  // state {next value, advantage}
  const E* r;
  const E* v;
  const E* term;
  const E* trunc;  // read iff TRUNC
  const E* boot;   // nullable, per boot_mode
  const E* mask;
  E* out;
  int boot_mode;
  float gamma, gl;  // gl = gamma*lambda


  template <int S>
  struct Regs {
    float r[S], v[S], te[S], tr[S], bt[S], mk[S];
    float blast;
  };

  template <class At>
  __device__ void load(const At& at, Regs<At::S>& R) const {
    at.seg(r, R.r);
    at.seg(v, R.v);
    at.seg(term, R.te);
    at.seg(mask, R.mk);
    if constexpr (TRUNC) {
      at.seg(trunc, R.tr);
      boot_load<true>(at, boot, boot_mode, R.bt, R.blast, r);
    } else {
      fill_regs(R.tr, 0.f), fill_regs(R.bt, 0.f);
      R.blast = 0.f;
    }
  }
  template <int S, int VEC>
  __device__ void prepare(Regs<S>& R, int64_t, int t0, int T) const {
    if constexpr (TRUNC) boot_prepare<S, true>(boot_mode, t0, T, R.bt, R.blast);
  }
  // state after the row: next value boot(T-1), advantage 0
  template <class At>
  __device__ NvX row_state(const At& at) const {
    return NvX{to_f32(*boot_last(at, boot, boot_mode)), 0.f};
  }

  template <int S, int VEC = kElementAligned>
  __device__ void coef(const Regs<S>& R, NoHalo, int64_t, int t0, int T, SkipAffine (&m)[S]) const {
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const bool sel = TRUNC && R.tr[i] == 1.f;
      const float done = TRUNC ? fminf(R.te[i] + R.tr[i], 1.f) : R.te[i];
      const float g1 = gamma * (1.f - R.te[i]);
      const float d = sel ? fmaf(gamma * R.bt[i], 1.f - R.te[i], R.r[i]) - R.v[i] : R.r[i] - R.v[i];
      const bool kept = (step_in<VEC>(t0, t0 + i, T)) && R.mk[i] != 0.f;  // padding steps too
      m[i] = kept ? SkipAffine{0.f, R.v[i], sel ? 0.f : g1, gl * (1.f - done), d}
                  : SkipAffine::identity();
    }
  }

  template <int S, int VEC, int SP = 0>
  __device__ void emit(const Regs<S>&, NoHalo, const NvX (&xs)[S], NvX, int64_t row, int t0,
                       int T) const {
    float a[S];
#pragma unroll
    for (int i = 0; i < S; ++i) a[i] = xs[i].x;
    store_seg<S, VEC>(out + row * (int64_t)T, t0, T, a, SP != 0);
  }
};

// ------------------------------------------------------------------------------------------
// Masked GAE with returns and statistics over the kept steps: the first half of
// compute_gae_normalized(..., mask=...), the masked whitening verl applies after its
// compute_gae_advantage_return.  Returns are A + values at every step; count, sum and sum of
// squares are of the kept steps only, and normalize_kernel rewrites every step's A.
// ------------------------------------------------------------------------------------------
template <bool TRUNC, class E = float>
struct MaskedGaeStatsOp : MaskedGaeOp<TRUNC, E> {
  static constexpr bool kBlockStats = true;
  E* returns;
  double* partials;
  template <int S>
  using Regs = typename MaskedGaeOp<TRUNC, E>::template Regs<S>;

  template <int S, int VEC, int SP>
  __device__ void emit_returns(const Regs<S>& R, const NvX (&xs)[S], int64_t row, int t0, int T) const {
    float rt[S];
#pragma unroll
    for (int i = 0; i < S; ++i) rt[i] = xs[i].x + R.v[i];
    store_seg<S, VEC>(returns + row * (int64_t)T, t0, T, rt, SP != 0);
  }
  template <int S, int VEC, int SP, class F>
  __device__ void emit_advantages(F f, const NvX (&xs)[S], int64_t row, int t0, int T) const {
    float a[S];
#pragma unroll
    for (int i = 0; i < S; ++i) a[i] = f(xs[i].x);
    store_seg<S, VEC>(this->out + row * (int64_t)T, t0, T, a, SP != 0);
  }

  template <int S, int VEC, int SP = 0>
  __device__ void emit(const Regs<S>& R, NoHalo, const NvX (&xs)[S], NvX, int64_t row, int t0,
                       int T) const {
    static_assert(VEC != kPhased, "stats() does not see the steps ahead of a phased row's tiles");
    float a[S], rt[S];
#pragma unroll
    for (int i = 0; i < S; ++i) {
      a[i] = xs[i].x;
      rt[i] = xs[i].x + R.v[i];
    }
    const int64_t o = row * (int64_t)T;
    store_seg<S, VEC>(this->out + o, t0, T, a, SP != 0);
    store_seg<S, VEC>(returns + o, t0, T, rt, SP != 0);
  }
  template <int S>
  __device__ void stats(const Regs<S>& R, const NvX (&xs)[S], int t0, int T, Stats& st) const {
#pragma unroll
    for (int i = 0; i < S; ++i)
      if (t0 + i < T && R.mk[i] != 0.f) st.add(xs[i].x);
  }
};

// ------------------------------------------------------------------------------------------
// V-trace: kernels/vtrace_fused.py:90-196 (vtrace_fused_kernel).
//   rho = min(exp(lpt - lpb), rho_bar),  c = min(exp(lpt - lpb), c_bar)
//   truncations:  v_next = values[t+1]*[t < T-1 and trunc == 0] + boot(t)   (additive)
//   otherwise:    v_next = boot(T-1) at t = T-1, values[t+1] elsewhere
//   add = rho*(r + gamma*v_next*(1-term) - v),  mul = gamma*c*(1-done),  x[T] = 0
//   targets = x + v;  next target by the same rule as v_next with targets for values
//   advantages = rho*(r + gamma*next_target*(1-term) - v)
// The reference passes targets[t+1] through global memory (store, barrier, reload,
// vtrace_fused.py:149-152); here it is the neighbouring register or lane.
// ------------------------------------------------------------------------------------------
template <bool TRUNC, class E = float>
struct VtraceOp {
  using Elem = E;  // storage type of the float arrays
  static constexpr bool kForward = false;
  static constexpr bool kBlockStats = false;  // no per-workgroup output statistics
  static constexpr int kLongThreads = 1024, kLongMaxSegments = 2;
  using Halo = float;  // values[t+1]
  using Map = Affine;  // one carried value
  const E* lpt;
  const E* lpb;
  const E* v;
  const E* r;
  const E* term;
  const E* trunc;  // read iff TRUNC
  const E* boot;   // nullable, per boot_mode
  E* targets;
  E* adv;
  int boot_mode;
  float gamma, rho_bar, c_bar;


  template <int S>
  struct Regs {
    float rho[S], c[S], v[S], r[S], te[S], tr[S], bt[S];  // rho, c: log-probs until prepare()
    float blast;
  };

  template <class At>
  __device__ void load(const At& at, Regs<At::S>& R) const {
    at.seg(lpt, R.rho);
    at.seg(lpb, R.c);
    at.seg(v, R.v);
    at.seg(r, R.r);
    at.seg(term, R.te);
    if constexpr (TRUNC) at.seg(trunc, R.tr);
    else fill_regs(R.tr, 0.f);
    boot_load<TRUNC>(at, boot, boot_mode, R.bt, R.blast, r);
  }
  template <int S, int VEC>
  __device__ void prepare(Regs<S>& R, int64_t, int t0, int T) const {
#pragma unroll
    for (int i = 0; i < S; ++i) {
      // hardware exp2 after a multiply by log2(e): a few ulp, far inside the parity
      // tolerance, and 2% off the [4096,128] call against the range-reduced expf
      const float ratio = __expf(R.rho[i] - R.c[i]);
      R.rho[i] = fminf(ratio, rho_bar);
      R.c[i] = fminf(ratio, c_bar);
    }
    boot_prepare<S, TRUNC>(boot_mode, t0, T, R.bt, R.blast);
  }
  template <int S>
  __device__ float export_first(const Regs<S>& R) const { return R.v[0]; }
  template <class At>
  __device__ float halo_load(const At& at, int t, const Regs<At::S>&) const { return to_f32(v[at.index(t)]); }

  // continuation value at step t from the raw next-step value (values or targets)
  // last: t == T - 1
  __device__ __forceinline__ float next_value(float raw, float tr, float bt, bool last) const {
    if constexpr (TRUNC) return ((!last && tr == 0.f) ? raw : 0.f) + bt;
    return last ? bt : raw;
  }

  template <int S, int VEC = kElementAligned>
  __device__ void coef(const Regs<S>& R, float vh, int64_t, int t0, int T, Affine (&m)[S]) const {
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int t = t0 + i;
      const bool last = VEC == kAligned ? (i == S - 1 && t0 + S == T) : (t == T - 1);
      const float vn = next_value((i + 1 < S) ? R.v[i + 1] : vh, R.tr[i], R.bt[i], last);
      const float done = TRUNC ? fminf(R.te[i] + R.tr[i], 1.f) : R.te[i];
      const float a = R.rho[i] * (fmaf(gamma * vn, 1.f - R.te[i], R.r[i]) - R.v[i]);
      const bool in = step_in<VEC>(t0, t, T);
      m[i].add = in ? a : 0.f;
      m[i].mul = in ? gamma * R.c[i] * (1.f - done) : 1.f;
    }
  }
  template <class At>
  __device__ const E* row_carry_src(const At&) const { return nullptr; }

  template <int S, int VEC, int SP = 0>
  __device__ void emit(const Regs<S>& R, float vh, const float (&xs)[S], float x_next, int64_t row,
                       int t0, int T) const {
    float tg[S], ad[S];
#pragma unroll
    for (int i = 0; i < S; ++i) tg[i] = xs[i] + R.v[i];
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const float raw = (i + 1 < S) ? tg[i + 1] : x_next + vh;
      const bool last = VEC == kAligned ? (i == S - 1 && t0 + S == T) : (t0 + i == T - 1);
      const float nt = next_value(raw, R.tr[i], R.bt[i], last);
      ad[i] = R.rho[i] * (fmaf(gamma * nt, 1.f - R.te[i], R.r[i]) - R.v[i]);
    }
    const int64_t o = row * (int64_t)T;
    store_seg<S, VEC>(targets + o, t0, T, tg, SP != 0);
    store_seg<S, VEC>(adv + o, t0, T, ad, SP != 0);
  }
};

// ------------------------------------------------------------------------------------------
// Action rows of any length A, reduced by a wave through LDS.
//
// A wave's segments are a contiguous run of steps, so their action rows are a contiguous run
// of words in pi and in nq.  Each lane reading its own steps' rows touches 64 cache lines per
// load, each line again by later loads, and the lines do not stay in L1 (A = 18: two arrays of
// 18 KB per wave): Retrace then ran at a quarter of the streaming rate.  Here the wave takes
// the run 64 rows at a time: word j*64 + lane of them goes to lane `lane` (each load 256
// contiguous bytes; bfloat16: pairs), from there to LDS at a row stride of A | 1 words (odd: the 64
// rows start in different banks), and lane l sums row l in order of the actions, the order
// (and the bits) of a loop over the row.  The next 64 rows' loads are issued before the sums.
// Short rows go 128 or 256 at a time (bfloat16 A = 6 [1024,250] 6.7 us at 64 rows), rows of
// more than kPipedActions actions in slices of 16 actions.  (The cap is where the largest
// straight-line batch that was built ends; 19 actions would fit the same LDS.  Slices cost a step
// there, and another from 33 actions on, us: [1024,256] A = 17 8.9, 18 10.2, 19 14.4, 24 15.4,
// 32 15.9, 33 20.0, 64 28.3; [4096,128] A = 17 15.0, 18 15.6, 19 19.4, 24 21.9.)
//
// Bound by HBM: on MI355X, float32, lane-by-lane rows -> this: A = 18 [4096,128] 78.3 -> 15.8
// us (94 MB, 6.0 TB/s), [256,2048] 138.6 -> 16.8, [64,8192] 115.5 -> 23.8; A = 6 [4096,128]
// 23.9 -> 8.6; bfloat16 A = 18 [4096,128] 108.1 -> 11.5.  A branch around each load or LDS
// read instead of the straight-line batches took 28.4 us at A = 18 [4096,128].  Lane-by-lane
// rows were faster for bfloat16 A = 5 between 131072 and 262144 steps only ([1024,256] 5.2 us,
// 5.4 so; [2000,100] 4.8, 5.5).
//
// LDS is the wave's own, dynamic (action_stage_bytes per wave): no barrier.
// ------------------------------------------------------------------------------------------
constexpr int kPipedActions = 18, kActionSlice = 16;
// Four bytes from an element's address on: one float, or a pair of bfloat16.
typedef uint32_t ua_u1 __attribute__((aligned(2)));
__device__ __forceinline__ uint32_t load_word_ua(const float* p) { return __float_as_uint(*p); }
__device__ __forceinline__ uint32_t load_word_ua(const bf16* p) { return *reinterpret_cast<const ua_u1*>(p); }
__host__ __device__ inline int action_stage_stride(int A) { return A <= kPipedActions ? (A | 1) : (kActionSlice | 1); }
// Two staged arrays of 64 rows (rows of up to 9 actions: 128, up to 5: 256), the last row read
// up to its batch's loads; later two result arrays of up to 256 steps.  At most 9728 bytes (17 and
// 18 actions): sixteen waves per CU.
__host__ __device__ inline int action_stage_bytes(int A) {
  const int rows = kWave * (A <= 5 ? 4 : A <= 9 ? 2 : 1);
  const int batch = A <= 5 ? 5 : A <= 6 ? 6 : A <= 9 ? 9 : A <= 12 ? 12 : kPipedActions;
  const int over = A < batch ? batch - A : 0;
  const int b = (2 * rows * action_stage_stride(A) + over) * (int)sizeof(float);
  return ((b < 2048 ? 2048 : b) + 15) & ~15;
}

// LDS accesses of one wave stay in program order across lanes.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The run of steps that the wave's lanes hold, as step indexes of the [E, T] arrays.  Lanes
// hold a row's segments in reverse (backward scans): the run starts at the last lane of the
// first row and ends with the first lane of the last one.  (Lanes of rows past E repeat row
// E - 1, whole.)
template <class At>
__device__ __forceinline__ void wave_run(const At& at, int64_t& first, int& steps) {
  constexpr int S = At::S;
  const int row_lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)at.row);
  const int row_hi = __builtin_amdgcn_readlane((int)(uint32_t)at.row, kWave - 1);
  const int in_lo = __popcll(__ballot((int)(uint32_t)at.row == row_lo));
  const int in_hi = __popcll(__ballot((int)(uint32_t)at.row == row_hi));
  const int t_lo = __builtin_amdgcn_readlane(at.t0, in_lo - 1);
  const int t_hi = __builtin_amdgcn_readlane(at.t0, kWave - in_hi) + S;
  const int64_t base = (int64_t)lane0_u64((uint64_t)at.index(0));
  first = base + t_lo;
  steps = (int)(uint32_t)(row_hi - row_lo) * at.T + (t_hi < at.T ? t_hi : at.T) - t_lo;
  if (steps < 0) steps = 0;
}

template <class At, class E>
__device__ __forceinline__ void reduce_actions(const At& at, const E* __restrict__ pi,
                                               const E* __restrict__ nq,
                                               const int64_t* __restrict__ act, int A,
                                               float (&enq)[At::S], float (&pa)[At::S],
                                               float& pa_next) {
  // Rows: the wave's run of steps, M * 64 of them per round.  Columns: step r of every chunk in
  // round r, each chunk's COLS rows a contiguous piece; lane l's own step is row l.
  constexpr int PIECE_ROWS = columns_of<At>::value;
  constexpr bool COLUMNS = PIECE_ROWS < kWave;
  constexpr int S = At::S, ROUNDS = S;
  extern __shared__ float s_actions[];
  const int lane = __lane_id();
  const int stride = action_stage_stride(A);
  float* sp = s_actions + (threadIdx.x / kWave) * (action_stage_bytes(A) / (int)sizeof(float));
  int64_t first = 0;
  int steps = kWave * S;
  if constexpr (!COLUMNS) wave_run(at, first, steps);
  // rows of round r's pieces of at most `most` rows, and the first one's step index
  auto rows_of = [&](int r, int most) {
    if constexpr (COLUMNS) return most < at.cols ? most : at.cols;
    else return steps - r * most < most ? steps - r * most : most;
  };
  auto piece_of = [&](int r, int most, int piece) -> int64_t {
    if constexpr (COLUMNS) {
      const int t = __builtin_amdgcn_readlane(at.t0, piece * most) + r;
      return at.first_col + (t < at.T ? t : at.T - 1) * at.ld;
    } else {
      return first + r * most;
    }
  };
  // The step after the wave's (the row's next; step T - 1 again where there is none): its action
  // is read ahead of the rows, its probability beside them, once the action is there.
  int64_t next;
  {
    const int t = at.t0 + S < at.T ? at.t0 + S : at.T - 1;
    if constexpr (COLUMNS) next = at.index(t);
    else next = (int64_t)lane0_u64((uint64_t)at.index(t));
  }
  const int64_t a_next = act[next];
  const E* p_next = pi + next * A + (a_next >= 0 && a_next < A ? a_next : 0);
  E raw_next{};
  float e[ROUNDS], p_taken[ROUNDS];
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) e[r] = p_taken[r] = 0.f;
  auto keep = [&](int r, float s, float pt) {
#pragma unroll
    for (int k = 0; k < ROUNDS; ++k) {
      e[k] = k == r ? s : e[k];
      p_taken[k] = k == r ? pt : p_taken[k];
    }
  };
  int Av = A;  // in a vector register: selects on it stay selects, not branches around reads
  asm("" : "+v"(Av));
  if (A <= kPipedActions) {
    // B >= A loads per array and lane, straight-line code (a branch per load made the compiler
    // wait at each): words past the run repeat its last one, sums past A are dropped.
    auto rounds = [&](auto b, auto m) {
      constexpr int B = decltype(b)::value;
      constexpr int M = S == 1 || COLUMNS ? 1 : decltype(m)::value, ROWS = M * kWave;  // per round
      constexpr int PR = COLUMNS ? PIECE_ROWS : ROWS, PIECES = ROWS / PR;  // rows per piece
      constexpr int PK = 4 / (int)sizeof(E);  // elements per 4-byte load
      constexpr int NL = (PR * B + PK * kWave - 1) / (PK * kWave);  // loads per lane and piece
      float* sn = sp + ROWS * stride;
      uint32_t vp[PIECES][NL], vn[PIECES][NL];
      int64_t a_t[M];
      // floor(w / A) for w < 2^11: (w * ceil(2^20 / A)) >> 20
      const uint32_t magic = (A & 1) ? 0u : ((1u << 20) + (uint32_t)A - 1) / (uint32_t)A;
      auto issue = [&](int r) {
        const int rows = rows_of(r, PR), last = rows * A - PK;
#pragma unroll
        for (int k = 0; k < M; ++k) {
          if constexpr (COLUMNS) {
            a_t[k] = act[at.index(at.t0 + r < at.T ? at.t0 + r : at.T - 1)];
          } else {
            const int i = k * kWave + lane;
            a_t[k] = act[first + r * ROWS + (i < rows ? i : rows - 1)];
          }
        }
#pragma unroll
        for (int c = 0; c < PIECES; ++c) {
          const int64_t base = piece_of(r, PR, c) * A;
#pragma unroll
          for (int j = 0; j < NL; ++j) {
            const int w = PK * (j * kWave + lane);
            vp[c][j] = load_word_ua(pi + base + (w < last ? w : last));
            vn[c][j] = load_word_ua(nq + base + (w < last ? w : last));
          }
        }
      };
      issue(0);
#pragma unroll 1
      for (int r = 0; r * ROWS < steps; ++r) {
        int64_t at_r[M];
#pragma unroll
        for (int k = 0; k < M; ++k) at_r[k] = a_t[k];
        const uint32_t end = rows_of(r, PR) * A;
#pragma unroll
        for (int c = 0; c < PIECES; ++c) {
#pragma unroll
          for (int j = 0; j < NL; ++j) {
            const uint32_t w = PK * (j * kWave + lane);
            // (whole waves of words: a scalar branch)
            if (PK == 1 && PR % kWave == 0 ? j * kWave < PR * A : w < (uint32_t)(PR * A)) {
              const uint32_t pos = c * PR * stride + w + ((w * magic) >> 20);
              if constexpr (PK == 1) {
                sp[pos] = __uint_as_float(vp[c][j]);
                sn[pos] = __uint_as_float(vn[c][j]);
              } else {
                // a pair lies in one row, or (odd A) rows follow each other without a gap.  The
                // run's last word alone was read with the one before it.
                const bool alone = w + 1 == end;
                const uint32_t up = alone ? vp[c][j] >> 16 : vp[c][j], un = alone ? vn[c][j] >> 16 : vn[c][j];
                sp[pos] = __uint_as_float(up << 16);
                sn[pos] = __uint_as_float(un << 16);
                if (w + 1 < (uint32_t)(PR * A)) {
                  sp[pos + 1] = __uint_as_float(up & 0xffff0000u);
                  sn[pos + 1] = __uint_as_float(un & 0xffff0000u);
                }
              }
            }
          }
        }
        wave_lds_fence();
        raw_next = *p_next;
        if ((r + 1) * ROWS < steps) issue(r + 1);
#pragma unroll
        for (int k = 0; k < M; ++k) {
          const int row = (k * kWave + lane) * stride;
          float s = 0.f;
#pragma unroll
          for (int a = 0; a < B; ++a) {
            const float t = fmaf(sp[row + a], sn[row + a], s);
            s = a < Av ? t : s;
          }
          keep(r * M + k, s, at_r[k] >= 0 && at_r[k] < A ? sp[row + (int)at_r[k]] : 0.f);
        }
        wave_lds_fence();
      }
    };
    if (steps > 0) {
      using std::integral_constant;
      if (A <= 5) rounds(integral_constant<int, 5>{}, integral_constant<int, 4>{});
      else if (A == 6) rounds(integral_constant<int, 6>{}, integral_constant<int, 2>{});
      else if (A <= 9) rounds(integral_constant<int, 9>{}, integral_constant<int, 2>{});
      else if (A <= 12) rounds(integral_constant<int, 12>{}, integral_constant<int, 1>{});
      else rounds(integral_constant<int, kPipedActions>{}, integral_constant<int, 1>{});
    }
  } else {
    constexpr int PR = PIECE_ROWS;
#pragma unroll 1
    for (int r = 0; r * kWave < steps; ++r) {
      const int rows = rows_of(r, PR);
      int64_t a_t;
      if constexpr (COLUMNS) a_t = act[at.index(at.t0 + r < at.T ? at.t0 + r : at.T - 1)];
      else a_t = act[first + r * kWave + (lane < rows ? lane : rows - 1)];
      raw_next = *p_next;
      float* sn = sp + kWave * stride;
      const int s_in = lane / kActionSlice, a_in = lane & (kActionSlice - 1);
      float s = 0.f, pt = 0.f;
#pragma unroll 1
      for (int a0 = 0; a0 < A; a0 += kActionSlice) {
        E vp[kActionSlice], vn[kActionSlice];
        const int a = a0 + a_in < A ? a0 + a_in : A - 1;
#pragma unroll
        for (int j = 0; j < kActionSlice; ++j) {
          const int sj = j * (kWave / kActionSlice) + s_in;  // row of the round
          // (a load's four rows lie in one piece)
          const int k = sj - (j * (kWave / kActionSlice)) / PR * PR;
          const int64_t w = (piece_of(r, PR, (j * (kWave / kActionSlice)) / PR) + (k < rows ? k : rows - 1)) * A + a;
          vp[j] = pi[w];
          vn[j] = nq[w];
        }
#pragma unroll
        for (int j = 0; j < kActionSlice; ++j) {
          const int sj = j * (kWave / kActionSlice) + s_in;
          sp[sj * stride + a_in] = to_f32(vp[j]);
          sn[sj * stride + a_in] = to_f32(vn[j]);
        }
        wave_lds_fence();
#pragma unroll
        for (int k = 0; k < kActionSlice; ++k) {
          const float t = fmaf(sp[lane * stride + k], sn[lane * stride + k], s);
          s = a0 + k < Av ? t : s;
        }
        const int64_t k_t = a_t - a0;
        if (k_t >= 0 && k_t < kActionSlice && a_t < A) pt = sp[lane * stride + (int)k_t];
        wave_lds_fence();
      }
      keep(r, s, pt);
    }
  }
  pa_next = a_next >= 0 && a_next < A ? to_f32(raw_next) : 0.f;
  if constexpr (COLUMNS) {
#pragma unroll
    for (int i = 0; i < S; ++i) enq[i] = e[i], pa[i] = p_taken[i];
    return;
  }
  // from "lane l has steps l, 64 + l, ..." of the run to each lane's own segment
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    sp[r * kWave + lane] = e[r];
    sp[(ROUNDS + r) * kWave + lane] = p_taken[r];
  }
  wave_lds_fence();
  const int local = (int)(at.index(at.t0) - first);
#pragma unroll
  for (int i = 0; i < S; ++i) {
    const int k = local + i < ROUNDS * kWave ? local + i : ROUNDS * kWave - 1;  // padding: any
    enq[i] = sp[k < 0 ? 0 : k];
    pa[i] = sp[ROUNDS * kWave + (k < 0 ? 0 : k)];
  }
  wave_lds_fence();
}

// ------------------------------------------------------------------------------------------
// Retrace(lambda): kernels/retrace_fused.py:116-201 (retrace_fused_kernel).
//   E_pi[Q'] = sum_a pi[t,a]*nq[t,a];  pi_a = pi[t, a_t] (0 if a_t outside [0, A))
//   rho = min(pi_a/mu, rho_bar),  c = lambda*min(pi_a/mu, c_bar)
//   add = r + gamma*E_pi[Q']*(1-term) - q,  mul = gamma*c[t+1]*(1-done),  c[T] = 0
//   Q_ret = x + q;  advantages = rho*(r + gamma*Q_ret[t+1]*(1-term) - q),  Q_ret[T] = 0
// NA > 0: compile-time action count (vector loads of the [S, A] block); NA == 0: any A
// (reduce_actions).
// ------------------------------------------------------------------------------------------
template <int NA, bool TRUNC, class E = float>
struct RetraceOp {
  using Elem = E;  // storage type of the float arrays
  static constexpr bool kForward = false;
  static constexpr bool kBlockStats = false;  // no per-workgroup output statistics
  static constexpr int kLongThreads = 512, kLongMaxSegments = 2;  // 256 VGPRs: the A-wide rows
  using Halo = Halo2;  // {c[t+1], q[t+1]}
  using Map = Affine;  // one carried value
  const E* pi;     // [E, T, A]
  const E* mu;     // [E, T]
  const E* q;
  const E* nq;     // [E, T, A]
  const int64_t* act;  // [E, T]
  const E* r;
  const E* term;
  const E* trunc;  // read iff TRUNC
  E* targets;
  E* adv;
  int A;
  float gamma, lambda, c_bar, rho_bar;


  template <int S>
  struct Regs {
    float q[S], r[S], te[S], tr[S], rho[S], c[S], enq[S];
    float pa_next;  // NA == 0: pi of the action taken at the step after the wave's (halo_load)
  };

  // rho and c at one step from the probability of its action under both policies
  __device__ __forceinline__ void clipped_ratios(float pa, float m, float& rho, float& c) const {
    const float ratio = pa / m;
    rho = fminf(ratio, rho_bar);
    c = lambda * fminf(ratio, c_bar);
  }

  // (rho, c, E_pi[Q']) at one step from its action row (NA > 0)
  template <class P>
  __device__ __forceinline__ void step_terms(const P* p, const P* n, int64_t a_t, float m,
                                             float& rho, float& c, float& enq) const {
    float e = 0.f, pa = 0.f;
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      const float pv = to_f32(p[a]);
      e = fmaf(pv, to_f32(n[a]), e);
      pa = (a == a_t) ? pv : pa;
    }
    clipped_ratios(pa, m, rho, c);
    enq = e;
  }

  // Unlike the other ops, the [S, A] action blocks are reduced to (rho, c, E_pi[Q']) here,
  // at load time, so a segment holds three values per step instead of 2A.
  template <class At>
  __device__ void load(const At& at, Regs<At::S>& R) const {
    constexpr int S = At::S, VEC = At::kVec;
    static_assert(VEC != kPhased, "the [E, T, A] arrays have no common row phase");
    const int t0 = at.t0, T = at.T;
    float m[S];
    at.seg(q, R.q);
    at.seg(r, R.r);
    at.seg(term, R.te);
    if constexpr (TRUNC) at.seg(trunc, R.tr);
    else fill_regs(R.tr, 0.f);
    at.seg(mu, m);
    if constexpr (NA == 0) {
      float pa[S];
      reduce_actions(at, pi, nq, act, A, R.enq, pa, R.pa_next);
#pragma unroll
      for (int i = 0; i < S; ++i) clipped_ratios(pa[i], m[i], R.rho[i], R.c[i]);
    } else {
      int64_t a_t[S];
      if constexpr (VEC == kAligned) {
        // a quad of actions is 32 contiguous bytes, 16-byte aligned (the launch checks the
        // pointer): two 16-byte loads instead of four 8-byte ones (Retrace [4096,128]
        // 6.60 -> 6.53 us on MI355X); a quad beyond T reads the row's last quad
        typedef long long i64x2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int qd = 0; qd < S / 4; ++qd) {
          const int t = t0 + 4 * qd;
          const i64x2* pq = reinterpret_cast<const i64x2*>(act + at.index(t < T ? t : T - 4));
          const i64x2 u = pq[0], w = pq[1];
          a_t[4 * qd] = u.x, a_t[4 * qd + 1] = u.y, a_t[4 * qd + 2] = w.x, a_t[4 * qd + 3] = w.y;
        }
      } else {
#pragma unroll
        for (int i = 0; i < S; ++i) a_t[i] = act[at.index(clamp_step(t0 + i, T))];
      }
      if constexpr (VEC == kAligned && (S * NA) % 4 == 0 && S * NA <= 16) {
        // the [S, NA] blocks are contiguous and 16-byte aligned; a quad beyond T reads the
        // row's first quad instead.
        float pb[S * NA], nb[S * NA];
        const E* pp = pi + at.index(t0) * NA;
        const E* np = nq + at.index(t0) * NA;
#pragma unroll
        for (int qd = 0; qd < S * NA / 4; ++qd) {
          const bool in = t0 + (4 * qd) / NA < T;
          const float4 a4 = load_quad(in ? pp + 4 * qd : pi + at.index(0) * NA);
          const float4 b4 = load_quad(in ? np + 4 * qd : nq + at.index(0) * NA);
          pb[4 * qd] = a4.x, pb[4 * qd + 1] = a4.y, pb[4 * qd + 2] = a4.z, pb[4 * qd + 3] = a4.w;
          nb[4 * qd] = b4.x, nb[4 * qd + 1] = b4.y, nb[4 * qd + 2] = b4.z, nb[4 * qd + 3] = b4.w;
        }
#pragma unroll
        for (int i = 0; i < S; ++i) step_terms(pb + i * NA, nb + i * NA, a_t[i], m[i], R.rho[i], R.c[i], R.enq[i]);
      } else {
#pragma unroll
        for (int i = 0; i < S; ++i) {
          const int64_t base = at.index(clamp_step(t0 + i, T)) * NA;
          step_terms(pi + base, nq + base, a_t[i], m[i], R.rho[i], R.c[i], R.enq[i]);
        }
      }
    }
  }
  template <int S, int VEC>
  __device__ void prepare(Regs<S>&, int64_t, int, int) const {}
  template <int S>
  __device__ Halo2 export_first(const Regs<S>& R) const { return Halo2{R.c[0], R.q[0]}; }
  template <class At>
  __device__ Halo2 halo_load(const At& at, int t, const Regs<At::S>& R) const {
    const int64_t i = at.index(t);
    float rho, c, enq;
    if constexpr (NA == 0) clipped_ratios(R.pa_next, to_f32(mu[i]), rho, c);
    else step_terms(pi + i * NA, nq + i * NA, act[i], to_f32(mu[i]), rho, c, enq);
    return Halo2{c, to_f32(q[i])};
  }

  template <int S, int VEC = kElementAligned>
  __device__ void coef(const Regs<S>& R, Halo2 h, int64_t, int t0, int T, Affine (&m)[S]) const {
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int t = t0 + i;
      const bool before_end = VEC == kAligned ? (i < S - 1 ? t0 < T : t0 + S < T) : (t < T - 1);
      const float c_next = before_end ? ((i + 1 < S) ? R.c[i + 1] : h.a) : 0.f;
      const float done = fminf(R.te[i] + R.tr[i], 1.f);
      const float a = fmaf(gamma * R.enq[i], 1.f - R.te[i], R.r[i]) - R.q[i];
      const bool in = step_in<VEC>(t0, t, T);  // vector segments are all-in or all-out
      m[i].add = in ? a : 0.f;
      m[i].mul = in ? gamma * c_next * (1.f - done) : 1.f;
    }
  }
  template <class At>
  __device__ const E* row_carry_src(const At&) const { return nullptr; }

  template <int S, int VEC, int SP = 0>
  __device__ void emit(const Regs<S>& R, Halo2 h, const float (&xs)[S], float x_next, int64_t row,
                       int t0, int T) const {
    float tg[S], ad[S];
#pragma unroll
    for (int i = 0; i < S; ++i) tg[i] = xs[i] + R.q[i];
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int t = t0 + i;
      const bool before_end = VEC == kAligned ? (i < S - 1 ? t0 < T : t0 + S < T) : (t < T - 1);
      const float nxt = before_end ? ((i + 1 < S) ? tg[i + 1] : x_next + h.b) : 0.f;
      ad[i] = R.rho[i] * (fmaf(gamma * nxt, 1.f - R.te[i], R.r[i]) - R.q[i]);
    }
    const int64_t o = row * (int64_t)T;
    store_seg<S, VEC>(targets + o, t0, T, tg, SP != 0);
    store_seg<S, VEC>(adv + o, t0, T, ad, SP != 0);
  }
};

// ------------------------------------------------------------------------------------------
// TD(lambda) returns: kernels/lambda_returns_fused.py:54-89.
//   nd = 1 - done;  add = r + gamma*(1-lambda)*nd*nv + gamma*trunc*boot(t);  mul = gamma*lambda*nd
//   x[T] = boot(T-1)
// Discounted returns: kernels/discounted_returns_fused.py:50-82 -- the same with
//   add = r + gamma*trunc*boot(t),  mul = gamma*nd  (NV = false: no next values).
// ------------------------------------------------------------------------------------------
template <bool NV, bool TRUNC, class E = float>
struct ReturnsOp {
  using Elem = E;  // storage type of the float arrays
  static constexpr bool kForward = false;
  static constexpr bool kBlockStats = false;  // no per-workgroup output statistics
  // plain discounted returns (two arrays read): 512-thread tiles of up to 8 segments per
  // thread measured 3% faster at [16,131072] than 1024 threads of 2 (same tile size)
  static constexpr int kLongThreads = (NV || TRUNC) ? 1024 : 512;
  static constexpr int kLongMaxSegments = (NV || TRUNC) ? 4 : 8;
  using Halo = NoHalo;
  using Map = Affine;  // one carried value
  const E* r;
  const E* nv;     // read iff NV
  const E* term;
  const E* trunc;  // read iff TRUNC
  const E* boot;   // nullable, per boot_mode
  E* out;
  int boot_mode;
  float gamma, g1l, gl;  // gamma, gamma*(1-lambda), gamma*lambda (discounted: gl = gamma)


  template <int S>
  struct Regs {
    float r[S], nv[S], te[S], tr[S], bt[S];
    float blast;
  };

  template <class At>
  __device__ void load(const At& at, Regs<At::S>& R) const {
    at.seg(r, R.r);
    if constexpr (NV) at.seg(nv, R.nv);
    else fill_regs(R.nv, 0.f);
    at.seg(term, R.te);
    if constexpr (TRUNC) {
      at.seg(trunc, R.tr);
      boot_load<true>(at, boot, boot_mode, R.bt, R.blast, r);
    } else {
      fill_regs(R.tr, 0.f), fill_regs(R.bt, 0.f);
      R.blast = 0.f;
    }
  }
  template <int S, int VEC>
  __device__ void prepare(Regs<S>& R, int64_t, int t0, int T) const {
    if constexpr (TRUNC) boot_prepare<S, true>(boot_mode, t0, T, R.bt, R.blast);
  }

  template <int S, int VEC = kElementAligned>
  __device__ void coef(const Regs<S>& R, NoHalo, int64_t, int t0, int T, Affine (&m)[S]) const {
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int t = t0 + i;
      const float nd = 1.f - (TRUNC ? fminf(R.te[i] + R.tr[i], 1.f) : R.te[i]);
      float a = NV ? fmaf(g1l * nd, R.nv[i], R.r[i]) : R.r[i];
      if constexpr (TRUNC) a = fmaf(gamma * R.tr[i], R.bt[i], a);
      const bool in = step_in<VEC>(t0, t, T);  // vector segments are all-in or all-out
      m[i].add = in ? a : 0.f;
      m[i].mul = in ? gl * nd : 1.f;
    }
  }
  template <class At>
  __device__ const E* row_carry_src(const At& at) const {
    return boot_mode == kBootNone ? nullptr : boot_last(at, boot, boot_mode);
  }

  template <int S, int VEC, int SP = 0>
  __device__ void emit(const Regs<S>&, NoHalo, const float (&xs)[S], float, int64_t row, int t0,
                       int T) const {
    store_seg<S, VEC>(out + row * (int64_t)T, t0, T, xs, SP != 0);
  }
};

// ------------------------------------------------------------------------------------------
// Forward scans gated on done.
//   eligibility traces (kernels/eligibility_traces_fused.py:67-84):
//       mul = gamma*lambda*(1 - done[t-1]), done[-1] = 0, add = g, x[-1] = seed
//   episodic prefix sum (kernels/prefix_sum_fused.py:63-84):
//       ends_at:   mul = 1 - done[t-1];  starts_at: mul = 1 - done[t];  add = x, x[-1] = seed
// (decay = gamma*lambda for traces, 1 for the prefix sum)
// ------------------------------------------------------------------------------------------
template <class E = float>
struct DoneGatedForwardOp {
  using Elem = E;  // storage type of the float arrays
  static constexpr bool kForward = true;
  static constexpr bool kBlockStats = false;
  static constexpr int kLongThreads = 1024, kLongMaxSegments = 8;
  using Halo = float;  // done[t-1]
  using Map = Affine;  // one carried value
  const E* x;
  const E* dones;
  const E* seed;  // nullable
  E* out;
  float decay;
  int ends_at;


  template <int S>
  struct Regs {
    float x[S], d[S];
  };

  template <class At>
  __device__ void load(const At& at, Regs<At::S>& R) const {
    at.seg(x, R.x);
    at.seg(dones, R.d);
  }
  template <int S, int VEC>
  __device__ void prepare(Regs<S>&, int64_t, int, int) const {}
  template <int S>
  __device__ float export_last(const Regs<S>& R) const { return R.d[S - 1]; }
  template <class At>
  __device__ float halo_load(const At& at, int t, const Regs<At::S>&) const { return to_f32(dones[at.index(t)]); }

  template <int S, int VEC = kElementAligned>
  __device__ void coef(const Regs<S>& R, float dh, int64_t, int t0, int T, Affine (&m)[S]) const {
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int t = t0 + i;
      float gate;
      if (ends_at) {
        // kPhased segments can hold step 0 past their first position, after steps of the
        // row before (done[-1] = 0 all the same)
        if constexpr (VEC == kPhased) gate = t == 0 ? 0.f : (i > 0 ? R.d[i - 1] : dh);
        else gate = (i > 0) ? R.d[i - 1] : (t == 0 ? 0.f : dh);
      } else {
        gate = R.d[i];
      }
      const bool in = step_in<VEC>(t0, t, T);  // vector segments are all-in or all-out
      m[i].mul = in ? decay * (1.f - gate) : 1.f;
      m[i].add = in ? R.x[i] : 0.f;
    }
  }
  template <class At>
  __device__ const E* row_carry_src(const At& at) const { return seed ? seed + at.row : nullptr; }

  template <int S, int VEC, int SP = 0>
  __device__ void emit(const Regs<S>&, float, const float (&xs)[S], float, int64_t row, int t0,
                       int T) const {
    store_seg<S, VEC>(out + row * (int64_t)T, t0, T, xs, SP != 0);
  }
};

// ------------------------------------------------------------------------------------------
// Generic affine scans (ops/_scan.py:69-213, kernels/scan.py:39-138):
//   backward A[t] = u[t] + v[t]*A[t+1], A[T] = carry;  forward e[t] = u[t] + v[t]*e[t-1], e[-1] = carry
// ------------------------------------------------------------------------------------------
template <bool FWD, class E = float>
struct AffineScanOp {
  using Elem = E;  // storage type of the float arrays
  static constexpr bool kForward = FWD;
  static constexpr bool kBlockStats = false;
  static constexpr int kLongThreads = 1024, kLongMaxSegments = 8;
  using Halo = NoHalo;
  using Map = Affine;  // one carried value
  const E* u;
  const E* v;
  const E* carry;  // nullable, [E]
  E* out;


  template <int S>
  struct Regs {
    float u[S], v[S];
  };
  template <class At>
  __device__ void load(const At& at, Regs<At::S>& R) const {
    at.seg(u, R.u);
    at.seg(v, R.v);
  }
  template <int S, int VEC>
  __device__ void prepare(Regs<S>&, int64_t, int, int) const {}
  template <int S, int VEC = kElementAligned>
  __device__ void coef(const Regs<S>& R, NoHalo, int64_t, int t0, int T, Affine (&m)[S]) const {
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const bool in = step_in<VEC>(t0, t0 + i, T);
      m[i].mul = in ? R.v[i] : 1.f;
      m[i].add = in ? R.u[i] : 0.f;
    }
  }
  template <class At>
  __device__ const E* row_carry_src(const At& at) const { return carry ? carry + at.row : nullptr; }
  template <int S, int VEC, int SP = 0>
  __device__ void emit(const Regs<S>&, NoHalo, const float (&xs)[S], float, int64_t row, int t0,
                       int T) const {
    store_seg<S, VEC>(out + row * (int64_t)T, t0, T, xs, SP != 0);
  }
};

}  // namespace rlk
