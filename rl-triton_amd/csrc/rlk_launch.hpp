// rlk_launch.hpp -- launch planning for librl_triton_amd.so: which kernel, workgroup, tile and
// store policy a call of an op runs with, and the launches themselves.  Each estimator's entry
// points (rlk_*.hip) instantiate launch() for their ops.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <map>
#include <mutex>
#include <utility>

#include "rl_triton_amd.h"
#include "rlk_ops.hpp"

namespace rlk {

// Launch geometry.
constexpr int kNT = 256;          // short rows: threads per workgroup of small calls (4 wavefronts)
constexpr int kNTWide = 512;      // short rows otherwise (8 wavefronts; one row of 1025..2048
                                  // steps where rows_strided_kernel is not used)
constexpr int kShortMaxT = 2048;  // rows up to this length are kept whole in one workgroup
constexpr int kStridedThreads = 256, kStridedSegments = 2;  // rows_strided_kernel's tile
static_assert(kNTWide >= kShortMaxT / 4, "a short row (up to 512 threads of 4 steps) fits one workgroup");
// Long rows: each op fixes its threads per workgroup (kLongThreads) and the most 4-step
// segments per thread its registers hold without spilling (kLongMaxSegments, 2..8).  The
// smallest tile any op uses sizes the workspace.
constexpr int kMinQ = 2;
constexpr int64_t kMinTile = (int64_t)512 * kSeg * kMinQ;  // 4096 steps

inline int ceil_log2(int64_t x) {
  int k = 0;
  while ((int64_t{1} << k) < x) ++k;
  return k;
}

// Compute units of the current device (cached per device; 256 on MI355X).  Threads that
// race on the first call store the same value.
inline int query_cus() {
  static std::atomic<int> cached[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}
// The rules below ask for it many times per call, and each question of the current device costs
// the host 30-50 ns: a CusScope answers those within it by one, on its thread (host time of a call,
// us: normalised GAE [8,16313] 9.7 -> 7.8, [1,8193] 10.2 -> 7.9, GAE [1,8193] 4.7 -> 3.8).
inline thread_local int t_scope_cus = 0;
class CusScope {
 public:
  CusScope() : outermost_(t_scope_cus == 0) {
    if (outermost_) t_scope_cus = query_cus();
  }
  ~CusScope() {
    if (outermost_) t_scope_cus = 0;
  }
  CusScope(const CusScope&) = delete;
  CusScope& operator=(const CusScope&) = delete;

 private:
  const bool outermost_;
};
inline int device_cus() { return t_scope_cus > 0 ? t_scope_cus : query_cus(); }

// Long rows: segments per thread.  Tiles are as large as the op's registers allow while
// the call still has one tile per compute unit: a longer tile shortens the look-back
// chain along a row, and a tile per CU keeps every CU streaming.
template <class Op>
int long_segments(int64_t E, int64_t T) {
  const int64_t cus = device_cus();
  for (int q = Op::kLongMaxSegments; q > kMinQ; q /= 2) {
    const int64_t tile = (int64_t)Op::kLongThreads * kSeg * q;
    if (E * ((T + tile - 1) / tile) >= cus) return q;
  }
  return kMinQ;
}

// Workspace for a long-row call: two places of status words for its tiles (the tile's own,
// and the one other workgroups publish into), counted at the smallest tile.
inline int64_t status_tiles(int64_t E, int64_t T) { return E * ((T + kMinTile - 1) / kMinTile); }
inline size_t workspace_bytes(int64_t E, int64_t T) {
  if (E <= 0 || T <= kShortMaxT) return 0;
  return (size_t)(kStatusOffset + 2 * kStatusWords * status_tiles(E, T)) * sizeof(uint64_t);
}

inline bool aligned16(const void* p) { return p == nullptr || (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Short rows: S steps per thread, L = 2^ceil(log2(ceil(T/S))) threads per row, NT/L rows
// per workgroup, grid = ceil(E / (NT/L)).
inline int64_t rows_grid(int64_t E, int64_t T, int S, int NT) {
  const int64_t rows_per_block = NT >> ceil_log2((T + S - 1) / S);
  return (E + rows_per_block - 1) / rows_per_block;
}

// Threads per workgroup of a short-row launch: 512 for rows over 1024 steps (one row per
// workgroup), and for shorter rows whenever 512-thread workgroups still give every compute
// unit one (GAE [4096,128] measured 4.26 -> 4.08 us, TD(lambda) 3.41 -> 3.26 us); 256 for
// smaller calls, which need the finer grid to reach the CUs.
inline int rows_threads(int64_t E, int64_t T) {
  if (T > 1024) return kNTWide;
  return rows_grid(E, T, 4, kNTWide) >= device_cus() ? kNTWide : kNT;
}

inline int64_t chain_grid(int64_t E, int64_t T, int NT, int Q) {
  const int64_t tile = (int64_t)NT * kSeg * Q;
  const int64_t nslots = lookback_slots(E);
  return nslots * (((E + nslots - 1) / nslots) * ((T + tile - 1) / tile));
}

// Short rows: steps per segment.  Four (one quad per array per thread) from four steps
// up; rows of 1-3 steps take one step per thread, element by element.
inline int rows_seg(int64_t T) { return T < 4 ? 1 : 4; }

// Long-row tile shapes (threads x 4-step segments per thread).  Each op has its own thread
// count and largest segment count (kLongThreads, kLongMaxSegments), and long_segments picks
// the largest tile that still gives every CU one.  Three kinds of call change the shape,
// where measured faster on MI355X (A/B twice, same box, both storage types alike so that a
// bfloat16 result stays the float32 result rounded):
//   * discounted returns without truncations (512-thread tiles of up to 8 segments), a call
//     that gives every CU a 16384-step tile: 1024 x 4 instead of 512 x 8, the same tiles
//     ([64,65536] 11.2 -> 10.3 us, [8,2^20] 23.1 -> 22.0 us; C5 [16,131072] keeps 512 x 4,
//     8.12 us, against 8.41 at 1024 x 2);
//   * discounted returns on rows of at least eight 8192-step tiles, whose 8192-step tiles
//     reach half the CUs but not all of them: 1024 x 2 (those tiles) instead of 512 x 2
//     (4096-step tiles, enough for every CU): [2,10^6] 10.3 -> 8.9 us, [3,500000]
//     8.20 -> 7.62 us, [8,200000] 9.15 -> 8.12 us; bfloat16 [3,500000] 7.60 -> 7.00 us.
//     Shorter rows lose to the last tile's padding ([100,10000] 6.19 -> 6.44 us);
//   * 1024-thread ops whose 8192-step tiles (1024 x 2) outnumber the CUs but not twice
//     over: a CU holds one 1024-thread workgroup of these kernels, so the tiles would run in
//     two rounds; 512 x 4 (the same tiles) fits two workgroups per CU.  TD(lambda)
//     [64,40000] 13.17 -> 11.89 us, [96,30000] 13.62 -> 11.92 us (bfloat16 11.53 -> 8.87),
//     [200,10000] 12.12 -> 10.37 us; GAE [64,40000] 17.46 -> 16.16 us, [200,10000]
//     16.16 -> 14.41 us; prefix sum [64,40000] 11.18 -> 8.93 us.  V-trace's registers allow
//     one 512 x 4 workgroup per CU, so it takes 512 x 2 (4096-step tiles, two workgroups
//     per CU): [64,40000] 18.6 -> 16.4 us, [200,10000] 17.2 -> 15.4 us, bfloat16
//     [96,30000] 15.7 -> 15.0 us, float32 [96,30000] 19.4 -> 19.7 us.  (Ops whose tile can
//     double take twice the tile first in these calls, one round of 16384-step tiles,
//     faster still (cu_shape); only V-trace still takes this rule.)
struct LongShape {
  int threads, segments;
};
template <class Op>
struct wide_long_tiles : std::false_type {};
template <class E>
struct wide_long_tiles<ReturnsOp<false, false, E>> : std::true_type {};
// segments per thread of the 512-thread tiles a 1024 x 2 call between one and two tiles
// per CU takes instead (0: keeps 1024 x 2)
template <class Op>
struct half_width_segments : std::integral_constant<int, 0> {};
template <bool TRUNC, class E>
struct half_width_segments<GaeOp<TRUNC, E>> : std::integral_constant<int, 4> {};
template <bool TRUNC, class E>
struct half_width_segments<GaeStatsOp<TRUNC, E>> : std::integral_constant<int, 4> {};
template <bool NV, bool TRUNC, class E>
struct half_width_segments<ReturnsOp<NV, TRUNC, E>> : std::integral_constant<int, (NV || TRUNC) ? 4 : 0> {};
template <class E>
struct half_width_segments<DoneGatedForwardOp<E>> : std::integral_constant<int, 4> {};
template <bool FWD, class E>
struct half_width_segments<AffineScanOp<FWD, E>> : std::integral_constant<int, 4> {};
template <bool TRUNC, class E>
struct half_width_segments<VtraceOp<TRUNC, E>> : std::integral_constant<int, 2> {};

template <class Op>
LongShape cu_shape(int64_t E, int64_t T) {
  const int64_t cus = device_cus();
  auto tiles = [&](int64_t tile) { return E * ((T + tile - 1) / tile); };
  if constexpr (wide_long_tiles<Op>::value) {
    if (tiles(1024 * kSeg * 4) >= cus) return {1024, 4};
    const int64_t t8 = tiles(1024 * kSeg * 2);
    if (T >= 8 * 8192 && t8 < cus && 2 * t8 >= cus) return {1024, 2};
  }
  int q = long_segments<Op>(E, T);
  // More tiles than CUs at that size, fewer at twice the size: the larger tiles, in one
  // round with some CUs idle, beat the smaller ones in two.  Measured on MI355X (the
  // larger tiles' share of the CUs 0.53-0.88, A/B in one process): GAE [150,10000]
  // 13.7 -> 10.3 us, [64,40000] 16.1 -> 14.2, TD(lambda) [160,10000] 10.1 -> 7.6, prefix
  // sum [48,131072] 18.6 -> 14.9, [40,100000] 14.6 -> 12.5.  Calls whose tiles already fit
  // one round keep them ([128,12000], [16,131072]: twice the tile lost 6-25%).
  if (q < Op::kLongMaxSegments) {
    const int64_t tile = (int64_t)Op::kLongThreads * kSeg * q;
    if (tiles(tile) > cus && tiles(2 * tile) < cus) q *= 2;
  }
  // (Below, q == 2 with more 8192-step tiles than CUs is left only to ops whose largest
  // tile that is: V-trace.)
  constexpr int hq = half_width_segments<Op>::value;
  if constexpr (hq != 0) {
    static_assert(Op::kLongThreads == 1024, "a 1024 x 2 call becomes 512 x hq");
    const int64_t t8 = tiles(1024 * kSeg * 2);
    if (q == 2 && t8 > cus && t8 <= 2 * cus) return {512, hq};
  }
  return {Op::kLongThreads, q};
}

inline int64_t tile_steps(LongShape s) { return (int64_t)s.threads * kSeg * s.segments; }

// The long-row tile shape of a call: cu_shape's, then two corrections.
//   * Calls that leave CUs idle even at the op's own smallest tile take 4096-step tiles
//     while those fit one round (below).
//   * Rows much shorter than the tiles.  cu_shape sizes a tile for the CUs and the
//     look-back chain along a row, so a call of many rows of a few thousand steps ran one
//     tile per row that was mostly padding: a 2560-step row in a 32768-step tile, the
//     prefix sum [4096,2560] at 114 us against 22 us for a streaming kernel of its bytes.
//     (Such rows are now held whole, see whole_row_segments; this serves longer ones and
//     Retrace's.)
//     Where more than a quarter of a row's tile steps would be padding, the call takes the
//     largest of the op's tiles that pads a row by at most a quarter, or else the one that
//     pads it least (the larger on a tie), unless its tiles fit the CUs in one round and
//     the smaller ones would not.
// Tiles of one size run at the op's own thread count, 4096-step tiles at 512 threads; an
// 8192-step tile of a 1024-thread op between one and two tiles per CU takes 512 threads,
// as in cu_shape.
template <class Op>
LongShape long_shape(int64_t E, int64_t T) {
  LongShape sh = cu_shape<Op>(E, T);
  {
    // Fewer tiles than CUs even at the op's own smallest tile (8192 steps for the
    // 1024-thread ops): 4096-step tiles, while those still fit the CUs in one round.  GAE
    // [16,40000] 8.07 -> 6.94 us, V-trace [24,20000] 8.11 -> 6.83, TD(lambda) [16,65536]
    // 6.90 -> 6.52, prefix sum [40,16384] 5.77 -> 5.22; calls that fill the CUs unchanged.
    const int64_t cus = device_cus(), tile = tile_steps(sh);
    const int64_t now = E * ((T + tile - 1) / tile), small = E * ((T + kMinTile - 1) / kMinTile);
    if (tile > kMinTile && now < cus && small > now && small <= cus) sh = {512, kMinQ};
  }
  auto padded = [&](int64_t tile) { return (T + tile - 1) / tile * tile; };
  auto fits = [&](int64_t tile) { return 4 * padded(tile) <= 5 * T; };  // padding <= T / 4
  if (fits(tile_steps(sh))) return sh;
  // the op's tiles, largest first: kLongThreads x q for q = kLongMaxSegments .. kMinQ, then
  // the 4096-step tile of 512 x kMinQ
  int64_t tiles[8];
  int n = 0;
  for (int q = Op::kLongMaxSegments; q >= kMinQ; q /= 2) tiles[n++] = (int64_t)Op::kLongThreads * kSeg * q;
  if (tiles[n - 1] > kMinTile) tiles[n++] = kMinTile;
  int64_t best = tiles[0];
  for (int i = 0; i < n; ++i) {
    if (fits(tiles[i])) {
      best = tiles[i];
      break;
    }
    if (padded(tiles[i]) < padded(best)) best = tiles[i];
  }
  // a call whose tiles fit the CUs in one round keeps them rather than take smaller tiles
  // in more than one
  const int64_t cus = device_cus(), t = E * ((T + best - 1) / best);
  const int64_t t_sh = E * ((T + tile_steps(sh) - 1) / tile_steps(sh));
  if (t_sh <= cus && t > cus) return sh;
  if (best == kMinTile) return {512, kMinQ};
  const LongShape r{Op::kLongThreads, (int)(best / ((int64_t)Op::kLongThreads * kSeg))};
  constexpr int hq = half_width_segments<Op>::value;
  if constexpr (hq != 0) {
    if (r.segments == 2 && t > cus && t <= 2 * cus) return {512, hq};
  }
  return r;
}

// Ops whose time is their action rows, not the [E, T] arrays (Retrace with any action count:
// at 18 actions the rows are 84% of the call's bytes): one form of each launch only,
// element-aligned with a run-time scan width, an eighth of the kernels of the other ops.
template <class Op>
struct one_form : std::false_type {};
template <bool TRUNC, class E>
struct one_form<RetraceOp<0, TRUNC, E>> : std::true_type {};

// Dynamic LDS of a launch with `threads` threads per workgroup.
template <class Op>
size_t dynamic_lds(const Op&, int) { return 0; }
template <bool TRUNC, class E>
size_t dynamic_lds(const RetraceOp<0, TRUNC, E>& op, int threads) {
  return (size_t)(threads / kWave) * action_stage_bytes(op.A);
}

// Such calls of few steps hold one step per thread, in rows of up to 512 steps: four times the
// waves, each with one block of 64 action rows instead of four in turn.  It pays while the
// waves are few enough to start at once; with more, four steps per thread keep the loads of the
// next rows in flight.  Measured on MI355X (us, four steps -> one, float32 / bfloat16): A = 18
// [64,64] 6.57 -> 3.50 / 7.34 -> 3.65, [300,250] 7.19 -> 5.18 / 7.88 -> 4.60, [1024,250] 10.03
// -> 10.76 / 9.42 -> 8.73, [4096,128] 16.02 -> 18.40 / 11.61 -> 12.85; A = 6 [64,64] 4.54 ->
// 2.88, [1024,250] 6.53 -> 7.26 / 7.20 -> 6.17.
template <class Op>
bool step_per_thread(int64_t E, int64_t T) {
  if constexpr (!one_form<Op>::value) return false;
  return T <= kNTWide && E * T <= 8 * kWave * (int64_t)device_cus();  // 8 waves per CU
}

// Rows of more than 2048 steps that one workgroup holds whole (rows_strided_kernel, as many waves
// as the row needs): no look-back, no padding to a tile, and for most ops up to 8192 steps few enough
// registers that two or more workgroups share a CU (Q segments of 4 steps per thread: up to
// 1024 * 4 * Q steps).  (The masked ops' Q = 2 instances hold 71 to 73 registers: two workgroups of
// up to 12 waves; the statistics ops' masked Q = 4 ones 128, and spill up to 20 bytes per lane: one.)
// Against the look-back's tiles, on MI355X (us):
//   * up to 8192 steps (Q = 1, 2) faster at every count of rows, from one on (0.53-0.99 of the tiles' time
//     for seven calls at 1 to 128 rows of 2049 to 8191 steps): GAE [4,2500] by 1.46x, [64,2049]
//     4.34 -> 2.73, [512,5000] 12.2 -> 11.2, masked GAE [512,6000] 14.6 -> 10.6, [2000,5000]
//     49.1 -> 34.1, V-trace [512,5000] 18.2 -> 13.3, bfloat16 [512,6000] 15.7 -> 9.3, TD(lambda)
//     [2000,2049] 15.7 -> 11.1, prefix sum [2000,2049] 14.7 -> 9.2, [256,8192] 5.4 -> 4.6;
//   * up to 16384 steps (Q = 4) with a row for every other CU: masked GAE [256,12000] 1.47x,
//     V-trace 1.40x, GAE [512,10000] 1.11x; fewer rows leave CUs idle that tiles use (GAE
//     [64,16384] 0.75x).  Element-aligned GAE and V-trace keep the phased tiles there ([512,15001]
//     0.96x, 0.98x).
// Retrace's action blocks fill the registers at Q = 2: rows above 4096 steps take it from a row
// per CU on (A = 4 [16,8000] 0.84x, [512,7001] 1.01x, [256,5001] 1.36x).
constexpr int kWholeRowThreads = 1024;
enum class WholeRow { kNever, kTwoSegments, kFourSegments, kFourSegmentsAligned };
template <class Op>
struct whole_row : std::integral_constant<WholeRow, WholeRow::kFourSegments> {};
template <bool TRUNC, class E>
struct whole_row<GaeOp<TRUNC, E>> : std::integral_constant<WholeRow, WholeRow::kFourSegmentsAligned> {};
template <bool TRUNC, class E>
struct whole_row<VtraceOp<TRUNC, E>> : std::integral_constant<WholeRow, WholeRow::kFourSegmentsAligned> {};
template <int NA, bool TRUNC, class E>
struct whole_row<RetraceOp<NA, TRUNC, E>>
    : std::integral_constant<WholeRow, NA == 0 ? WholeRow::kNever : WholeRow::kTwoSegments> {};

// Segments per thread of such a call, 0 for others.
template <class Op>
int whole_row_segments(int64_t E, int64_t T, bool vec) {
  constexpr WholeRow k = whole_row<Op>::value;
  constexpr int64_t steps = kWholeRowThreads * kSeg;
  if (k == WholeRow::kNever || T <= kShortMaxT || T > 4 * steps) return 0;
  if (T <= steps) return 1;
  if (T <= 2 * steps) return k != WholeRow::kTwoSegments || E >= device_cus() ? 2 : 0;
  if (k == WholeRow::kTwoSegments || 2 * E < device_cus()) return 0;
  return vec || k != WholeRow::kFourSegmentsAligned ? 4 : 0;
}

// Workgroups of the launch that launch() makes for Op at [E, T] (E, T > 0).  (The grid of the
// statistics ops, whose callers count workgroups, does not depend on vec.)
template <class Op>
int64_t launch_grid(int64_t E, int64_t T, bool vec = true) {
  if (T > kShortMaxT) {
    if (whole_row_segments<Op>(E, T, vec) > 0) return E;
    const LongShape sh = long_shape<Op>(E, T);
    return chain_grid(E, T, sh.threads, sh.segments);
  }
  if (rows_seg(T) == 1) return rows_grid(E, T, 1, kNT);
  if (step_per_thread<Op>(E, T)) return rows_grid(E, T, 1, T <= kNT ? kNT : kNTWide);
  return rows_grid(E, T, 4, rows_threads(E, T));
}

// Ops whose aligned short rows of 65..128 steps run two row groups per thread
// (rows_pair_kernel): in place of a 512-thread workgroup, a 256-thread one whose threads
// each hold a row of the first and of the second half (same grid, half the waves, twice the
// loads in flight per wave).  float32 Retrace (nine arrays per step) gains from it: C4
// [4096,128] 6.55 -> 6.41 us on MI355X.  Elsewhere the second row's scan lengthens each
// wave's path after its loads: GAE [4096,128] 3.81 -> 3.98 us, V-trace 3.99 -> 4.22 us,
// TD(lambda) 3.11 -> 3.18 us, bfloat16 Retrace 4.77 -> 5.20 us; Retrace [8192,64] is
// unchanged (6.39-6.58 us either way).
template <class Op>
struct paired_rows : std::false_type {};
template <int NA, bool TRUNC>
struct paired_rows<RetraceOp<NA, TRUNC, float>> : std::bool_constant<(NA > 0)> {};

// Whether a launch is one for the normalisation in the scan's own launch: at most `most`
// workgroups that all fit the GPU at once (a wrong answer costs time, not results, but much of it:
// the workgroups that are resident wait out their polls).  The runtime's answer per kernel and
// workgroup size is kept.  It is asked for whole fours of waves: a CU deals a workgroup's waves to
// its four SIMDs, so one of 14 takes four wave slots of the fullest, and two of them do not fit
// SIMDs of seven slots, of which the runtime counts 28 (72-register masked kernels, [300,7000]:
// 350 us in one launch, 23 in two).
inline bool all_resident(const void* kernel, int64_t blocks, int64_t most, int threads, size_t lds) {
  static std::mutex mu;
  static std::map<std::pair<const void*, int>, int> per_cu;
  if (blocks > most || threads < kNormPollers) return false;
  constexpr int kSimdWaves = 4 * kWave;
  threads = (threads + kSimdWaves - 1) / kSimdWaves * kSimdWaves;
  std::lock_guard<std::mutex> lock(mu);
  auto it = per_cu.find({kernel, threads});
  if (it == per_cu.end()) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, lds) != hipSuccess) n = 0;
    it = per_cu.emplace(std::make_pair(kernel, threads), n).first;
  }
  return blocks <= (int64_t)it->second * device_cus();
}

// Most workgroups of a normalised GAE in one launch.  Beyond kNormPollers the exchange costs more
// than a second launch for rows of up to 1024 steps ([6000,128] 8.5 -> 9.5 us, [2000,300] 8.0 ->
// 10.3, [1024,1000] 9.5 -> 11.1), and less where each workgroup holds a longer row: kNormMaxBlocks
// ([512,2048] 9.5 -> 8.9, [512,4096] 16.0 -> 13.8, masked [512,6000] 22.5 -> 19.1, [512,8192]
// 25.8 -> 22.0), for masked rows of up to 2048 steps kNormMaskedBlocks (one launch over two at 300
// rows 0.89-0.96, at 384 0.97-1.03, at 448 1.02-1.07, at 512 1.02-1.08).
constexpr int64_t kNormMaskedBlocks = 384;
inline int64_t one_launch_blocks(int64_t T, bool masked) {
  if (T <= kShortMaxT / 2) return kNormPollers;
  return masked && T <= kShortMaxT ? kNormMaskedBlocks : kNormMaxBlocks;
}
template <class Op>
struct masked_stats : std::false_type {};
template <bool TRUNC, class E>
struct masked_stats<OneLaunchOp<MaskedGaeStatsOp<TRUNC, E>>> : std::true_type {};

// A kernel launch of an op.  hipErrorNotReady, and nothing launched: a OneLaunchOp with more than
// `most` workgroups, or more than fit at once.
template <class Op>
hipError_t launch_kernel(const void* kernel, const Op& op, int64_t blocks, int threads, void** args, hipStream_t stream,
                         int64_t most = kNormPollers) {
  const size_t lds = dynamic_lds(op, threads);
  if constexpr (in_one_launch<Op>::value) {
    if (!all_resident(kernel, blocks, most, threads, lds)) return hipErrorNotReady;
  }
  return hipLaunchKernel(kernel, dim3((unsigned)blocks), dim3(threads), args, lds, stream);
}

template <class Op, int NT, int S, int VEC, int SP>
hipError_t launch_rows(const Op& op, int64_t E, int T, hipStream_t stream) {
  int log2L = ceil_log2((T + S - 1) / S);
  const int64_t grid = rows_grid(E, T, S, NT);
  if (grid * NT > 0xffffffffLL) return hipErrorInvalidValue;  // launch() splits such calls
  void* args[] = {const_cast<Op*>(&op), &E, &T, &log2L};
  // 4-step rows of 33..2048 steps: the instance whose scan width is fixed
  const void* k = reinterpret_cast<const void*>(&rows_kernel<Op, NT, S, VEC, 0, SP>);
  if constexpr (S == 4 && VEC == kAligned && NT == kNTWide && paired_rows<Op>::value) {
    if (log2L == 5) {
      k = reinterpret_cast<const void*>(&rows_pair_kernel<Op, NT / 2, 32, SP>);
      return hipLaunchKernel(k, dim3((unsigned)grid), dim3(NT / 2), args, 0, stream);
    }
  }
  if constexpr (S == 4 && !one_form<Op>::value) {
    if (log2L == 4) k = reinterpret_cast<const void*>(&rows_kernel<Op, NT, S, VEC, 16, SP>);
    else if (log2L == 5) k = reinterpret_cast<const void*>(&rows_kernel<Op, NT, S, VEC, 32, SP>);
    else if (log2L >= 6) k = reinterpret_cast<const void*>(&rows_kernel<Op, NT, S, VEC, kWave, SP>);
  }
  return launch_kernel(k, op, grid, NT, args, stream);
}

// Aligned rows of 1025..2048 steps: one row per 256-thread workgroup, two wave-strided
// segments per thread (rows_strided_kernel), grid = E, for every op but V-trace and
// Retrace, in both storage types (so that a bfloat16 result stays the float32 kernels'
// result rounded).  Against rows_kernel's 512 threads of one segment, on MI355X:
// TD(lambda) [256,2048] 3.47 -> 3.35 us, prefix sum [256,2048] 3.28 -> 3.09 us (bfloat16
// 3.12 -> 3.06), GAE [256,2048] 4.33 -> 4.27 us, TD(lambda) [512,1100] 4.14 -> 4.00 us,
// the other bfloat16 calls unchanged.  V-trace (4.42 -> 4.44 us, bfloat16 3.88 -> 3.99)
// and Retrace (6.66 -> 6.64 us, bfloat16 5.47 -> 5.74) keep rows_kernel, as do
// element-aligned rows ([256,2047] 3.76 -> 3.78 us).
template <class Op>
struct strided_rows : std::true_type {};
template <bool TRUNC, class E>
struct strided_rows<VtraceOp<TRUNC, E>> : std::false_type {};
template <int NA, bool TRUNC, class E>
struct strided_rows<RetraceOp<NA, TRUNC, E>> : std::false_type {};

// One row per workgroup of `threads` (at most NT), Q segments of 4 steps per thread.
template <class Op, int NT, int Q, int VEC>
hipError_t launch_strided(const Op& op, int64_t E, int T, int threads, hipStream_t stream) {
  if (E * threads > 0xffffffffLL) return hipErrorInvalidValue;  // launch() splits such calls
  int unused = 0;
  void* args[] = {const_cast<Op*>(&op), &E, &T, &unused};
  return launch_kernel(reinterpret_cast<const void*>(&rows_strided_kernel<Op, NT, Q, VEC, 1>), op, E, threads, args,
                       stream, one_launch_blocks(T, masked_stats<Op>::value));
}

template <class Op, int VEC>
hipError_t launch_whole_row(const Op& op, int64_t E, int T, int segments, hipStream_t stream) {
  const int wave_steps = kWave * kSeg * segments;
  const int threads = kWave * ((T + wave_steps - 1) / wave_steps);
  if (segments == 1) return launch_strided<Op, kWholeRowThreads, 1, VEC>(op, E, T, threads, stream);
  if constexpr (whole_row<Op>::value != WholeRow::kTwoSegments) {
    if (segments == 4) return launch_strided<Op, kWholeRowThreads, 4, VEC>(op, E, T, threads, stream);
  }
  return launch_strided<Op, kWholeRowThreads, 2, VEC>(op, E, T, threads, stream);
}

// Look-back poll budgets (rlk_debug_lookback): polls before a wait gives up (~1 s), and
// polls before a wait on a predecessor that has published nothing computes it instead.
constexpr int kFallbackPolls = 256;
inline std::atomic<int> g_spin_limit{kSpinLimit};
inline std::atomic<int> g_fallback_polls{kFallbackPolls};

// Long rows: one tile of kLongThreads * 4 * Q steps per workgroup, grid = nslots * (tiles
// of the fullest slot) (see chain_kernel in rlk_engine.hpp).
//
// Placement of the tiles in the block index.  By default the slots interleave (block b
// holds a tile of slot b % nslots), so position j of every row is dispatched before
// position j + 1 of any, and with 8 XCDs taking blocks round-robin a row's tiles share one
// XCD.  A call of at most 16 rows whose tiles fill every CU at least once takes the rows
// one after another instead (a row's tiles consecutive, spread over the XCDs).  Measured on
// MI355X, A/B twice in one process, bit-identical results: V-trace [16,131072]
// 13.39 -> 12.50 us, GAE [16,131072] 12.78 -> 11.69, TD(lambda) [16,131072] 9.65 -> 8.86,
// discounted returns [8,262144] 9.18 -> 8.46 and [16,131072] 8.28 -> 8.22, prefix sum
// [16,131072] 8.32 -> 7.80; [8,2^20], [4,2^19..2^21] unchanged.  Where the grid is smaller
// than the chip ([16,65536], [12,131072], [16,40000]) or the rows are many ([32..200] rows)
// the row-major order lost up to 1.35 us (TD(lambda) [96,30000]), so those keep the
// interleave.
inline int chain_row_major(int64_t E, int64_t grid) { return E <= 16 && grid >= device_cus() ? 1 : 0; }

// VEC = kPhased: phase0 = the element phase of row 0's arrays.
template <class Op, int Q, int VEC, int SP, int NT = Op::kLongThreads>
hipError_t launch_chain(const Op& op, int64_t E, int T, uint64_t* ws, hipStream_t stream, int phase0) {
  static_assert(NT * kSeg * Q >= kMinTile, "the workspace is sized for the smallest tile");
  constexpr int64_t tile = (int64_t)NT * kSeg * Q;
  int tpr = (int)((T + tile - 1) / tile);
  const int64_t grid = chain_grid(E, T, NT, Q);
  if (grid * NT > 0xffffffffLL) return hipErrorInvalidValue;  // launch() splits such calls
  uint64_t* fb = ws + kStatusOffset + kStatusWords * status_tiles(E, T);
  int spin_limit = g_spin_limit.load(std::memory_order_relaxed);
  int fallback_polls = g_fallback_polls.load(std::memory_order_relaxed);
  int row_major = chain_row_major(E, grid);
  void* args[] = {const_cast<Op*>(&op), &E, &T, &tpr, &ws, &fb, &spin_limit, &fallback_polls,
                  &row_major, &phase0};
  return hipLaunchKernel(reinterpret_cast<const void*>(&chain_kernel<Op, NT, Q, VEC, SP>),
                         dim3((unsigned)grid), dim3(NT), args, dynamic_lds(op, NT), stream);
}

template <class Op, int VEC, int SP>
hipError_t launch_long(const Op& op, int64_t E, int T, uint64_t* ws, hipStream_t stream, int phase0) {
  const LongShape sh = long_shape<Op>(E, T);
  if constexpr (wide_long_tiles<Op>::value) {
    if (sh.threads == 1024 && sh.segments == 4) return launch_chain<Op, 4, VEC, SP, 1024>(op, E, T, ws, stream, phase0);
    if (sh.threads == 1024 && sh.segments == 2) return launch_chain<Op, 2, VEC, SP, 1024>(op, E, T, ws, stream, phase0);
  }
  constexpr int hq = half_width_segments<Op>::value;
  if constexpr (hq != 0) {
    if (sh.threads == 512 && sh.segments == hq) return launch_chain<Op, hq, VEC, SP, 512>(op, E, T, ws, stream, phase0);
  }
  if constexpr (Op::kLongThreads == 1024 && hq != kMinQ) {
    if (sh.threads == 512 && sh.segments == kMinQ) return launch_chain<Op, kMinQ, VEC, SP, 512>(op, E, T, ws, stream, phase0);
  }
  const int q = sh.segments;
  if constexpr (Op::kLongMaxSegments >= 8)
    if (q == 8) return launch_chain<Op, 8, VEC, SP>(op, E, T, ws, stream, phase0);
  if constexpr (Op::kLongMaxSegments >= 4)
    if (q == 4) return launch_chain<Op, 4, VEC, SP>(op, E, T, ws, stream, phase0);
  return launch_chain<Op, 2, VEC, SP>(op, E, T, ws, stream, phase0);
}

// Output stores: non-temporal (the default) or write-through (sc1, store_quad_wt), per
// launch, by what measured faster on MI355X (one process, three builds -- nt, sc1 and
// plain stores -- alternated, 88 op x shape x storage cases; µs, nt -> sc1):
//   * bfloat16 outputs: sc1 everywhere, 1-4% faster in every case but one (Retrace
//     [4096,128], equal): V-trace [4096,128] 3.49 -> 3.34, prefix sum [16,131072]
//     6.77 -> 6.54, TD(lambda) [16,131072] 7.07 -> 6.83;
//   * float32 short rows that span several waves (more than 256 steps) in launches writing
//     at least 1 MB, or launches writing at least 12 MB: sc1, 2-4% (TD(lambda) [256,2048]
//     3.35 -> 3.25, Retrace [256,2048] 6.71 -> 6.49, V-trace [1024,512] 4.38 -> 4.21,
//     V-trace [16384,128] 11.19 -> 10.75); rows of up to 256 steps in smaller launches keep
//     nt (GAE [4096,128] 3.77 against 3.94, V-trace 3.99 against 4.20, GAE [2048,256] 3.83
//     against 3.98), as does GAE [64,512] (128 KB written, 2.25 against 2.27);
//   * float32 long rows: sc1 when the grid is at most one tile per CU, for every op but
//     V-trace and Retrace (discounted returns [16,131072] 8.00 -> 7.86, prefix sum
//     [16,131072] 7.66 -> 7.49, TD(lambda) [8,262144] 8.92 -> 8.79); nt with more tiles
//     (discounted [64,40000] 8.99 against 9.58) and for V-trace ([16,131072] 12.40 against
//     12.70);
//   * rows held whole by a workgroup (rows_strided_kernel): sc1, 2-15% (GAE [256,2500] 3.63
//     against 4.19, V-trace [512,4096] 10.2 against 10.8; equal at 2049 steps).
// Plain stores were never the fastest by more than 3% and lost up to 13% elsewhere.  The
// policy is a kernel template argument (SP), so a non-temporal instance is the same code
// as before write-through stores existed.
template <class Op>
struct n_outputs : std::integral_constant<int, 1> {};
template <bool TRUNC, class E>
struct n_outputs<VtraceOp<TRUNC, E>> : std::integral_constant<int, 2> {};
template <int NA, bool TRUNC, class E>
struct n_outputs<RetraceOp<NA, TRUNC, E>> : std::integral_constant<int, 2> {};
template <bool TRUNC, class E>
struct n_outputs<GaeStatsOp<TRUNC, E>> : std::integral_constant<int, 2> {};
template <bool TRUNC, class E>
struct n_outputs<MaskedGaeStatsOp<TRUNC, E>> : std::integral_constant<int, 2> {};
template <class StatsOp>
struct n_outputs<OneLaunchOp<StatsOp>> : n_outputs<StatsOp> {};
template <class Op>
struct long_rows_write_through : std::true_type {};
template <bool TRUNC, class E>
struct long_rows_write_through<VtraceOp<TRUNC, E>> : std::false_type {};
template <int NA, bool TRUNC, class E>
struct long_rows_write_through<RetraceOp<NA, TRUNC, E>> : std::false_type {};

enum class Kernel { kRows, kChain };
// The policies a kernel can be launched with for an op: bfloat16 outputs always write through
// (as rows_strided_kernel does), float32 V-trace and Retrace long rows never; only the policies
// listed here are instantiated.
template <class Op, Kernel K>
struct store_policies {
  static constexpr bool kBf16 = std::is_same<typename Op::Elem, bf16>::value;
  static constexpr bool kWriteThrough = kBf16 || (K != Kernel::kChain && !one_form<Op>::value) || long_rows_write_through<Op>::value;
  static constexpr bool kNonTemporal = !kBf16;
  static_assert(kWriteThrough || kNonTemporal, "some store policy");
};
template <class Op, Kernel K>
int store_write_through(int64_t E, int64_t T) {
  using P = store_policies<Op, K>;
  if constexpr (!P::kNonTemporal) return 1;
  if constexpr (!P::kWriteThrough) return 0;
  if constexpr (K == Kernel::kChain) return launch_grid<Op>(E, T) <= device_cus() ? 1 : 0;
  const int64_t out_bytes = E * T * (int64_t)sizeof(float) * n_outputs<Op>::value;
  return (((T + 3) / 4 > kWave && out_bytes >= (int64_t{1} << 20)) || out_bytes >= (int64_t{12} << 20)) ? 1 : 0;
}
// rlk_debug_store_policy: -1 the rule above, 0 / 1 non-temporal / write-through wherever
// the launch has an instance of that policy.
inline std::atomic<int> g_store_policy{-1};

// Calls f(std::integral_constant<int, SP>) with SP the launch's store policy.
template <class Op, Kernel K, class F>
hipError_t dispatch_store_policy(int64_t E, int64_t T, F&& f) {
  using P = store_policies<Op, K>;
  if constexpr (P::kWriteThrough && P::kNonTemporal) {
    const int forced = g_store_policy.load(std::memory_order_relaxed);
    if (forced >= 0 ? forced == 1 : store_write_through<Op, K>(E, T) != 0)
      return f(std::integral_constant<int, 1>{});
    return f(std::integral_constant<int, 0>{});
  } else {
    return f(std::integral_constant<int, P::kWriteThrough ? 1 : 0>{});
  }
}

// Ops that take long rows in the phased access mode: all but Retrace (whose [E, T, A]
// arrays have no common row phase) and the statistics ops of compute_gae_normalized (the
// steps a phased row takes ahead of its tiles would be missing from their statistics).
template <class Op>
struct phased_rows : std::true_type {};
template <int NA, bool TRUNC, class E>
struct phased_rows<RetraceOp<NA, TRUNC, E>> : std::false_type {};
template <bool TRUNC, class E>
struct phased_rows<GaeStatsOp<TRUNC, E>> : std::false_type {};
template <bool TRUNC, class E>
struct phased_rows<MaskedGaeStatsOp<TRUNC, E>> : std::false_type {};

// ---------------------------------------------------------------------------------------
// Calls beyond one launch.  HIP launches at most 2^32 - 1 work-items per grid dimension
// (hip_runtime_api.h, hipLaunchKernel), and every launch here is one-dimensional with at
// most 1024 threads per workgroup.  Rows are independent, so a call whose launch would
// need more than kMaxLaunchBlocks workgroups runs as calls over consecutive row ranges,
// in row order on the same stream, each within the limit.  Short rows reach it from 0.8
// billion steps (3-step rows, 64 per workgroup: 3.2 GB per float32 array) to 8.6 billion,
// long rows from ~4.2 million rows of one tile each: sizes MI355X's 288 GB holds.
// ---------------------------------------------------------------------------------------
constexpr int64_t kMaxLaunchBlocks = ((int64_t{1} << 32) - 1) / 1024;

template <class P>
void skip(P*& p, int64_t n) {
  if (p != nullptr) p += n;
}
// boot: one value per row (RLK_BOOT_ROW) or [E, T] (RLK_BOOT_FULL)
template <class E>
void skip_boot(const E*& boot, int boot_mode, int64_t r0, int64_t T) {
  skip(boot, boot_mode == RLK_BOOT_FULL ? r0 * T : r0);
}

// An op's arrays advanced by r0 rows: [E, T] arrays by r0 * T elements, [E, T, A] ones by
// r0 * T * A, per-row ones by r0.  (The statistics ops' partials are placed by the caller.)
template <bool TR, class E>
void skip_rows(GaeOp<TR, E>& op, int64_t r0, int64_t T) {
  const int64_t n = r0 * T;
  skip(op.r, n), skip(op.v, n), skip(op.term, n), skip(op.trunc, n), skip(op.out, n);
  skip_boot(op.boot, op.boot_mode, r0, T);
}
template <bool TR, class E>
void skip_rows(GaeStatsOp<TR, E>& op, int64_t r0, int64_t T) {
  skip_rows(static_cast<GaeOp<TR, E>&>(op), r0, T);
  skip(op.returns, r0 * T);
}
template <bool TR, class E>
void skip_rows(MaskedGaeOp<TR, E>& op, int64_t r0, int64_t T) {
  const int64_t n = r0 * T;
  skip(op.r, n), skip(op.v, n), skip(op.term, n), skip(op.trunc, n), skip(op.mask, n);
  skip(op.out, n);
  skip_boot(op.boot, op.boot_mode, r0, T);
}
template <bool TR, class E>
void skip_rows(MaskedGaeStatsOp<TR, E>& op, int64_t r0, int64_t T) {
  skip_rows(static_cast<MaskedGaeOp<TR, E>&>(op), r0, T);
  skip(op.returns, r0 * T);
}
template <bool TR, class E>
void skip_rows(VtraceOp<TR, E>& op, int64_t r0, int64_t T) {
  const int64_t n = r0 * T;
  skip(op.lpt, n), skip(op.lpb, n), skip(op.v, n), skip(op.r, n), skip(op.term, n);
  skip(op.trunc, n), skip(op.targets, n), skip(op.adv, n);
  skip_boot(op.boot, op.boot_mode, r0, T);
}
template <int NA, bool TR, class E>
void skip_rows(RetraceOp<NA, TR, E>& op, int64_t r0, int64_t T) {
  const int64_t n = r0 * T;
  skip(op.pi, n * op.A), skip(op.nq, n * op.A);
  skip(op.mu, n), skip(op.q, n), skip(op.act, n), skip(op.r, n), skip(op.term, n);
  skip(op.trunc, n), skip(op.targets, n), skip(op.adv, n);
}
template <bool NV, bool TR, class E>
void skip_rows(ReturnsOp<NV, TR, E>& op, int64_t r0, int64_t T) {
  const int64_t n = r0 * T;
  skip(op.r, n), skip(op.nv, n), skip(op.term, n), skip(op.trunc, n), skip(op.out, n);
  skip_boot(op.boot, op.boot_mode, r0, T);
}
template <class E>
void skip_rows(DoneGatedForwardOp<E>& op, int64_t r0, int64_t T) {
  const int64_t n = r0 * T;
  skip(op.x, n), skip(op.dones, n), skip(op.out, n), skip(op.seed, r0);
}
template <bool FWD, class E>
void skip_rows(AffineScanOp<FWD, E>& op, int64_t r0, int64_t T) {
  const int64_t n = r0 * T;
  skip(op.u, n), skip(op.v, n), skip(op.out, n), skip(op.carry, r0);
}

// Rows per launch of a call: all E when one launch holds the call, else the most rows
// (a multiple of 512 where that is at least 512: whole workgroups of every short-row shape)
// whose launch stays within kMaxLaunchBlocks.
template <class Op>
int64_t rows_per_launch(int64_t E, int64_t T, bool vec = true) {
  const int64_t g = launch_grid<Op>(E, T, vec);
  if (g <= kMaxLaunchBlocks) return E;
  int64_t n = (int64_t)((double)E * (double)kMaxLaunchBlocks / (double)g);  // grid ~ rows
  n = n < 1 ? 1 : n > E ? E : n;
  for (const int64_t unit : {int64_t{512}, int64_t{1}}) {
    if (n < unit) continue;
    int64_t m = n / unit * unit;
    while (m > unit && launch_grid<Op>(m, T, vec) > kMaxLaunchBlocks) m -= unit;
    if (launch_grid<Op>(m, T, vec) <= kMaxLaunchBlocks) return m;
  }
  return 1;  // one row of at most 2^30 steps is at most 2^18 tiles
}

// Workgroups of all the launches of a call, following launch()'s row ranges: the
// statistics ops write one partial per workgroup.
template <class Op>
int64_t call_blocks(int64_t E, int64_t T) {
  if (E <= 0 || T <= 0) return 0;
  const int64_t rows = rows_per_launch<Op>(E, T);
  if (rows >= E) return launch_grid<Op>(E, T);
  int64_t total = 0;
  for (int64_t r0 = 0; r0 < E; r0 += rows) total += call_blocks<Op>(rows < E - r0 ? rows : E - r0, T);
  return total;
}

// launch()'s answer to a OneLaunchOp where the call is not one for it.
constexpr int kNotTaken = 1;
inline int status_of(hipError_t e) {
  return e == hipSuccess ? RLK_OK : e == hipErrorNotReady ? kNotTaken : RLK_ERR_LAUNCH;
}

// vec: kAligned access.  phase0 >= 0: the element phase every [E, T] array of the call
// shares at row 0 (common_phase), for the phased access of long rows when T % 4 != 0.
template <class Op>
int launch(const Op& op, int64_t E, int64_t T, bool vec, void* workspace, size_t workspace_bytes_given,
           void* stream, int phase0 = -1) {
  if (E < 0 || T < 0 || T > (int64_t{1} << 30)) return RLK_ERR_INVALID_ARGUMENT;
  if (E == 0 || T == 0) return RLK_OK;
  const CusScope cus;
  const int64_t rows = rows_per_launch<Op>(E, T, vec);
  if constexpr (in_one_launch<Op>::value) {
    if (rows < E) return kNotTaken;
  } else if (rows < E) {
    int64_t blocks = 0;  // the statistics ops' partials of the ranges before this one
    for (int64_t r0 = 0; r0 < E; r0 += rows) {
      const int64_t n = rows < E - r0 ? rows : E - r0;
      Op part = op;
      skip_rows(part, r0, T);
      if constexpr (Op::kBlockStats) part.partials = op.partials + kStatWords * blocks;
      const int ph = phase0 < 0 ? -1 : (int)((phase0 + (r0 & 3) * (T & 3)) & 3);
      const int st = launch(part, n, T, vec, workspace, workspace_bytes_given, stream, ph);
      if (st != RLK_OK) return st;
      blocks += call_blocks<Op>(n, T);
    }
    return RLK_OK;
  }
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int Ti = (int)T;
  hipError_t e = hipErrorInvalidValue;
  if (T > kShortMaxT) {
    uint64_t* ws = reinterpret_cast<uint64_t*>(workspace);
    if (!in_one_launch<Op>::value && (ws == nullptr || workspace_bytes_given < workspace_bytes(E, T) || !aligned16(ws)))
      return RLK_ERR_WORKSPACE;
    if constexpr (whole_row<Op>::value != WholeRow::kNever) {
      const int segments = whole_row_segments<Op>(E, T, vec);
      if (segments > 0) {
        e = vec ? launch_whole_row<Op, kAligned>(op, E, Ti, segments, s)
                : launch_whole_row<Op, kElementAligned>(op, E, Ti, segments, s);
        return status_of(e);
      }
    }
    if constexpr (in_one_launch<Op>::value) return kNotTaken;
    const bool phased = phased_rows<Op>::value && !vec && phase0 >= 0 && T % 4 != 0;
    if constexpr (!in_one_launch<Op>::value) e = dispatch_store_policy<Op, Kernel::kChain>(E, T, [&](auto sp) {
      constexpr int SP = decltype(sp)::value;
      if constexpr (phased_rows<Op>::value) {
        if (phased) return launch_long<Op, kPhased, SP>(op, E, Ti, ws, s, phase0);
      }
      if constexpr (!one_form<Op>::value) {
        if (vec) return launch_long<Op, kAligned, SP>(op, E, Ti, ws, s, 0);
      }
      return launch_long<Op, kElementAligned, SP>(op, E, Ti, ws, s, 0);
    });
  } else if (strided_rows<Op>::value && vec && T > kShortMaxT / 2) {
    if constexpr (strided_rows<Op>::value) {
      static_assert(kStridedThreads * kSeg * kStridedSegments == kShortMaxT, "one row per workgroup");
      e = launch_strided<Op, kStridedThreads, kStridedSegments, kAligned>(op, E, Ti, kStridedThreads, s);
    }
  } else {
    e = dispatch_store_policy<Op, Kernel::kRows>(E, T, [&](auto sp) {
      constexpr int SP = decltype(sp)::value;
      if (rows_seg(T) == 1) return launch_rows<Op, kNT, 1, kElementAligned, SP>(op, E, Ti, s);
      if constexpr (one_form<Op>::value) {
        if (step_per_thread<Op>(E, T))
          return T <= kNT ? launch_rows<Op, kNT, 1, kElementAligned, SP>(op, E, Ti, s)
                          : launch_rows<Op, kNTWide, 1, kElementAligned, SP>(op, E, Ti, s);
      }
      const bool narrow = rows_threads(E, T) == kNT;
      if constexpr (!one_form<Op>::value) {
        if (vec)
          return narrow ? launch_rows<Op, kNT, 4, kAligned, SP>(op, E, Ti, s)
                        : launch_rows<Op, kNTWide, 4, kAligned, SP>(op, E, Ti, s);
      }
      return narrow ? launch_rows<Op, kNT, 4, kElementAligned, SP>(op, E, Ti, s)
                    : launch_rows<Op, kNTWide, 4, kElementAligned, SP>(op, E, Ti, s);
    });
  }
  return status_of(e);
}

// Empty shapes are a successful no-op (their data pointers may be null); negative sizes
// are rejected by launch().
inline bool is_empty(int64_t E, int64_t T) { return (E == 0 && T >= 0) || (T == 0 && E >= 0); }

inline bool valid_boot(const void* boot, int mode) {
  if (mode == RLK_BOOT_NONE) return true;
  if (mode == RLK_BOOT_ROW || mode == RLK_BOOT_FULL) return boot != nullptr;
  return false;
}

// Vector segments need every [E, T] array aligned to four elements (absent ones pass).
template <class E>
bool quad_aligned(const E* p) {
  return p == nullptr || (reinterpret_cast<uintptr_t>(p) % (4 * sizeof(E))) == 0;
}
template <class E, class... R>
bool quad_aligned(const E* p, const R*... rest) {
  return quad_aligned(p) && quad_aligned(rest...);
}
// The element phase (address / sizeof(E), mod 4) that every non-null array shares, or -1
// when two differ or one is not element-aligned.  Arrays of one call hold [E, T] rows at
// the same offsets, so a shared phase at row 0 makes every row's phase shared too.
template <class E, class... P>
int common_phase(const P*... ptrs) {
  int ph = -1;
  for (const E* p : {static_cast<const E*>(ptrs)...}) {
    if (p == nullptr) continue;
    const uintptr_t a = reinterpret_cast<uintptr_t>(p);
    if (a % sizeof(E) != 0) return -1;
    const int q = (int)((a / sizeof(E)) & 3);
    if (ph >= 0 && q != ph) return -1;
    ph = q;
  }
  return ph;
}

// rlk_bf16 (raw bits) <-> the kernels' bf16 storage type
inline const bf16* B(const rlk_bf16* p) { return reinterpret_cast<const bf16*>(p); }
inline bf16* B(rlk_bf16* p) { return reinterpret_cast<bf16*>(p); }

}  // namespace rlk
