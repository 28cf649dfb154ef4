// Host-side pieces shared by the translation units of the library: launch planning,
// device checks, the ordering of scans across streams, residency of a kernel.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include <initializer_list>
#include <mutex>

#include "../../include/fss_scan.h"
#include "fss_device.h"

namespace fss {

extern thread_local int tls_hip_error;  // hipError_t of this thread's last failed HIP call
extern thread_local uint64_t tls_plans_computed;  // fss_debug_plans_computed
extern uint32_t g_spin_limit;           // polls before a look-back gives up (a test may lower it)
#ifdef FSS_TRACE
extern uint64_t *g_trace;
#endif

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Register budget: packed dwords a lane may hold per input tensor.
inline int max_vec_steps(int dtype) { return dtype != FSS_F32 ? 64 : 32; }  // vec*steps

// Most waves a workgroup of the row-major kernels may have, by what a lane holds: the kernels
// are compiled for that many (launch bounds), so that their registers fit without spilling.
// 16 waves leave a lane 128 registers: enough for 64 dwords of rows with up to two channels
// per lane.  Wider lanes (whose chaining state grows with the channels) and the plain
// backward with 32 steps of two channels (three tensors) get 256 or 512 registers instead.
constexpr int max_waves(int esize, int vec, int steps, bool bwd, bool gated) {
  const int dwords = vec * esize >= 4 ? vec * esize / 4 : 1;  // per lane and row
  if (vec >= 8) return 4;
  if (vec >= 4) return 8;
  if (!gated && vec >= 2 && dwords * steps * (bwd ? 3 : 2) > 64) return 8;
  return 16;
}

// LDS: one (A,B) slot per lane and vector element for every wave, twice (tiles
// alternate between two sets), and the same for every wave that looks back (per
// column tile of the workgroup).  `waves` counts all waves of the workgroup, of which
// waves/cols lie along time.
constexpr size_t kLdsBudget = 60 * 1024;
inline int look_waves(int waves, int vec, int cols = 1) {
  const int along_time = waves / cols;
  int look = along_time < kMaxLookWaves ? along_time : kMaxLookWaves;
  while (look > 1 && static_cast<size_t>(2 * waves + look * cols) * vec * 512 > kLdsBudget) --look;
  return look;
}
inline size_t lds_bytes(int waves, int vec, int cols = 1) {
  return static_cast<size_t>(2 * waves + look_waves(waves, vec, cols) * cols) * vec * 512;
}

inline bool config_valid(const fss_config &c, int dtype, bool gated = false, int dir = FSS_FWD) {
  // the gated kernels exist for 4 bytes (or one element) per lane; their backward holds
  // four tensors, so at most 16 timesteps per lane
  if (gated && (c.vec > (dtype != FSS_F32 ? 2 : 1) || (dir == FSS_BWD && c.steps > 16))) return false;
  const bool vec_ok = dtype != FSS_F32 ? (c.vec == 1 || c.vec == 2 || c.vec == 4 || c.vec == 8)
                                        : (c.vec == 1 || c.vec == 2 || c.vec == 4);
  const bool steps_ok = c.steps == 8 || c.steps == 16 || c.steps == 32;
  if (!vec_ok || !steps_ok) return false;
  if (c.vec * c.steps > max_vec_steps(dtype)) return false;
  if (dtype != FSS_F32 && c.vec == 1 && c.steps > 32) return false;
  if (c.waves < 1 || c.waves > max_waves(dtype != FSS_F32 ? 2 : 4, c.vec, c.steps, (dir & 1) == FSS_BWD, gated)) return false;
  if (c.cols != 1 && c.cols != 2) return false;
  if (c.waves % c.cols != 0) return false;
  if (lds_bytes(c.waves, c.vec, c.cols) > kLdsBudget) return false;
  return true;
}

// CUs of an unpartitioned MI355X: what "one tile per CU" means when a launch is planned
// (planning must work without a device; the grid itself is sized from the runtime's count).
constexpr int64_t kCus = 256;

// Chunks of one sequence that a full grid works on at once: the spacing of the chain's anchors
// (chain_anchor in fss_device.h).  Planned from a nominal device - kCus compute units holding
// 16 waves of a scan each, though kernels of up to 16 steps have registers for 24: with 8 or 12 waves a grid of those
// works on one and a half or two periods at once, and a chunk's anchor may still be in flight - and from nothing that can differ between two launches of one
// configuration (not the grid actually launched, not the device's own CU count), so that the
// order in which carries are composed, and with it every bit of the result, is fixed by the
// shape and the configuration.
inline int chain_period(int64_t n_groups, int waves) {
  const int64_t per_cu = waves >= 16 ? 1 : 16 / (waves > 0 ? waves : 1);
  const int64_t nominal_grid = kCus * per_cu;
  const int64_t period = ceil_div(nominal_grid, n_groups > 0 ? n_groups : 1);
  return static_cast<int>(period < 1 ? 1 : (period > (1 << 20) ? (1 << 20) : period));
}

// The divisors of a launch whose other numbers are set (the tile order's come with the grid); a launch
// that chains nothing, as a decode step's, needs only the first two.
inline void set_divisors(ScanArgs &args) {
  args.by_groups = fast_div(static_cast<uint32_t>(args.n_groups));
  args.by_row = fast_div(static_cast<uint32_t>(args.tiles_per_row));
  args.by_period = args.by_reach = args.by_look = FastDiv{1u, 0, 0};
  if (args.n_chunks <= 1) return;
  args.by_period = fast_div(static_cast<uint32_t>(args.period));
  args.by_reach = fast_div(static_cast<uint32_t>(args.look_waves * kMaxSpan));
  args.by_look = fast_div(static_cast<uint32_t>(args.look_waves));
}

// One candidate launch configuration: taken when it yields at least `need` tiles.
struct Rung {
  int vec, steps, waves;
  int64_t need;
};

// Column tiles a workgroup covers side by side (fss_config.cols) when the caller leaves the
// choice open; vec, steps and waves of `c` are already fixed.  Two column tiles make every row a
// workgroup touches 512 contiguous bytes instead of 256 and its chunks half as long.  Measured in
// the forward with 4 bytes per lane, 32 steps and 16 waves (bf16, 49 shapes, bs 2..16, seq
// 2048..16384, d 512..4096, tensor sets in rotation so that nothing is found in a cache): where
// the launch has more than one and at most two tiles per CU, 5-13 % faster on 8 shapes of 9;
// with four tiles per CU +-0, with eight 1 % slower; in the backward, whose chunks would shrink
// to 128 steps, slower throughout.  At bs 8 seq 4096 d 1024: forward 42.8 -> 40.9 us and the
// forward+backward step 105.4 -> 103.3 us over tensor sets in rotation, a forward behind flushed
// caches 48.2 -> 45.6 us; when the tensors are found in the memory-side cache again (forward and
// backward alternating on one set of tensors) forward 31.0 -> 32.2 us, step 88.6 -> 90.5 us.  The
// library cannot know which of the two it is in and takes what serves the caller whose tensors
// come from memory.  The choice depends on the shape alone - never on a policy or on earlier
// calls - because a different tiling rounds the carries differently.
inline int choose_cols(const fss_config &c, int64_t bs, int64_t seq, int64_t d, int dtype, int dir, bool gated) {
  if (gated || dir != FSS_FWD) return 1;
  const int esize = dtype != FSS_F32 ? 2 : 4;
  if (c.vec * esize != 4 || c.steps != 32 || c.waves != 16) return 1;
  const int64_t tiles_per_row = ceil_div(d, 64 * static_cast<int64_t>(c.vec));
  if (tiles_per_row % 2 != 0) return 1;
  const int64_t tiles = bs * tiles_per_row * ceil_div(seq, static_cast<int64_t>(c.steps) * c.waves);
  return tiles > kCus && tiles <= 2 * kCus ? 2 : 1;
}

// An estimate, in ns, of what a launch of a forward kernel takes with a tiling, for comparing tilings of one shape.  A
// regression on eight terms: a launch, the steps that a wave takes one after the other, the same times channels per lane, the
// chain (a round trip to memory, and more maps to find the more chunks of a sequence are in flight at
// once), every round of the resident workgroups after the first, and the bytes, padding included: what the busiest
// compute unit moves, and all of them together.  Fitted to 4600 pairs of a shape of 2^17 to 2^25 elements (bs 1..64, seq
// 16..65536, d 64..4096, a quarter of the widths odd or ragged) and a configuration, each weighted by how near it came to
// the shape's fastest.  The terms grow together in such pairs (steps with bytes, channels with both), so no coefficient is
// a cost by itself: the negative `channel_step` of 16 bits does not say that a step of two channels takes less time than
// one of one.  What the estimate is good for is measured on 480 other shapes (profiles/forward_tilings_pairs.csv, 5166 pairs,
// checked by tests/test_forward_tilings.py): its values scatter by 11 to 12 % around the plain kernels' times and 20 % around
// the gated.
struct ForwardCost {
  double launch, step, channel_step, chain, depth, round, unit_bytes, all_bytes;
};
constexpr ForwardCost kForwardCost[2][2] = {  // [16 bits, 32 bits][plain, gated]
    {{3315, 55, -15, 772, 564, 2166, 11.47e-3, 17.98e-3}, {3230, 170, -54, 935, 545, 2786, 20.11e-3, 16.54e-3}},
    {{2870, 11, 2, 847, 621, 3097, 8.80e-3, 18.24e-3}, {3203, 15, 15, 511, 493, 2282, 8.51e-3, 23.92e-3}}};
inline double forward_ns(const ForwardCost &m, int64_t bs, int64_t seq, int64_t d, int esize, int vec, int steps, int waves) {
  const int64_t columns = bs * ceil_div(d, 64 * static_cast<int64_t>(vec));
  const int64_t chunks = ceil_div(seq, static_cast<int64_t>(steps) * waves), tiles = columns * chunks;
  // (registers: six waves of up to 16 steps on a SIMD, four of 32)
  const int64_t resident = kCus * ((steps <= 16 ? 6 : 4) / ((waves + 3) / 4));
  const int64_t in_flight = ceil_div(resident, columns) < chunks ? ceil_div(resident, columns) : chunks;
  const double tile_bytes = 3.0 * 64 * vec * steps * waves * esize;
  return m.launch + m.step * steps + m.channel_step * vec * steps + (chunks > 1 ? m.chain : 0) +
         m.depth * __builtin_sqrt(static_cast<double>(in_flight - 1)) + m.round * static_cast<double>(ceil_div(tiles, resident) - 1) +
         tile_bytes * (m.unit_bytes * static_cast<double>(ceil_div(tiles, kCus)) + m.all_bytes / kCus * static_cast<double>(tiles));
}

// Forwards of fewer elements than this take the tiling that forward_ns finds fastest, if it is clearly faster
// than the ladder's (complete_config): the ladder was drawn from launches that fill the device, and
// below them "the largest tile that leaves one per compute unit" is the wrong question.  What a choice loses against the fastest of
// about eleven tilings on those 480 shapes, in the mean, ladder and estimate, below a sixteenth of the limit, a quarter, half
// and the limit, and from there to twice it (where the ladder is taken):
//   bf16   25.6 and 3.6 %, 12.6 and 3.1, 9.2 and 2.1, 6.1 and 3.2;   5.6 and 2.4
//   gated  27.7 and 1.9 %, 34.4 and 5.6, 33.9 and 9.9, 20.8 and 7.3;  3.4 and 5.6
//   fp32   below a quarter 19.1 and 3.8 %, 14.9 and 4.6, 8.2 and 3.3;  4.5 and 3.8
//   gated  19.1 and 2.5 %, 22.7 and 8.5, 10.7 and 4.3, 4.2 and 4.3;  7.5 and 9.8
// So the gated limits lie where the ladder becomes the better one; the plain ones lie lower than they could, at the sizes
// (for 16 bits just below 2^24 elements) that the ladder's own sweeps cover.  The margin keeps out what the
// estimate cannot tell apart: of the 349 shapes below the limits 8 are slower by it than with the ladder, gated ones
// all, (3, 9524, 128) 11.3 -> 13.1 us the furthest.  Furthest from the fastest: gated (30, 610, 144) 16.7 us, two channels and
// 12 waves 10.8.
constexpr int64_t forward_model_elems(bool narrow, bool gated) {
  return narrow ? (gated ? int64_t{1} << 23 : int64_t{15} << 20) : int64_t{1} << (gated ? 22 : 21);
}
// Chaining words a tiling chosen that way may need (smaller tiles need more than the ladder's): far below what
// any caller's scratch is limited to.
constexpr int64_t kModelWordBytes = int64_t{4} << 20;

// Fills the zero fields of `c`.  `align` is the common alignment in bytes of all
// tensors of the call.
//
// From sweeps over bs 1..64, seq 256..16384, d 256..4096 per storage type and kernel
// family (every shape against 8-11 configurations): for lengths and widths that tiles divide,
// the largest tile that still leaves one tile per CU wins.  Large tiles mean few chunks per
// sequence (a short chain) and long uninterrupted streams per wave; 16 waves of 32
// (backward 16) timesteps with 4 bytes per lane is the largest that fits the register
// file.  So the choice walks down a ladder of tile sizes, each half the one before, and
// takes the first with at least one tile per CU; which of time, channels per lane and waves
// is halved at each rung is what the sweeps decided.  Odd and line-sharing widths, ragged lengths and the gated
// kernels differ from that; each such rung says by how much.  Forwards that leave the device idle are
// weighed by forward_ns, whatever the ladder says.
inline void complete_config(fss_config &c, int64_t bs, int64_t seq, int64_t d, int dtype, int dir,
                     size_t align, bool gated = false) {
  const bool narrow = dtype != FSS_F32;  // 16-bit storage
  const int esize = narrow ? 2 : 4;
  // two channels per lane: even d, 2-element alignment, and never pad a row to twice its width
  const bool can2 = d % 2 == 0 && align % (2 * static_cast<size_t>(esize)) == 0 &&
                    ceil_div(d, 128) * 128 < 2 * ceil_div(d, 64) * 64;
  // The rungs marked `open`, and the estimate at the end, choose a tiling as a whole: with numbers of waves or of tiles per
  // row that a caller's two column tiles do not divide, or lanes that a caller's steps do not fit.  Where the caller
  // names any part of the tiling, the ladder is the one without them.
  const bool open = !c.vec && !c.steps && !c.waves && !c.cols;
  // fp32, very large tensors with wide rows (56 shapes of 2^24..2^27 elements, d 512..4096, seq
  // 512..8192, six configurations each).  Forward from 2^26 elements: 16 steps per lane are 2-6 %
  // faster than 32 up to seq 4096, and 8 bytes per lane another 3-8 % at seq 512 (4-9 % slower
  // from seq 2048).  Backward: 8 bytes per lane with 8 steps are 4-11 % faster from 2^27 elements
  // and 3-10 % slower at 2^26.
  const int64_t elems = bs * seq * d;
  const bool big32 = !narrow && !gated && d >= 512 && elems >= (static_cast<int64_t>(1) << 26);
  const bool wide32_fwd = big32 && can2 && seq <= 512;
  const bool wide32_bwd = big32 && can2 && elems >= (static_cast<int64_t>(1) << 27);
  // Rows of three 64-channel tiles, in large launches: with two channels per lane a quarter of the lanes idles.
  // One launch behind the other, backward (6, 40000, 192) 106 -> 92 us, (30, 2000, 192) 29.3 -> 27.7; ten of eleven shapes 2 to
  // 13 % faster, (8, 40000, 192) 120 -> 123.  Forward, 8 waves, from 2^24 elements (below them nothing): (4, 57534, 192) 71 ->
  // 61, (7, 30000, 192) 61.8 -> 55.5, (30, 13002, 192) 97 -> 88, (11, 56047, 192) 151 -> 138; of 17 shapes from 45 Mi to 2^27
  // elements, 7 % in the mean, the slowest is (8, 42392, 192), 88.4 -> 88.8; (8, 40000, 192) 80.6 -> 84.1.  Not where 16 waves cover the
  // sequence in one chunk and 8 do not: (591, 268, 192) 44.6 and 55.5, (878, 284, 192) 71 and 79.  The forward's words,
  // a third and more above those with two channels, have to stay within the scratch of the entry point that allocates
  // nothing.  Other widths with idle lanes: 320 channels and 448 gain up to 5 % in the backward and lose as much as
  // they gain in the forward; rows below 192 that share sectors are a case of their own (160: 114 -> 121 us backward).
  const bool three_tiles = open && narrow && !gated && d == 3 * 64;
  Rung ladder[8];
  int n = 0;
  auto rung = [&](int v, int s, int w, int64_t need = kCus) { ladder[n++] = Rung{v, s, w, need}; };
  const bool fwd = dir == FSS_FWD;
  if (!gated && fwd) {
    if (three_tiles && elems >= (int64_t{1} << 24) && (seq <= 256 || seq > 512) &&
        bs * 3 * ceil_div(seq, 256) * 3 * 64 * static_cast<int64_t>(sizeof(uint64_t)) + static_cast<int64_t>(kHeaderBytes) <= FSS_NOALLOC_SCRATCH_BYTES)
      rung(1, 32, 8);
    if (narrow) rung(2, 32, 16);
    // (one channel per lane, where two do not go, and sequences that 512-step chunks pad a quarter further than 128-step ones:
    // (24, 384, 1735) 23.2 -> 19.2 us, (29, 574, 1319) 44.4 -> 33.6, (28, 748, 445) 15.8 -> 13.7; 15 shapes above 15 Mi
    // elements 8 % faster in the mean, the slowest (21, 277, 3669) 36.9 -> 37.9.  Where less padding goes, and where one chunk
    // of 256 steps covers the sequence, the smaller tiles lose 2 % in the mean: (36, 393, 1921) 43.5 -> 48.6, (35, 169, 2995)
    // 25.9 -> 30.6.  Up to 64 steps, at any size, half the steps and twice the waves are 9 % faster in the mean of 19 shapes,
    // (208, 59, 97) 6.9 -> 5.0, (122, 44, 1043) 10.3 -> 9.5, the slowest (2675, 20, 113) 11.5 -> 12.8); their words, twice to four times as many, well within the scratch of the entry point that
    // allocates nothing
    const int64_t reach = ceil_div(seq, 128), short_tiles = bs * ceil_div(d, 64) * reach;
    if (open && narrow && !can2 && (seq <= 64 || (seq > 256 && seq <= 1024 && reach * 128 * 5 <= ceil_div(seq, 512) * 512 * 4)) &&
        short_tiles * 3 * 64 * static_cast<int64_t>(sizeof(uint64_t)) <= FSS_NOALLOC_SCRATCH_BYTES / 2)
      rung(1, 16, 8);
    if (wide32_fwd) rung(2, 16, 16);
    else if (big32 && seq <= 4096) rung(1, 16, 16);
    rung(1, 32, 16);
    if (seq <= 2048) rung(1, 16, 16);
    rung(1, 32, 8, 0);
  } else if (!gated) {
    // 32-step slices would cost the backward a dozen spilled registers per lane
    if (narrow) {
      // (one channel per lane, where two do not go, in very large launches: (7, 4958, 3767) 8 waves 370 us, 16 waves
      // 300; (4, 8354, 1531) 142 and 122; of 2^24 elements, (31, 607, 1041), 45 and 53.  Not where 256-step chunks pad the
      // sequence a fifth further than 128-step ones: (28, 525, 2681) 108 and 117, (57, 261, 2529) 111 and 131; 16 shapes of 513 to
      // 640 steps the same in the mean, but 30 of 769 to 896, a seventh further, 3 % faster, (40, 870, 3567) 338 and 292, the slowest
      // (133, 769, 385) 111 and 117.  Nor in narrow rows: 65 to 87 channels 3 % slower in the mean of 16 shapes, (212, 2488, 67) 130 and 148,
      // (75, 11521, 71) 229 and 240, and below 64 no faster (64, whose lanes are all busy, 3 % in the mean
      // of 13, (2721, 214, 64) 83 and 71, the slowest (433, 1391, 64) by 7 %); from 93 to 191, 7 % faster in the mean of 28, the slowest (252, 4063,
      // 97) 279 and 284; 82 wider ones 10 %.  8 of them cover 65 to 128 steps: 8 steps and 8 waves take 17 % longer there in the
      // mean of 29 shapes, (512, 66, 3475) 431 and 285, the least (190, 128, 2633) 160 and 160; for fewer steps they are 3 % faster)
      const int64_t of128 = ceil_div(seq, 128) * 128, of192 = ceil_div(seq, 192) * 192, of256 = ceil_div(seq, 256) * 256;
      if (open && !can2 && (d >= 88 || d == 64) && elems >= (static_cast<int64_t>(1) << 25) && seq > 64 && (seq <= 128 || of256 * 7 <= of128 * 8))
        rung(1, 16, 16);
      if (three_tiles && elems >= (static_cast<int64_t>(1) << 23)) rung(1, 16, 16);
      // (rows that share sectors, in very large launches: with 12 waves what is in flight leaves the L2 room to put the seams
      // between column tiles together.  So not for rows of one tile, which have no seam: (48, 17050, 82) 162 -> 175 us, 23 shapes 2 %
      // slower in the mean, but where 192-step chunks pad the sequence a quarter less, (3249, 269, 112) 259 -> 217.  One launch
      // behind the other, (27, 8422, 210) 140 -> 111, (54, 5718, 146) 147 -> 114, (26, 3001, 526) 110
      // -> 100, (13, 2846, 1194) 115 -> 104; some 290 shapes of 2^25 to 2^27 elements that the lines below leave in are 5 % faster in
      // the mean: 84 of 257 to 1023 steps 6 %, the slowest (24, 956, 2034) 105 -> 107; 99 of up to 16383 4 %, the slowest (106,
      // 1942, 246) 112 -> 121; 93 longer ones 4 %, (14, 54771, 174) 448 -> 319, the slowest (4, 25461, 382) 94 -> 101.  Fewer than 97
      // steps are covered by fewer waves, 6 for 12: 49 to 64 by 6 8 % faster than by 4, (420, 51, 3588) 172 -> 158; 97 to 128 by 12
      // 11 % faster than by 8, (1362, 124, 692) 324 -> 226, the slowest (953, 98, 624) 119 -> 121; 65 to 96 by 6 3 % slower than
      // by 8, and fewer than 49 the same.  Left out as well: where 192-step chunks pad the sequence a tenth further, (43, 235,
      // 3380) 79 -> 92, (232, 406, 364) 79 -> 90 - but 449 to 512 steps, whose third chunk is a third full and more, 3 % faster in the
      // mean of 13, (340, 457, 222) 98 -> 87, the slowest (127, 456, 1948) by 3 % - or as far with a last one that is nearly
      // empty, (54, 608, 2168) 160 -> 167; and from 16384 steps on rows of up to 144 channels, 10 shapes 4 % slower, (14, 51817, 144) 252 -> 264.  Below 2^25 elements, (8,
      // 16359, 232), 73.6 -> 77.3)
      if (open && can2 && shares_sectors(d * esize) && (d > 128 || of192 * 4 <= of256 * 3) && elems >= (static_cast<int64_t>(1) << 25) &&
          (seq > 96 || (seq > 48 && seq <= 64)) && (seq < 16384 || d > 144) &&
          ((seq > 448 && seq <= 512) || (of192 * 10 <= of256 * 11 && (of192 < of256 || seq > 640))))
        rung(2, 16, 12);
      rung(2, 16, 16);
      if (seq >= 16384) rung(1, 16, 16); else rung(2, 16, 8);
      if (seq > 256) rung(1, 16, 8); else rung(2, 8, 8);
    } else {
      if (wide32_bwd) rung(2, 8, 16);
      rung(1, 16, 16);
      rung(1, 16, 8);
    }
    if (seq >= 2048) rung(1, 16, 8, 0); else rung(1, 8, 8, 0);
  } else if (fwd) {
    // The gated kernels spend as much time on arithmetic as on memory and like more, smaller
    // waves; a sequence that 8 waves cover wants two workgroups per CU before it takes them.
    // (below: where the estimate starts from)  Not a launch of the limit's size itself that the ladder's tile covers in one
    // round, as powers of two do: 16-bit, two channels, (16, 2048, 256) 13.9 us and 14.5 with 8 waves, (32, 256, 1024) 12.3
    // and 13.5; one channel from 4096 steps, (8, 4096, 256) 14.6 and 16.3, (1, 32768, 256) 16.4 and 23.9; fp32 (8, 2048, 256)
    // 11.5 and 14.6 with 12.  42 shapes in 16 bits 8 % faster in the mean, 27 in fp32 of more than 512 steps 15 %; the slowest is
    // (1, 2048, 4096) in 16 bits, 14.7 -> 15.8
    const int64_t ones = bs * ceil_div(d, 64), twos = bs * ceil_div(d, 128), big = (narrow ? twos : ones) * ceil_div(seq, 512);
    const int64_t round = !narrow ? ones * ceil_div(seq, 256) : seq >= 4096 ? ones * ceil_div(seq, 512) : can2 ? twos * ceil_div(seq, 256) : 0;
    const bool filled = open && elems >= forward_model_elems(narrow, gated) && round != kCus;
    const bool twelve = ceil_div(seq, 192) * 192 * 10 <= ceil_div(seq, 128) * 128 * 11;
    if (narrow && filled && !can2) {
      // one channel per lane (odd widths, or rows that two would pad too far): 16 steps and 12 waves, two workgroups on a
      // compute unit, whatever the length, or 8 waves and three, where 12 pad the sequence by a tenth more.  One launch behind
      // the other, 32 steps and 16 waves / 16 steps and 8 / 16 steps and 12: (11, 7957, 369) 96.6, 106.6 and 77.1 us; (13, 6000,
      // 749) 154.7, 197.8, 127.0; (5, 25000, 383) 143.1, 165.7, 112.5; (18, 7063, 287) 112, 86.6, 85.8; (23, 1901, 985) 121,
      // 98.1, 92.4.  8 waves lose most where the column tiles are a multiple of three, as the launch's 768 workgroups are; of 34
      // shapes 12 are 10 % faster than 8 in the mean, the slowest (83, 1166, 405) 97.5 -> 104.8.
      rung(1, 16, twelve ? 12 : 8, 0);
    } else if (narrow && filled) {
      // the largest tile where there is just one for every compute unit: (4, 2048, 2048) one launch behind the other
      // 23.0 us, 16 steps and 8 waves 27.2 (from 8192 steps two 8-wave workgroups are 3-5 % faster than one of 16: 8 shapes of 9).
      // 16 shapes of 252 to 256 such tiles are 2 % faster with them in the mean, the slowest (16, 721, 968) 18.9 -> 22.0; 23 of
      // 225 to 251 1 % slower; 5 of 260, (1, 5120, 3328) among them, 28.7 and 38.9
      if (seq > 256 && seq < 8192 && big <= kCus && big * 50 >= kCus * 49) rung(2, 32, 16, 0);
      // and in many rounds of rows that share sectors, where one covers the sequence and pads it by less than a third: (129, 410,
      // 3944) 345 -> 311 us, (256, 400, 1182) 211 -> 195; 14 shapes 7 % faster in the mean, the slowest (89, 478, 3226) 209 -> 210.
      // Of 7 to 8.5 rounds, or padding it further, (230, 404, 1134) 173 and 176, (116, 455, 1948) 163 and 162, (123, 265, 3048)
      // 162 and 180; of fewer, (47, 436, 1536) 45 and 56; of narrow rows, (2429, 416, 86) 152 and 181.
      if (shares_sectors(d * esize) && d >= 1024 && seq > 384 && seq <= 512 && big * 2 >= 17 * kCus) rung(2, 32, 16, 0);
      // the same as with one channel per lane, for sequences of few chunks ((9, 1695, 1792) 42.6 -> 37.5 us against 32 steps and
      // 16 waves, (34, 1201, 776) 64.9 -> 55.6, (26, 859, 1548) 61 -> 51); half as long where that pads the sequence by a
      // tenth less ((29, 299, 1680) 34.4 -> 20.7)
      if (seq <= 2048) rung(2, 16, ceil_div(seq, 64) * 64 * 10 <= ceil_div(seq, 128) * 128 * 9 ? 4 : 8);
      // (longer chains want longer chunks, (8, 3000, 1024) 16 steps 35.2 us, 32 steps 29.9, where three quarters of the device's
      // 8-wave workgroups have a tile; one channel per lane never: (1, 8379, 1740) 47.7 us, two channels 23.7)
      if (seq > 2048 && seq < 8192) rung(2, 32, 16);
      if (seq > 2048) rung(2, 32, 8, kCus * 3 / 2);
      rung(2, 16, 8, 0);
    } else if (narrow) {
      if (seq >= 8192) rung(2, 32, 8, 2 * kCus);
      if (seq > 256) rung(2, 32, 16); else rung(2, 32, 8, 2 * kCus);
      if (seq >= 4096) rung(1, 32, 16); else rung(2, 16, 16);
      if (seq >= 16384) rung(1, 32, 8);
      rung(1, 16, 16);
      if (seq >= 1024) rung(1, 16, 8, 0); else rung(1, 16, 16, 0);
    } else {
      // fp32: the largest tile where its rounds are whole ((8, 4096, 1024) 32 steps and 16 waves 83 us, 16 steps 86),
      // elsewhere 16 steps and 12 waves ((10, 24028, 128) 87 -> 78, (11, 1623, 1152) 62 -> 51, (9, 7795, 67) 33 -> 24),
      // or 8 waves where 12 pad the sequence by a tenth more ((34, 214, 664) 17.2 -> 17.1, with 12 21.0).  What a sequence of up to
      // 512 steps gains by those 8 hangs on the steps of the last wave of the larger tile, which all the others wait for: 16 to
      // 31 of 32, 30 % in the mean of 88 shapes, (237, 59, 704) 43.3 -> 29.5, the slowest (186, 80, 3063) 168 -> 192.  Fewer or
      // all 32, nothing in the mean of 81; above 64 steps, in rows of whole sectors, a loss of 3 % in the mean of 48, (60, 78, 1024)
      // 16.1 -> 23.3, (142, 386, 1088) 134 -> 155: there the ladder keeps its tile, at a loss of at most 9 % ((149, 206, 896) 77.5
      // -> 84.9).
      // Not 12 waves where just a few of their tiles go into a second round, in a launch that the largest tile does not fill: (7, 5420,
      // 175) 28.4 and 31.9 us, (2, 1306, 2560) 20.8 and 22.9; 38 shapes with up to a fifth of a second round are 3 % faster
      // without in the mean, the slowest (1, 17281, 347) 25.8 -> 28.2; 16 with more of it 1 %, 12 with none 6 % slower.
      // Nor in large launches of wide rows that share sectors, (6, 12955, 2369) 493 and 580, (44, 1451, 1809) 327 and 385: 24 shapes from 80 Mi
      // elements and 1280 channels on, padded by up to a quarter, are 8 % faster with the largest tile in the mean, the slowest
      // (2, 15075, 3558) 307 -> 314.  Of 48 to 80 Mi elements they are 3 % slower (11 shapes), narrower 4 % (11), padded further 5 % (11); one
      // chunk of that tile, 410 to 512 steps, is 13 % faster to 17 % slower and the same in the mean of 14.
      // Known to be slower: with 8 waves (226, 635, 371) 203 -> 238 us, with 12 (12, 12130, 782) 323 -> 341, (40, 942, 1345) 151 -> 165; 80 shapes from
      // 4 Mi to 128 Mi elements are 13 % faster in the mean.
      const int64_t of_round = ceil_div(big, kCus) * kCus;
      const bool ladder = !twelve && seq > 64 && seq <= 512 && seq % 32 < 16 && !shares_sectors(d * esize);
      const bool spills = twelve && seq > 512 && big <= kCus && ones * ceil_div(seq, 192) > 2 * kCus && ones * ceil_div(seq, 192) * 5 <= 2 * kCus * 6;
      const bool wide = shares_sectors(d * esize) && d >= 1280 && seq > 512 && elems >= (int64_t{80} << 20) && ceil_div(seq, 512) * 512 * 4 <= seq * 5;
      if (filled && !ladder && !spills && !wide && (big * 50 < of_round * 49 || seq * 50 < ceil_div(seq, 512) * 512 * 49)) rung(1, 16, twelve ? 12 : 8, 0);
      if (seq > 256) rung(1, 32, 16); else rung(1, 32, 8, 2 * kCus);
      rung(1, 16, 16, 0);
    }
  } else {
    // gated backward: four tensors per timestep, at most 16 steps per lane (fp32: 8 are faster)
    if (narrow) {
      // (many short sequences: two 8-wave workgroups per CU are 3-16 % faster: 6 shapes of 7 at 2^25 elements)
      if (seq <= 1024) rung(2, 16, 8, 8 * kCus);
      if (seq > 256) rung(2, 16, 16); else rung(2, 16, 8, 4 * kCus);
      rung(2, 8, 16);
      rung(2, 8, 8, seq <= 256 ? 1 : kCus);
      rung(1, 8, 8, 0);
    } else {
      if (seq > 256) rung(1, 8, 16);
      rung(1, 8, 8, 0);
    }
  }
  fss_config pick = {0, 0, 0, 0, 0};
  for (int i = 0; i < n; ++i) {
    // what the caller fixed stays fixed
    int v = c.vec ? c.vec : ladder[i].vec;
    int s = c.steps ? c.steps : ladder[i].steps;
    int w = c.waves ? c.waves : ladder[i].waves;
    if (!c.vec && v == 2 && !can2) continue;
    // never more waves or steps than the sequence needs
    while (!c.waves && w > 1 && static_cast<int64_t>(s) * (w / 2) >= seq) w /= 2;
    while (!c.steps && s > 8 && s / 2 >= seq) s /= 2;
    while (!c.waves && w > max_waves(esize, v, s, !fwd, gated)) w /= 2;  // (only when the caller fixed a wide lane)
    while (!c.waves && w > 1 && lds_bytes(w, v) > kLdsBudget) --w;
    pick = fss_config{v, s, w, 0, 0};
    if (bs * ceil_div(d, 64 * static_cast<int64_t>(v)) * ceil_div(seq, static_cast<int64_t>(s) * w) >= ladder[i].need) break;
  }
  // Forward and gated backward, 16-wave workgroups (one per CU) whose last round would fill less than 90 % of the
  // CUs: the same tile shape as 8-wave workgroups, two per CU, spreads that round over all CUs
  // (7-18 % faster on 59 of 182 shapes with lengths and widths that are no powers of two; the
  // plain backward measured no gain from it, the gated backward 5-16 % on 6 shapes of 6).
  if ((fwd || gated) && !c.waves && pick.waves == 16) {
    const int64_t tiles = bs * ceil_div(d, 64 * static_cast<int64_t>(pick.vec)) * ceil_div(seq, static_cast<int64_t>(pick.steps) * 16);
    const int64_t rounds = ceil_div(tiles, kCus);
    if (rounds >= 2 && tiles * 10 < rounds * kCus * 9) pick.waves = 8;
  }
  if (fwd && open && seq > 64 && elems < forward_model_elems(narrow, gated)) {
    const ForwardCost &model = kForwardCost[narrow ? 0 : 1][gated ? 1 : 0];
    double best = forward_ns(model, bs, seq, d, esize, pick.vec, pick.steps, pick.waves) /
                  (elems < (int64_t{1} << 21) ? 1.04 : 1.08);
    constexpr Rung shapes[] = {{0, 32, 16, 0}, {0, 32, 8, 0}, {0, 16, 16, 0}, {0, 16, 12, 0}, {0, 16, 8, 0}, {0, 8, 16, 0}, {0, 8, 8, 0}};
    for (int v = can2 ? 2 : 1; v >= 1; --v)
      for (const Rung &r : shapes) {
        int s = r.steps, w = r.waves;
        if (v * s > max_vec_steps(dtype) || (gated && !narrow && v > 1)) continue;
        while (w > 1 && static_cast<int64_t>(s) * (w / 2) >= seq) w /= 2;
        while (s > 8 && s / 2 >= seq) s /= 2;
        const int64_t columns = bs * ceil_div(d, 64 * static_cast<int64_t>(v)), chunks = ceil_div(seq, static_cast<int64_t>(s) * w);
        if (columns * chunks * v * (3 * 64 * static_cast<int64_t>(sizeof(uint64_t))) > kModelWordBytes) continue;
        const double ns = forward_ns(model, bs, seq, d, esize, v, s, w);
        if (ns < best) {
          best = ns;
          pick = fss_config{v, s, w, 0, 0};
        }
      }
  }
  c.vec = pick.vec;
  c.steps = pick.steps;
  c.waves = pick.waves;
  if (!c.cols) c.cols = choose_cols(c, bs, seq, d, dtype, dir, gated);
}

struct Plan {
  fss_config cfg;
  int alt_policy = 0;  // cache_variant
  int64_t tiles_per_row, n_ctiles, n_chunks;
  int64_t n_groups;  // column groups per chunk: n_ctiles / cfg.cols
  int64_t n_tiles;   // what the workgroups walk: n_groups * n_chunks
  size_t ws_bytes;
};

inline int compute_plan(Plan &pl, int64_t bs, int64_t seq, int64_t d, int dtype, int dir, size_t align,
              const fss_config *user) {
  if (bs < 0 || seq < 0 || d < 0) return FSS_ERR_BAD_SHAPE;
  if (dtype != FSS_BF16 && dtype != FSS_F32 && dtype != FSS_F16) return FSS_ERR_BAD_CONFIG;
  if (dir < FSS_FWD || dir > FSS_GATED_BWD) return FSS_ERR_BAD_CONFIG;
  const bool gated = dir >= FSS_GATED_FWD;
  dir &= 1;
  const int esize = dtype != FSS_F32 ? 2 : 4;
  // bs*seq*d*esize must fit int64
  if (bs > 0 && seq > 0 && d > 0) {
    const __int128 total = static_cast<__int128>(bs) * seq * d * esize;
    if (total > (static_cast<__int128>(1) << 62)) return FSS_ERR_BAD_SHAPE;
  }
  fss_config c = {0, 0, 0, 0, 0};
  if (user) c = *user;
  if (c.max_groups < 0 || c.cols < 0) return FSS_ERR_BAD_CONFIG;
  const int64_t dd = d > 0 ? d : 1, ss = seq > 0 ? seq : 1, bb = bs > 0 ? bs : 1;
  complete_config(c, bb, ss, dd, dtype, dir, align, gated);
  if (!config_valid(c, dtype, gated, dir)) return FSS_ERR_BAD_CONFIG;
  if (dd % c.vec != 0) return FSS_ERR_BAD_CONFIG;
  if (align % (static_cast<size_t>(c.vec) * esize) != 0) return FSS_ERR_MISALIGNED;
  pl.cfg = c;
  pl.tiles_per_row = ceil_div(dd, 64 * c.vec);
  if (pl.tiles_per_row % c.cols != 0) return FSS_ERR_BAD_CONFIG;
  pl.n_ctiles = bb * pl.tiles_per_row;
  pl.n_chunks = ceil_div(ss, static_cast<int64_t>(c.waves / c.cols) * c.steps);
  pl.n_groups = pl.n_ctiles / c.cols;
  pl.n_tiles = pl.n_groups * pl.n_chunks;
  if (pl.n_ctiles > INT32_MAX || pl.n_chunks > INT32_MAX || pl.n_ctiles * pl.n_chunks > INT32_MAX) return FSS_ERR_BAD_SHAPE;
  pl.ws_bytes = kHeaderBytes;
  if (pl.n_chunks > 1)
    pl.ws_bytes += static_cast<size_t>(pl.n_ctiles * pl.n_chunks) * 3 * 64 * c.vec * sizeof(uint64_t);
  return FSS_OK;
}

// The same, with the plans of the shapes a thread launched last kept: what is planned is a function of these
// arguments alone, and weighing a dozen tilings takes the host 0.5 us of a launch of a few.  The alignment shifts the
// slot, so that the plans for 2 to 16 bytes, which fss_workspace_bytes asks for in turn, never replace each other.
inline int make_plan(Plan &pl, int64_t bs, int64_t seq, int64_t d, int dtype, int dir, size_t align,
                     const fss_config *user) {
  if (user) return compute_plan(pl, bs, seq, d, dtype, dir, align, user);
  struct Kept {
    int64_t bs = -1, seq = 0, d = 0;
    int dtype = 0, dir = 0;
    size_t align = 0;
    Plan plan;
  };
  constexpr uint32_t kKept = 16;
  static thread_local Kept kept[kKept];
  const uint64_t mix = (static_cast<uint64_t>(bs) * 0x9e3779b97f4a7c15ull ^ static_cast<uint64_t>(seq)) * 0xff51afd7ed558ccdull ^
                       (static_cast<uint64_t>(d) * 8 + static_cast<uint64_t>(dtype * 4 + dir)) * 0xc4ceb9fe1a85ec53ull;
  Kept &k = kept[((mix >> 43) + kKept / 4 * static_cast<uint32_t>(__builtin_ctzll(align))) % kKept];
  if (k.bs == bs && k.seq == seq && k.d == d && k.dtype == dtype && k.dir == dir && k.align == align && bs >= 0) {
    pl = k.plan;
    return FSS_OK;
  }
  const int rc = compute_plan(pl, bs, seq, d, dtype, dir, align, nullptr);
  ++tls_plans_computed;
  if (rc == FSS_OK) {
    k.bs = bs;
    k.seq = seq;
    k.d = d;
    k.dtype = dtype;
    k.dir = dir;
    k.align = align;
    k.plan = pl;
  }
  return rc;
}

// Which cache hints a launch carries (ALT of scan_kernel).  The instantiations without hints exist for up to two
// channels per lane, which is what the library chooses; wider ones are only named by a caller and keep
// to the sizes.
inline int cache_variant(const Plan &pl, int64_t bs, int64_t seq, int64_t d, int64_t esize, bool gated, int dir, bool streaming) {
  if (pl.cfg.vec <= 2 && shares_sectors(d * esize)) return 3;
  if (gated) return 0;
  // (variant 2 exists for the kernels large shapes run - the forward with 32 steps per lane, the
  // backward with 16 steps and 4 bytes per lane; elsewhere the forward runs as 0, the backward as 1)
  const int64_t tensor_bytes = bs * seq * d * esize;
  const bool large = streaming || tensor_bytes > kStreamDoutBytes;
  if (dir == FSS_FWD) return large ? 2 : (tensor_bytes <= kKeepOutBytes ? 1 : 0);
  return streaming ? 2 : (large ? 1 : 0);
}

inline size_t common_alignment(std::initializer_list<const void *> ptrs) {
  uintptr_t bits = 0;
  for (const void *p : ptrs) bits |= reinterpret_cast<uintptr_t>(p);
  bits |= 16;  // 16 bytes is all any path needs
  return static_cast<size_t>(bits & (~bits + 1));
}

inline int check_device() {
  static int cached[64];  // 0 unknown, 1 ok, 2 unsupported
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return FSS_ERR_LAUNCH;
  if (dev < 0 || dev >= 64) return FSS_OK;
  int state = __atomic_load_n(&cached[dev], __ATOMIC_RELAXED);
  if (state == 0) {
    hipDeviceProp_t prop;
    hipError_t e = hipGetDeviceProperties(&prop, dev);
    if (e != hipSuccess) {
      tls_hip_error = static_cast<int>(e);
      return FSS_ERR_LAUNCH;
    }
    state = strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? 1 : 2;
    __atomic_store_n(&cached[dev], state, __ATOMIC_RELAXED);
  }
  return state == 1 ? FSS_OK : FSS_ERR_UNSUPPORTED_DEVICE;
}

// Scans of one process never overlap on a device.  A scan's workgroups wait for each
// other and its grid is sized to fill the device, so two scans sharing the device
// could each hold the compute units the other's unscheduled workgroups need, and
// both would sit there until their waits give up.  Launches on one stream are
// ordered anyway; when the stream changes, the new launch is made to wait for
// everything queued on the previous stream.  The lock is held across the launch, so
// that the event recorded by the next caller lands behind this one's kernel.
// Streams under graph capture are left alone (a captured scan is ordered by its
// graph; do not replay two graphs holding scans concurrently).
struct ScanOrder {
  std::mutex lock;
  hipStream_t last = nullptr;
  bool any = false;
  hipEvent_t event = nullptr;
};
extern ScanOrder g_scan_order[64];

inline bool stream_is_capturing(hipStream_t s) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &status) != hipSuccess) {
    (void)hipGetLastError();
    return true;  // unknown: do not touch it
  }
  return status != hipStreamCaptureStatusNone;
}

class ScanOrderGuard {
 public:
  explicit ScanOrderGuard(hipStream_t s) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return;
    order_ = &g_scan_order[dev];
    order_->lock.lock();
    if (stream_is_capturing(s)) return;
    if (order_->any && order_->last != s && !stream_is_capturing(order_->last)) {
      if (!order_->event && hipEventCreateWithFlags(&order_->event, hipEventDisableTiming) != hipSuccess) {
        order_->event = nullptr;
        (void)hipGetLastError();
      }
      // a stream the caller has destroyed since makes the record fail: nothing to wait for then
      if (order_->event && hipEventRecord(order_->event, order_->last) == hipSuccess)
        (void)hipStreamWaitEvent(s, order_->event, 0);
      (void)hipGetLastError();
    }
    order_->last = s;
    order_->any = true;
  }
  ~ScanOrderGuard() {
    if (order_) order_->lock.unlock();
  }
  ScanOrderGuard(const ScanOrderGuard &) = delete;
  ScanOrderGuard &operator=(const ScanOrderGuard &) = delete;

 private:
  ScanOrder *order_ = nullptr;
};

inline int cu_count_of_current_device() {
  static int cached[64];  // by device; 0 = not asked yet
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  const bool slot = dev >= 0 && dev < 64;
  if (slot && (n = __atomic_load_n(&cached[dev], __ATOMIC_RELAXED)) > 0) return n;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 0;
  if (slot) __atomic_store_n(&cached[dev], n, __ATOMIC_RELAXED);
  return n;
}

// Workgroups of `kernel` that are certainly resident together on one compute unit (0 on
// error).  Deliberately not the runtime's occupancy query: the kernel's waits
// need a lower bound, and that query bounds by vector registers and LDS only.
// These kernels hold many scalar registers as well (a row pointer per load); a
// wave may be allocated 128 of the 800 a SIMD has, which caps a SIMD at 6 waves -
// the residency measured on MI355X for the scalar-heaviest variants.
template <typename Kernel>
int resident_workgroups_per_cu(Kernel kernel, int waves, size_t lds) {
  hipFuncAttributes attr;
  const hipError_t e = hipFuncGetAttributes(&attr, reinterpret_cast<const void *>(kernel));
  if (e != hipSuccess) {
    tls_hip_error = static_cast<int>(e);
    return 0;
  }
  int vgprs = attr.numRegs > 0 ? attr.numRegs : 128;
  vgprs = (vgprs + 7) / 8 * 8;                    // allocation granule
  int per_simd = 512 / vgprs;                      // 512 vector registers per lane per SIMD
  if (per_simd > 6) per_simd = 6;                  // scalar-register bound, see above
  if (per_simd < 1) return 0;
  int per_cu;
  if (waves >= 4)
    per_cu = per_simd / ((waves + 3) / 4);         // a workgroup puts ceil(waves/4) waves on a SIMD
  else
    per_cu = per_simd * (waves == 1 ? 4 : waves == 2 ? 2 : 1);
  const size_t lds_alloc = (lds + attr.sharedSizeBytes + 1023) / 1024 * 1024;
  const int by_lds = static_cast<int>((160 * 1024) / (lds_alloc ? lds_alloc : 1024));
  if (per_cu > by_lds) per_cu = by_lds;
  if (per_cu > 32) per_cu = 32;
  return per_cu;
}

// The same for the whole current device.  `cache` (one slot per waves-per-workgroup value
// of one kernel instantiation) keeps the per-CU answer, which is a property of the code
// object; the CU count is the current device's.
template <typename Kernel>
int resident_workgroups(Kernel kernel, int waves, size_t lds, int *cache) {
  int per_cu = __atomic_load_n(&cache[waves], __ATOMIC_RELAXED);
  if (per_cu == 0) {
    per_cu = resident_workgroups_per_cu(kernel, waves, lds);
    if (per_cu <= 0) return 0;
    __atomic_store_n(&cache[waves], per_cu, __ATOMIC_RELAXED);
  }
  return per_cu * cu_count_of_current_device();
}

// ---- channel-major planning -------------------------------------------------------------

// rows per wave: 4 bytes-per-lane budgets as in the row-major kernels (two tensors of
// 8 rows x 16 bytes forward, three of 4 rows backward)
constexpr int kCmRowsFwd = 8, kCmRowsBwd = 4;

struct CmPlan {
  int vec, waves;
  int row_lanes_log2;  // below 6: several rows share a wave's vectors (rows of at most 32 lanes)
  int64_t n_rowtiles, n_chunks, n_tiles;
  size_t ws_bytes;
};

inline int make_cm_plan(CmPlan &pl, int64_t rows, int64_t seq, int dtype, int dir, size_t align, const fss_config *user) {
  if (rows < 0 || seq < 0) return FSS_ERR_BAD_SHAPE;
  if (dtype != FSS_BF16 && dtype != FSS_F32 && dtype != FSS_F16) return FSS_ERR_BAD_CONFIG;
  if (dir != FSS_FWD && dir != FSS_BWD) return FSS_ERR_BAD_CONFIG;
  const int esize = dtype != FSS_F32 ? 2 : 4;
  const int64_t rr = rows > 0 ? rows : 1, ss = seq > 0 ? seq : 1;
  if (static_cast<__int128>(rr) * ss * esize > (static_cast<__int128>(1) << 62)) return FSS_ERR_BAD_SHAPE;
  const int widest = 16 / esize;  // 16 bytes per lane and load
  int vec = user ? user->vec : 0, waves = user ? user->waves : 0;
  if (user && (user->max_groups < 0 || user->steps != 0)) return FSS_ERR_BAD_CONFIG;
  // 16 bytes per lane whatever the rows' length and alignment, from the length that fills one lane on
  // (a configuration that names the vector width keeps to naturally aligned accesses).  Below it two
  // 16-bit steps per lane where rows and tensors allow: bf16 forward (64, 4096, 6) 51.9 us with one, 48.9 with
  // two, (64, 4096, 4) 50.2 and 49.3.
  const bool any_rows = vec == 0;
  const bool pairs = esize == 2 && ss % 2 == 0 && align % 4 == 0;
  if (any_rows) vec = ss >= widest ? widest : pairs ? 2 : 1;
  const bool vec_ok = vec == 1 || vec == widest || (vec == 2 && esize == 2);
  if (!vec_ok) return FSS_ERR_BAD_CONFIG;
  if (!any_rows && ss % vec != 0) return FSS_ERR_BAD_CONFIG;
  if (!any_rows && align % (static_cast<size_t>(vec) * esize) != 0) return FSS_ERR_MISALIGNED;
  if (waves == 0) {
    const int64_t w = ceil_div(ss, static_cast<int64_t>(64) * vec);
    waves = static_cast<int>(w < 8 ? w : 8);
    // forward, a chained sequence with few rows: half-size workgroups double the tiles in
    // flight (10-15 % at bs1 d256 seq16384)
    const int64_t chunks8 = ceil_div(ss, static_cast<int64_t>(8) * 64 * vec);
    if (dir == FSS_FWD && waves == 8 && chunks8 >= 2 && ceil_div(rr, kCmRowsFwd) * chunks8 < 1024) waves = 4;
    // a chained sequence that half-size workgroups cover with less padding (seq 5120: three
    // chunks of 2048 steps instead of two of 4096; 7-9 % faster)
    const int64_t reach4 = static_cast<int64_t>(4) * 64 * vec;
    if (waves == 8 && chunks8 >= 2 && ceil_div(ss, reach4) * reach4 < chunks8 * 2 * reach4) waves = 4;
  }
  if (waves < 1 || waves > 16) return FSS_ERR_BAD_CONFIG;
  pl.vec = vec;
  pl.waves = waves;
  // rows of at most half a wave share its vectors (SHORT in fss_scan_cm.hip: faster from one row to
  // a million, 1.1 times where a row takes 32 lanes, 8 times where it takes four); shorter than one lane's
  // 16 bytes they keep the one-step kernels
  pl.row_lanes_log2 = 6;
  if (any_rows && vec == widest && waves == 1)
    for (int l = 5; l >= 0 && ss <= (static_cast<int64_t>(vec) << l); --l) pl.row_lanes_log2 = l;
  const int vectors = dir == FSS_BWD || pl.row_lanes_log2 < 6 ? kCmRowsBwd : kCmRowsFwd;
  pl.n_rowtiles = ceil_div(rr, static_cast<int64_t>(vectors) << (6 - pl.row_lanes_log2));
  pl.n_chunks = ceil_div(ss, static_cast<int64_t>(waves) * 64 * vec);
  pl.n_tiles = pl.n_rowtiles * pl.n_chunks;
  if (pl.n_rowtiles > INT32_MAX || pl.n_chunks > INT32_MAX || pl.n_tiles > INT32_MAX) return FSS_ERR_BAD_SHAPE;
  pl.ws_bytes = kHeaderBytes;
  if (pl.n_chunks > 1) pl.ws_bytes += static_cast<size_t>(pl.n_tiles) * 3 * 64 * sizeof(uint64_t);
  return FSS_OK;
}


// ---- what each translation unit provides --------------------------------------------------

// fss_scan_rm.hip, compiled once per storage type and direction: launches the row-major
// kernel (plain, with states, or gated) the plan asks for.
#define FSS_DECLARE_RM_LAUNCH(name)                                                                        \
  int name(const ScanArgs &args, const StateArgs<true> &state, const Plan &pl, bool gated, bool with_state, \
           hipStream_t stream)
FSS_DECLARE_RM_LAUNCH(launch_rm_bf16_fwd);
FSS_DECLARE_RM_LAUNCH(launch_rm_bf16_bwd);
FSS_DECLARE_RM_LAUNCH(launch_rm_f16_fwd);
FSS_DECLARE_RM_LAUNCH(launch_rm_f16_bwd);
FSS_DECLARE_RM_LAUNCH(launch_rm_f32_fwd);
FSS_DECLARE_RM_LAUNCH(launch_rm_f32_bwd);
#undef FSS_DECLARE_RM_LAUNCH

// fss_scan_cm.hip
int run_cm_scan(int dtype, int dir, const void *alpha, const void *in_b, const void *in_h, void *out0, void *out1,
                int64_t bs, int64_t d, int64_t seq, void *workspace, size_t workspace_bytes, void *stream,
                const fss_config *cfg);

}  // namespace fss
