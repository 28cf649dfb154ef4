// Channel-major (bs, d, seq) scan kernels and their host side.
#include "fss_device.h"
#include "fss_host.h"

namespace fss {

// ---- channel-major layout: (bs, d, seq), time contiguous ---------------------------
//
// Every (batch, channel) pair is a contiguous row of seq elements, so time runs
// across the lanes: a lane holds VEC consecutive timesteps of ROWS rows (one 16-byte
// load per row and tensor at full width), a wave 64*VEC consecutive timesteps of
// those rows, the waves of a workgroup consecutive slices of the same rows.  A lane
// folds its VEC steps into an affine map, a shuffle scan over the 64 lanes turns
// the maps into prefixes, and the last lane's prefix is the wave's map.  From
// there on the rows of a tile play the part the channels play in the row-major
// kernels: lane r carries row r's map into the same chain phase (other lanes carry
// identity maps), and gets back the state entering the wave's slice, which every
// lane then pushes through its own exclusive prefix before re-running its VEC steps.
// With 8 waves of 512 timesteps a workgroup covers 4096 timesteps, so sequences up
// to that length never touch the workspace.
//
// The backward runs over reversed time with lanes in scan order: lane l of slice k
// holds scan positions (k*64 + l)*VEC .. +VEC-1, i.e. timesteps descending from
// seq-1-(k*64+l)*VEC, and takes alpha[t+1] / h[t-1] of its first / last step from
// the neighbouring lane (or, at a slice edge, from a one-element load).
//
// Rows need no alignment beyond an element's and no length that is a multiple of VEC: global
// accesses work at any address (DwordIO), and the one lane per row whose vector would reach past
// the end of the scan loads one that ends there and shifts it.  Kernels with one timestep per
// lane for such rows (128 bytes per wave and load, chunks of 512 steps instead of 4096) took three
// times as long: bf16 forward and backward of (8, 1024, 2047) 158 -> 53.4 us (2048: 48.5), of
// (8, 1024, 4095) 349 -> 119 us (4096: 107), of (1, 256, 65521) 186 -> 61 us.  What is left between
// odd and aligned rows is the price of 16-byte accesses at odd addresses; keeping the stores'
// lines in L2 for the neighbouring wave (no streaming hint) costs another 3-5 %.

__device__ __forceinline__ float lane_read(float v, int lane) {
  return as_f32(__builtin_amdgcn_readlane(as_u32(v), lane));
}

template <bool B>
struct Flag {
  static constexpr bool value = B;
};

// RAGGED: seq is no multiple of VEC (a kernel of its own: the shifts cost the forward four spilled
// registers, 2 % of the time of rows that need none).
// SHORT: rows that half a wave's lanes cover.  They lie back to back in memory, so 64/L of them share a
// vector - L lanes each, a power of two, with the lane scan confined to them - instead of leaving
// most lanes idle: a wave's load then is as long as other waves' are, and the kernel is bound by memory
// again.  bf16, one row to a wave -> shared: (64, 4096, 64) forward 62 -> 16.7 us, backward 84 -> 28.8 (5.8
// TB/s); (64, 1024, 250) 29.4 -> 17.6 and 40.2 -> 30.7 us; (2, 1024, 256) 6.4 -> 4.4 and 5.7 -> 5.0; (64, 4096,
// 23), before with one step per lane, 52 -> 11.6 and 63 -> 19.1.
template <typename E, int VEC, int ROWS, bool BWD, bool RAGGED, bool SHORT, bool CHAINED>
__device__ __forceinline__ void cm_tile(const ScanArgs &p, TileCtx &c, int64_t row0, int64_t n_rows) {
  using RowT = Row<E, VEC>;
  using OneT = Row<E, 1>;
  const int64_t seq = c.seq;
  // lanes of a row, this lane's place among them, and the row's place among those that share the vector
  const int lanes = SHORT ? 1 << p.row_lanes_log2 : 64;
  const int lane = SHORT ? c.lane & (lanes - 1) : c.lane;
  const int row_of_lane = SHORT ? c.lane >> p.row_lanes_log2 : 0;
  const int rows_per_vector = SHORT ? 64 >> p.row_lanes_log2 : 1;
  const int64_t slice = static_cast<int64_t>(c.chunk) * c.n_waves + c.wave;
  const int64_t r_base = (slice * 64 + lane) * VEC;             // first scan position of this lane
  const bool in_seq = r_base < seq;
  // The last lane of the scan may hold fewer than VEC steps (backward: the missing ones are the low end
  // of its vector, timesteps below 0).  It loads the VEC timesteps that end (backward: start) with the
  // sequence and moves them to their places, so that no lane reads outside its row and no load waits.
  const bool ragged = RAGGED && (SHORT || (slice * 64 * VEC < seq && seq < (slice + 1) * 64 * VEC));  // in this slice
  const int missing = ragged && in_seq && seq - r_base < VEC ? VEC - static_cast<int>(seq - r_base) : 0;
  const int64_t t_lo = BWD ? seq - r_base - VEC : r_base;       // lowest timestep of the vector
  const int64_t t_hi = t_lo + VEC - 1;
  // wave-uniform base (the lowest timestep any lane of the slice holds) + a 32-bit lane offset
  const int64_t t_base = BWD ? seq - (slice * 64 + lanes) * VEC : slice * 64 * VEC;
  const uint32_t lane_off = static_cast<uint32_t>((BWD ? lanes - 1 - lane : lane) * RowT::kBytes) +
                            (SHORT ? static_cast<uint32_t>(row_of_lane) * static_cast<uint32_t>(seq) * E::kBytes : 0u);

  RowT a[ROWS], b[ROWS], hp[BWD ? ROWS : 1];
  float edge_a[BWD ? ROWS : 1], edge_h[BWD ? ROWS : 1];
  bool ok[ROWS];
  constexpr int kBack = BWD || !RAGGED ? 0 : VEC * E::kBytes;  // (lane offsets are unsigned: the base makes room)
  const uint32_t load_off = lane_off + kBack + (BWD ? missing : -missing) * E::kBytes;
  auto load_vector = [&](RowT &v, const char *tensor, int64_t off, auto nt) {
    v.template load<decltype(nt)::value>(uniform_ptr((gcptr_t)tensor + off - kBack) + load_off);
  };
  auto place = [&](RowT &v) {
    if (BWD)
      v.shift_up(missing);
    else
      v.shift_down(missing);
  };
  auto store_vector = [&](const RowT &v, char *tensor, int64_t off, auto nt) {
    const gptr_t base = uniform_ptr((gptr_t)tensor + off) + lane_off;
    if (missing == 0)
      v.template store<decltype(nt)::value>(base);
    else
      v.store_some(base, BWD ? missing : 0, BWD ? VEC : VEC - missing);
  };

  // ---- phase 1a: loads ---------------------------------------------------------------
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int64_t row = row0 + r * rows_per_vector;
    ok[r] = in_seq && row + row_of_lane < n_rows;
    a[r].fill(1.0f);  // outside: identity steps
    b[r].fill(0.0f);
    if (ok[r]) {
      const int64_t off = (row * seq + t_base) * E::kBytes;
      load_vector(a[r], p.in_a, off, Flag<(BWD ? kNtABwd : kNtAFwd)>());
      load_vector(b[r], p.in_b, off, Flag<(BWD ? kNtBBwd : kNtBFwd)>());
    }
  }
  if (ragged) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      place(a[r]);
      place(b[r]);
    }
  }
  if (BWD) {
    // alpha[t_hi+1] for the first step: from the neighbouring lane, except at the end of
    // the wave's slice
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      OneT ea;
      ea.fill(0.0f);
      if (!SHORT && lane == 0 && ok[r] && t_hi + 1 < seq) ea.load((gcptr_t)p.in_a + ((row0 + r) * seq + t_hi + 1) * E::kBytes);
      const float from_prev = __shfl_up(a[r].get(0), 1);  // lane-1 holds timesteps just above ours
      edge_a[r] = lane == 0 ? ea.get(0) : from_prev;
    }
  }
  // The saved h only feeds phase 3: its loads go out inside the chain phase, behind the
  // look-back's, and travel while the chain is resolved.
  OneT eh[BWD ? ROWS : 1];
  auto load_h = [&] {
    if (BWD) {
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        eh[r].fill(0.0f);
        hp[r].fill(0.0f);
        if (ok[r]) {
          const int64_t off = ((row0 + r * rows_per_vector) * seq + t_base) * E::kBytes;
          load_vector(hp[r], p.in_h, off, Flag<kNtH>());
        }
        if (!SHORT && lane == 63 && ok[r] && t_lo >= 1) eh[r].load((gcptr_t)p.in_h + ((row0 + r) * seq + t_lo - 1) * E::kBytes);
      }
    }
  };

  // coefficient, addend and saved h of scan step j of row r
  auto coef = [&](int r, int j) -> float {
    if (BWD) return j == 0 ? edge_a[BWD ? r : 0] : a[r].get(VEC - j);
    return a[r].get(j);
  };
  auto addend = [&](int r, int j) -> float { return b[r].get(BWD ? VEC - 1 - j : j); };
  auto h_prev = [&](int r, int j) -> float {
    return j == VEC - 1 ? edge_h[BWD ? r : 0] : hp[BWD ? r : 0].get(VEC - 2 - j > 0 ? VEC - 2 - j : 0);
  };
  // the scan's first step has no predecessor, whatever alpha holds there
  const bool first_lane = slice == 0 && lane == 0;

  // ---- phase 1b: lane maps, then inclusive prefixes over the lanes --------------------
  float A[ROWS], B[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    A[r] = 1.0f;
    B[r] = 0.0f;
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const float av = (j == 0 && first_lane) ? 0.0f : coef(r, j);
      B[r] = __builtin_fmaf(av, B[r], addend(r, j));
      A[r] *= av;
    }
  }
#pragma unroll
  for (int off = 1; off < (SHORT ? 32 : 64); off <<= 1) {
    if (SHORT && off >= lanes) break;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const float pa = __shfl_up(A[r], off), pb = __shfl_up(B[r], off);
      if (lane >= off) {
        B[r] = fma0(A[r], pb, B[r]);
        A[r] *= pa;
      }
    }
  }
  // lane r takes row r's wave map into the chain phase; the other lanes identity maps
  float mA = 1.0f, mB = 0.0f;
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const float wa = lane_read(A[r], 63), wb = lane_read(B[r], 63);
    if (lane == r) {
      mA = wa;
      mB = wb;
    }
  }
  // exclusive prefixes: what the lanes before this one do to the slice's incoming state
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const float pa = __shfl_up(A[r], 1), pb = __shfl_up(B[r], 1);
    A[r] = lane == 0 ? 1.0f : pa;
    B[r] = lane == 0 ? 0.0f : pb;
  }

  float slice_in = 0.0f;
  if (!SHORT && (CHAINED || c.n_waves > 1)) {
    c.tag = launch_tag(c);
    chain_chunks<1, BWD, kFoldBatch<1>, !CHAINED>(p, c, &mA, &mB, nullptr, &slice_in, load_h);
  } else {
    load_h();
  }
  if (BWD && ragged) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) place(hp[r]);
  }
  if (BWD) {
    // h[t_lo-1] for the last step: from the neighbouring lane, except at the end of the slice
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const float from_next = __shfl_down(hp[r].get(VEC - 1), 1);  // lane+1 holds timesteps just below ours
      edge_h[r] = lane == lanes - 1 ? eh[r].get(0) : from_next;
    }
  }

  // ---- phase 3 ---------------------------------------------------------------------------
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    keep_packed(a[r]);
    keep_packed(b[r]);
    if (BWD) keep_packed(hp[r]);
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    float state = SHORT ? B[r] : fma0(A[r], lane_read(slice_in, r), B[r]);
    float o0[VEC], o1[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const float av = (j == 0 && first_lane) ? 0.0f : coef(r, j);
      state = __builtin_fmaf(av, state, addend(r, j));
      o0[BWD ? VEC - 1 - j : j] = state;
      if (BWD) o1[VEC - 1 - j] = state * h_prev(r, j);
    }
    if (ok[r]) {
      const int64_t off = ((row0 + r * rows_per_vector) * seq + t_base) * E::kBytes;
      RowT o;
      o.pack(o0);
      store_vector(o, p.out0, off, Flag<(BWD ? kNtOutBwd : kNtOutFwd)>());
      if (BWD) {
        RowT oa;
        oa.pack(o1);
        store_vector(oa, p.out1, off, Flag<kNtOutBwd>());
      }
    }
  }
}

// ScanArgs here: seq = the contiguous length, d = number of rows (bs * channels),
// n_ctiles = ceil(rows / ROWS) row groups, n_chunks = ceil(seq / (waves*64*VEC)).
//
// CHAINED: more than one chunk.  Later chunks wait for a chunk's map, so wave 0 folds what has arrived after one look at
// all the waves' words; in a launch of one chunk only the workgroup's own waves wait, and wave 0 awaits
// their maps in fours.  Kernels of their own because a branch inside one kernel pays for both: the part that
// chains costs a backward 25 vector registers and 33 spilled scalar ones, a forward 11 and 29.  bf16, one launch behind the
// other, fours everywhere / one look everywhere / as it is: chained forwards (13, 768, 4859) 69.6, 66.0 and 65.7 us, (6, 192,
// 32814) 53.7, 50.8 and 51.1; unchained (8, 1024, 2047) 22.0, 22.8 and 21.4, (8, 1024, 1023) 14.8, 14.3 and 13.5, (8, 1024,
// 4095) 45.4, 44.1 and 43.0, backward (8, 1024, 4096) 59.0, 59.1 and 56.0.  22 shapes in both directions and in bf16 and
// fp32: 1.5 % faster in the mean than fours everywhere, 0.8 % than one look; the slowest, forwards (8, 1024, 4096)
// 40.1 -> 40.7 and (4, 300, 9001) 19.8 -> 20.1.  One look without a chain: 0.4 % slower in the mean, forward (8,
// 1024, 1023) 13.8.
template <typename E, int VEC, int ROWS, bool BWD, bool RAGGED, bool SHORT, bool CHAINED>
__global__ __launch_bounds__(1024) void cm_scan_kernel(const ScanArgs p) {
  extern __shared__ float lds[];
  __shared__ uint32_t s_ready[16];  // per wave: see announce_map

  TileCtx c;
  c.wcol = 0;
  c.lane = threadIdx.x & 63;
  c.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  c.n_waves = blockDim.x >> 6;
  c.look = p.look_waves;
  float2 *const lds_maps = reinterpret_cast<float2 *>(lds);  // laid out as in scan_kernel with one slot per lane
  c.lds_pred = lds_maps + 2 * c.n_waves * 64;
  c.seq = p.seq;
  c.s_ready = s_ready;
  if (threadIdx.x < 16) s_ready[threadIdx.x] = threadIdx.x < static_cast<uint32_t>(c.n_waves) ? 0u : ~0u;
  __syncthreads();
  c.row_bytes = 0;
  c.lane_off = 0;
  c.col_ok = true;
  c.tile_base = c.chan_row = c.r0 = 0;
#ifdef FSS_TRACE
  c.trace_wave = 0;
#endif
  c.chained = CHAINED;
  c.epoch = CHAINED ? read_epoch(p) : 0u;
  c.tag = 0u;
  c.anchor = c.span = 0;

  uint32_t parity = 0;
  uint32_t tile_no = 0;
  for (uint32_t tile = blockIdx.x; tile < static_cast<uint32_t>(p.n_tiles); tile += gridDim.x, parity ^= 1u) {
    c.tile_no = ++tile_no;
    c.lds_map = lds_maps + parity * c.n_waves * 64;
    const ScanArgs &plan = fresh_args();
    const uint32_t chunk = divide(tile, plan.by_groups);
    const uint32_t ctile = tile - chunk * static_cast<uint32_t>(p.n_ctiles);
    c.chunk = static_cast<int>(chunk);
    c.ctile = static_cast<int>(ctile);
    c.last = c.chunk == p.n_chunks - 1;
    place_in_chain(plan, c);
    cm_tile<E, VEC, ROWS, BWD, RAGGED, SHORT, CHAINED>(p, c, static_cast<int64_t>(ctile) * (SHORT ? ROWS * (64 >> p.row_lanes_log2) : ROWS), p.d);
  }
  count_out(p, c);
}

// ---- launching ---------------------------------------------------------------------

template <typename E, int VEC, bool BWD, bool RAGGED, bool SHORT, bool CHAINED>
int launch_cm_kernel(const ScanArgs &args, const CmPlan &pl, int max_groups, hipStream_t stream) {
  constexpr int kRows = BWD || SHORT ? kCmRowsBwd : kCmRowsFwd;  // (eight vectors a lane would cost SHORT 23 spilled registers)
  static int resident[17] = {0};
  const int waves = pl.waves;
  const size_t lds = lds_bytes(waves, 1);
  const int fit = resident_workgroups(cm_scan_kernel<E, VEC, kRows, BWD, RAGGED, SHORT, CHAINED>, waves, lds, resident);
  if (fit <= 0) return FSS_ERR_LAUNCH;
  int64_t n_groups = pl.n_tiles < fit ? pl.n_tiles : fit;
  if (max_groups > 0 && max_groups < n_groups) n_groups = max_groups;
  hipLaunchKernelGGL((cm_scan_kernel<E, VEC, kRows, BWD, RAGGED, SHORT, CHAINED>), dim3(static_cast<uint32_t>(n_groups)),
                     dim3(static_cast<uint32_t>(waves) * 64), lds, stream, args);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    tls_hip_error = static_cast<int>(e);
    return FSS_ERR_LAUNCH;
  }
  return FSS_OK;
}

template <typename E, int VEC, bool BWD, bool RAGGED = false, bool SHORT = false>
int launch_cm_one(const ScanArgs &args, const CmPlan &pl, int max_groups, hipStream_t stream) {
  if constexpr (!SHORT)  // (whose rows are one lane group's, in one chunk)
    if (pl.n_chunks > 1) return launch_cm_kernel<E, VEC, BWD, RAGGED, SHORT, true>(args, pl, max_groups, stream);
  return launch_cm_kernel<E, VEC, BWD, RAGGED, SHORT, false>(args, pl, max_groups, stream);
}

template <typename E, bool BWD>
int launch_cm(const ScanArgs &args, const CmPlan &pl, int max_groups, hipStream_t stream) {
  constexpr int kWidest = 16 / E::kBytes;
  if (pl.row_lanes_log2 < 6) return launch_cm_one<E, kWidest, BWD, true, true>(args, pl, max_groups, stream);
  if (pl.vec == kWidest)
    return args.seq % kWidest == 0 ? launch_cm_one<E, kWidest, BWD>(args, pl, max_groups, stream)
                                   : launch_cm_one<E, kWidest, BWD, true>(args, pl, max_groups, stream);
  if (pl.vec == 1) return launch_cm_one<E, 1, BWD>(args, pl, max_groups, stream);
  if constexpr (E::kBytes == 2) {
    if (pl.vec == 2) return launch_cm_one<E, 2, BWD>(args, pl, max_groups, stream);
  }
  return FSS_ERR_BAD_CONFIG;
}

int run_cm_scan(int dtype, int dir, const void *alpha, const void *in_b, const void *in_h, void *out0, void *out1,
                int64_t bs, int64_t d, int64_t seq, void *workspace, size_t workspace_bytes, void *stream,
                const fss_config *cfg) {
  if (bs < 0 || seq < 0 || d < 0) return FSS_ERR_BAD_SHAPE;
  if (dtype != FSS_BF16 && dtype != FSS_F32 && dtype != FSS_F16) return FSS_ERR_BAD_CONFIG;
  if (bs == 0 || seq == 0 || d == 0) return FSS_OK;
  if (bs > INT64_MAX / d) return FSS_ERR_BAD_SHAPE;
  if (!alpha || !in_b || !out0) return FSS_ERR_NULL_POINTER;
  if (dir == FSS_BWD && (!in_h || !out1)) return FSS_ERR_NULL_POINTER;
  const size_t esize = dtype != FSS_F32 ? 2 : 4;
  const size_t align = dir == FSS_BWD ? common_alignment({alpha, in_b, in_h, out0, out1})
                                      : common_alignment({alpha, in_b, out0});
  if (align < esize) return FSS_ERR_MISALIGNED;
  CmPlan pl;
  int rc = make_cm_plan(pl, bs * d, seq, dtype, dir, align, cfg);
  if (rc != FSS_OK) return rc;
  if (pl.n_chunks > 1) {
    if (!workspace || workspace_bytes < pl.ws_bytes) return FSS_ERR_WORKSPACE_SMALL;
    if (reinterpret_cast<uintptr_t>(workspace) % 256 != 0) return FSS_ERR_MISALIGNED;
  }
  rc = check_device();
  if (rc != FSS_OK) return rc;
  ScanArgs args;
  args.in_a = static_cast<const char *>(alpha);
  args.in_b = static_cast<const char *>(in_b);
  args.in_h = static_cast<const char *>(in_h);
  args.out0 = static_cast<char *>(out0);
  args.out1 = static_cast<char *>(out1);
  args.in_x = nullptr;
  args.seq = seq;
  args.d = bs * d;  // rows
  args.tiles_per_row = 1;
  args.row_lanes_log2 = pl.row_lanes_log2;
  args.n_ctiles = static_cast<int32_t>(pl.n_rowtiles);
  args.n_chunks = static_cast<int32_t>(pl.n_chunks);
  args.n_tiles = static_cast<int32_t>(pl.n_tiles);
  args.n_groups = static_cast<int32_t>(pl.n_rowtiles);
  args.look_waves = look_waves(pl.waves, 1);
  args.period = chain_period(pl.n_rowtiles, pl.waves);
  set_divisors(args);
  args.spin_limit = __atomic_load_n(&g_spin_limit, __ATOMIC_RELAXED);
  args.hdr = static_cast<uint32_t *>(workspace);
  args.words = workspace ? reinterpret_cast<uint64_t *>(static_cast<char *>(workspace) + kHeaderBytes) : nullptr;
#ifdef FSS_TRACE
  args.trace = nullptr;
#endif
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int max_groups = cfg ? cfg->max_groups : 0;
  const bool bwd = dir == FSS_BWD;
  const ScanOrderGuard ordered(s);
  if (dtype == FSS_BF16) return bwd ? launch_cm<BF16, true>(args, pl, max_groups, s) : launch_cm<BF16, false>(args, pl, max_groups, s);
  if (dtype == FSS_F16) return bwd ? launch_cm<F16, true>(args, pl, max_groups, s) : launch_cm<F16, false>(args, pl, max_groups, s);
  return bwd ? launch_cm<F32, true>(args, pl, max_groups, s) : launch_cm<F32, false>(args, pl, max_groups, s);
}

}  // namespace fss
