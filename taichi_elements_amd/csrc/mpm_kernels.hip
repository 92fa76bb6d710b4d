// gfx950 kernels of the MLS-MPM substep.
//
// One substep (mpm_solver.py:789-799) is:
//   k_keys            block key of every particle + per-block counts   (build_pid, mpm:344-361;
//                     first substep, or positions set by the host)
//   k_bscan*          scan of the dense block window: particle offsets,
//                     transfer work items (chunks), active grid blocks  (replaces the pointer
//                                                                        SNodes and deactivate_all)
//   k_onesweep        stable LSD radix sort of slots by block key (with k_keys)
//   k_p2g             per chunk: its particles (from the sort, or in the
//                     steady state from g2p's direction lists),
//                     constitutive update + scatter into an
//                     LDS tile of (4+2)^d nodes, tile written to HBM     (p2g, mpm:487-584);
//                     every few substeps the particle state also moves
//                     into the sorted order
//   k_grid_op         per active node: sum of the overlapping tiles,
//                     normalisation, gravity, post-process              (mpm:586-692)
//   k_g2p             per chunk: LDS tile of grid velocity, gather,
//                     advection, max |v|, next binning's lists          (g2p, mpm:694-735)
// Small scenes run the grid operator inside k_g2p, in 2D also the scan inside
// k_p2g.
// use_g2p2g replaces p2g / grid op / g2p with k_g2p2g + k_grid_op_g2p2g
// (mpm_g2p2g.h); the differentiable backward runs the adjoints of
// mpm_adjoint.h.  Particles are read and written through Particles<D, Q>
// (mpm_particles.h), instantiated for the float and the packed layout.
#include "mpm_kernels.h"

#include <map>
#include <mutex>

#include "mpm_binning.h"
#include "mpm_adjoint.h"
#include "mpm_g2p2g.h"

namespace mpm {

// ---------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ int4 add4(int4 a, int4 b) {
  return make_int4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}

__device__ __forceinline__ int4 wave_inclusive_scan4(int4 v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    int4 t;
    t.x = __shfl_up(v.x, off);
    t.y = __shfl_up(v.y, off);
    t.z = __shfl_up(v.z, off);
    t.w = __shfl_up(v.w, off);
    if (lane >= off) v = add4(v, t);
  }
  return v;
}

// Set bits of mask below this lane.
__device__ __forceinline__ int lanes_before(unsigned long long mask) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
}

// Exclusive scan of one int4 per thread over a kThreads workgroup.
__device__ __forceinline__ int4 block_exscan4(int4 v, int4* total, int4* wsum) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int4 inc = wave_inclusive_scan4(v);
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
  int4 pre = make_int4(0, 0, 0, 0), tot = make_int4(0, 0, 0, 0);
#pragma unroll
  for (int w = 0; w < kThreads / 64; w++) {
    if (w < wave) pre = add4(pre, wsum[w]);
    tot = add4(tot, wsum[w]);
  }
  __syncthreads();
  *total = tot;
  return make_int4(pre.x + inc.x - v.x, pre.y + inc.y - v.y, pre.z + inc.z - v.z,
                   pre.w + inc.w - v.w);
}

// ---------------------------------------------------------------------------
// binning: block keys and per-block counts (build_pid, mpm_solver.py:357-361)
// ---------------------------------------------------------------------------
template <int D, bool Q>
__global__ __launch_bounds__(kThreads) void k_keys(const Params* __restrict__ scenes,
                                                   const float* __restrict__ pf,
                                                   const int* __restrict__ pi, int64_t cap, int n,
                                                   int total_blocks, int* __restrict__ keys,
                                                   int* __restrict__ count, int* __restrict__ err) {
  using L = Layout<D>;
  const int lane = threadIdx.x & 63;
  for (int i0 = blockIdx.x * kThreads; i0 < n; i0 += gridDim.x * kThreads) {
    const int i = i0 + threadIdx.x;
    bool valid = false;
    int key = total_blocks;
    if (i < n) {
      const Params& P = scenes[pi[(int64_t)L::SCENE * cap + i]];
      float xi[3];
      Particles<D, Q>::load_x(pf, cap, i, xi);
      int lin = 0;
      valid = true;
#pragma unroll
      for (int a = D - 1; a >= 0; a--) {
        int base;
        float fx;
        base_fx(xi[a], P.inv_dx, base, fx);
        const int lb = (base >> 2) - P.blo[a];
        // the block and its +1 neighbour must lie inside the scene's window
        if (lb < 0 || lb >= P.bnl[a] - 1) valid = false;
        lin = lin * P.bn[a] + lb + (a == D - 1 ? P.zoff : 0);
      }
      key = valid ? lin : total_blocks;
      keys[i] = key;
      if (!valid) atomicOr(err, 1);
    }
    // wave-aggregated counting (count[total_blocks] counts escaped particles):
    // sorted input gives 1-3 distinct keys per wave
    const bool in = i < n;
    unsigned long long pending = __ballot(in);
    while (pending) {
      const int leader = __ffsll(pending) - 1;
      const int lk = __shfl(key, leader);
      const unsigned long long same = __ballot(in && key == lk);
      if (lane == leader) atomicAdd(&count[lk], (int)__popcll(same));
      pending &= ~same;
    }
  }
}

// Per-block values of the dense window scan: (particles, chunks, active grid
// block, non-empty particle block).  A grid block is active when one of the
// particle blocks b - {0,1}^d holds particles (their stencils reach it).
template <int D>
__device__ __forceinline__ int4 block_values(int bid, const int lb[3],
                                             const int* __restrict__ count, const Params& P) {
  const int c = count[bid];
  // p2g reaches blocks b + {0, 1}^d of a particle block b; the fused g2p2g
  // transfer (new positions up to one cell away) b + {-1, 0, 1}^d.  The loads
  // are unconditional (past the window's edge: the block's own count), so
  // that all of them are in flight at once.
  const int sx = 1, sy = P.bn[0], sz = P.bn[0] * P.bn[1];
  int any = 0;
  if (!P.g2p2g) {
#pragma unroll
    for (int k = 0; k < (D == 3 ? 8 : 4); k++) {
      const int dx = k & 1, dy = (k >> 1) & 1, dz = k >> 2;
      const bool in = lb[0] >= dx && lb[1] >= dy && lb[2] >= dz;
      any |= count[in ? bid - dx * sx - dy * sy - dz * sz : bid];
    }
  } else {
#pragma unroll
    for (int k = 0; k < (D == 3 ? 27 : 9); k++) {
      const int dx = k % 3 - 1, dy = (k / 3) % 3 - 1, dz = D == 3 ? k / 9 - 1 : 0;
      const int q[3] = {lb[0] - dx, lb[1] - dy, lb[2] - dz};
      const bool in = q[0] >= 0 && q[1] >= 0 && q[2] >= 0 && q[0] < P.bn[0] && q[1] < P.bn[1] &&
                      (D == 2 || q[2] < P.bn[2]);
      any |= count[in ? bid - dx * sx - dy * sy - dz * sz : bid];
    }
  }
  const bool act = any != 0;  // counts are not negative
  return make_int4(c, 0, act ? 1 : 0, c > 0 ? 1 : 0);
}

template <int D>
__device__ __forceinline__ int4 block_values(int bid, const int* __restrict__ count,
                                             const Params& P, int chunk) {
  int lb[3];
  decode_local<D>(bid, P, lb);
  int4 v = block_values<D>(bid, lb, count, P);
  v.y = (v.x + chunk - 1) / chunk;
  return v;
}

// ---------------------------------------------------------------------------
// the radix passes' scans with decoupled look-back (Merrill & Garland 2016)
//
// Status word: value in bits 0-31, flag in bits 32-33 (1 = tile aggregate,
// 2 = inclusive prefix), launch epoch in bits 34-63.  Words left by earlier
// launches carry an older epoch and read as "not ready", so the status
// arrays are never cleared.  Past kRadixSmallTiles tiles they are numbered in
// the order workgroups start (an atomic ticket), so a tile only waits on tiles
// that are already running; the last workgroup to finish resets the ticket and
// advances the epoch, which keeps the kernels free of host-side per-launch
// state.
// ---------------------------------------------------------------------------
constexpr unsigned long long kFlagAgg = 1ull << 32, kFlagPre = 2ull << 32;
// Polls (of a microsecond or more) after which a wait for another tile gives
// up: seconds, because a tile that is not running yet starts only when other
// work on the device makes room for it.
constexpr int kWaitLimit = 1 << 22;

__device__ __forceinline__ unsigned long long lb_epoch_bits(unsigned epoch) {
  return (unsigned long long)(epoch & 0x3fffffffu) << 34;
}

__device__ __forceinline__ void lb_publish(unsigned long long* p, unsigned long long flag,
                                           unsigned epoch, unsigned value) {
  __hip_atomic_store(p, lb_epoch_bits(epoch) | flag | (unsigned long long)value, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

// Exclusive prefix of channel `chan` for tile `tile` (status[t * stride + chan]).
// A bounded wait: past kWaitLimit polls it flags err bit 1 and returns what it has.
__device__ __forceinline__ unsigned lb_lookback(const unsigned long long* status, int stride,
                                                int tile, int chan, unsigned epoch, int* err) {
  constexpr int W = 8;  // predecessors read at once: one round trip, not eight in turn
  const unsigned long long ep = lb_epoch_bits(epoch);
  unsigned excl = 0;
  int spins = 0;
  for (int t = tile - 1; t >= 0;) {
    unsigned long long w[W];
#pragma unroll
    for (int j = 0; j < W; j++)
      w[j] = t - j >= 0 ? __hip_atomic_load(&status[(int64_t)(t - j) * stride + chan],
                                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                        : (ep | kFlagPre);
    bool ready = true, done = false;
    int used = 0;
#pragma unroll
    for (int j = 0; j < W; j++) {
      ready &= (w[j] & ~0x3ffffffffull) == ep && (w[j] & (kFlagAgg | kFlagPre));
      if (ready && !done) {
        excl += (unsigned)w[j];
        done = (w[j] & kFlagPre) != 0;
        used++;
      }
    }
    if (done) break;
    t -= used;
    if (used < W) {
      if (++spins > kWaitLimit) {
        atomicOr(err, 2);
        return excl;
      }
      __builtin_amdgcn_s_sleep(1);
    }
  }
  return excl;
}

struct LBTicket {
  int tile;
  unsigned epoch;
};

// A few tiles find room on the device whatever else runs there and take no
// ticket (a round trip more: 200k keys 12.5 us a pass, 11.0 without); the epoch
// changes only after every tile has read it.
__device__ __forceinline__ LBTicket lb_acquire(LBState* st, LBTicket* sh, int ntiles) {
  if (ntiles <= kRadixSmallTiles)
    return {(int)blockIdx.x,
            __hip_atomic_load(&st->epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)};
  if (threadIdx.x == 0) {
    sh->tile = (int)atomicAdd(&st->tile_ctr, 1ull);
    sh->epoch = __hip_atomic_load(&st->epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  return *sh;
}

__device__ __forceinline__ void lb_release(LBState* st, int ntiles, unsigned epoch) {
  if (threadIdx.x == 0) {
    const unsigned long long d = atomicAdd(&st->done_ctr, 1ull);
    if (d == (unsigned long long)(ntiles - 1)) {
      __hip_atomic_store(&st->tile_ctr, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(&st->done_ctr, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(&st->epoch, epoch + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// ---------------------------------------------------------------------------
// scan of the dense block window (one launch): particle offsets, chunk list,
// active grid blocks, and the radix digit histograms of the block keys
// weighted by the particle counts (count[total_blocks] holds the particles
// outside the window, whose key is total_blocks).
//
// Bound by its chain of dependent round trips to memory: the counts, then the
// other tiles' sums.  Up to kScanTilesOnePass tiles every tile publishes its
// four sums and adds up those of all tiles before it (one wave per sum, seven
// words per lane): nobody waits for somebody else's prefix.
// status[tile][channel] holds kScanReady | sum and is cleared by the substep's
// first transfer, so there is no ticket, no epoch and no release.  With tickets, a look-back over prefixes and each
// neighbour's count loaded behind a branch: 1M particles (99 tiles) 11.8 ->
// 7.0 us, 2D 20k 6.1 -> 4.6, unbounded 50k 16.4 -> 7.8, use_g2p2g 300k 13.9 ->
// 8.1.  Larger windows take the tile sums from k_bscan_reduce, which also adds
// them up by groups of kScanGroup tiles: every tile adds up the groups before
// its own and the tiles of its own before it, a round of loads each up to the
// largest window (2^24 blocks, 256 groups), and there is no kernel between the
// two.  Substeps of 1M particles with a kernel between that scans the tile sums,
// with every tile adding up all tiles before it, and with groups: 512^3 (4.6k
// tiles) 212, 160 and 156 us, 800^3 (16.8k) 338, 287 and 232, 1000^3 (32.4k)
// 493, 537 and 330 (the first with the other kernels of its time, ~45 us more).
// ---------------------------------------------------------------------------
constexpr unsigned long long kScanReady = 1ull << 32;

// Sum of channel c of the tiles before `tile`, by one wave.  Tiles that are
// not running yet (other work holds the device) start as that work ends, so
// the wait is long but bounded: past kWaitLimit polls it flags err bit 1 and
// counts what it has.
__device__ __forceinline__ unsigned scan_before(const unsigned long long* status, int tile, int c,
                                                int* err) {
  constexpr int W = kScanTilesOnePass / 64;
  const int lane = threadIdx.x & 63;
  unsigned long long w[W];
#pragma unroll
  for (int j = 0; j < W; j++) w[j] = lane + 64 * j < tile ? 0ull : kScanReady;
  for (int spins = 0;; spins++) {
    bool ready = true;
#pragma unroll
    for (int j = 0; j < W; j++) {
      if (!(w[j] & kScanReady))
        w[j] = __hip_atomic_load(&status[(int64_t)(lane + 64 * j) * 4 + c], __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
      ready &= (w[j] & kScanReady) != 0;
    }
    if (__all(ready)) break;
    if (spins > kWaitLimit) {
      atomicOr(err, 2);
      break;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  unsigned v = 0;
#pragma unroll
  for (int j = 0; j < W; j++) v += (unsigned)w[j];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

template <int D>
__global__ __launch_bounds__(kThreads) void k_bscan(
    const Params* __restrict__ scenes, const int* __restrict__ count, int* __restrict__ count_next, int total_blocks,
    int chunk, int ntiles, int passes, int* __restrict__ pstart, int* __restrict__ pchunk_begin,
    int* __restrict__ pchunk_cnt, int4* __restrict__ chunks, int* __restrict__ active,
    int* __restrict__ totals, int* __restrict__ ghist, int* __restrict__ ghist_next,
    unsigned long long* __restrict__ status, const int4* __restrict__ tile_sums,
    const int4* __restrict__ group_sums, int* __restrict__ err, int* __restrict__ step) {
  // one launch per substep: the substep counter of the max-velocity slots
  if (step && blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(step, 1);
  __shared__ int4 wsum[kThreads / 64];
  __shared__ unsigned excl_sh[4];
  __shared__ int lh[kMaxRadixPasses][kRadixBins];
  const Params& P = scenes[0];  // the combined window extents
  const int tile = blockIdx.x;
  if (passes > 0)
    for (int i = threadIdx.x; i < kMaxRadixPasses * kRadixBins; i += kThreads) (&lh[0][0])[i] = 0;

  const int first = tile * kScanTile + threadIdx.x * kScanItems;
  int4 vals[kScanItems];
  int4 acc = make_int4(0, 0, 0, 0);
#pragma unroll
  for (int k = 0; k < kScanItems; k++) {
    const int bid = first + k;
    vals[k] = bid < total_blocks ? block_values<D>(bid, count, P, chunk) : make_int4(0, 0, 0, 0);
    acc = add4(acc, vals[k]);
  }
  int4 tot;
  int4 pre = block_exscan4(acc, &tot, wsum);  // contains __syncthreads (lh zeroed)

  // digit histograms of the keys, weighted by particle counts
#pragma unroll
  for (int k = 0; k < kScanItems; k++) {
    const int bid = first + k;
    if (bid < total_blocks && vals[k].x > 0)
      for (int ps = 0; ps < passes; ps++) atomicAdd(&lh[ps][(bid >> (8 * ps)) & 255], vals[k].x);
  }
  if (tile == 0 && threadIdx.x == 0) {
    const int inval = count[total_blocks];
    if (inval > 0)
      for (int ps = 0; ps < passes; ps++)
        atomicAdd(&lh[ps][(total_blocks >> (8 * ps)) & 255], inval);
  }

  static_assert(kThreads == 256, "one wave per scanned channel");
  if (tile_sums) {
    int4 before = make_int4(0, 0, 0, 0), all;
    const int group = tile / kScanGroup;
    for (int i = threadIdx.x; i < group; i += kThreads) before = add4(before, group_sums[i]);
    for (int i = group * kScanGroup + threadIdx.x; i < tile; i += kThreads)
      before = add4(before, tile_sums[i]);
    block_exscan4(before, &all, wsum);
    if (threadIdx.x < 4) {
      const int c = threadIdx.x;
      excl_sh[c] = (unsigned)(c == 0 ? all.x : c == 1 ? all.y : c == 2 ? all.z : all.w);
    }
  } else {
    // wave c takes channel c
    const int c = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const unsigned agg = (unsigned)(c == 0 ? tot.x : c == 1 ? tot.y : c == 2 ? tot.z : tot.w);
    if (lane == 0)
      __hip_atomic_store(&status[(int64_t)tile * 4 + c], kScanReady | (unsigned long long)agg,
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned excl = scan_before(status, tile, c, err);
    if (lane == 0) excl_sh[c] = excl;
  }
  __syncthreads();
  pre = add4(pre, make_int4((int)excl_sh[0], (int)excl_sh[1], (int)excl_sh[2], (int)excl_sh[3]));
#pragma unroll
  for (int k = 0; k < kScanItems; k++) {
    const int bid = first + k;
    if (bid >= total_blocks) break;
    const int4 v = vals[k];
    pstart[bid] = pre.x;
    pchunk_begin[bid] = pre.y;
    pchunk_cnt[bid] = v.y;
    for (int c = 0; c < v.y; c++) {
      const int b0 = pre.x + c * chunk;
      const int b1 = min(b0 + chunk, pre.x + v.x);
      chunks[pre.y + c] = make_int4(bid, b0, b1, 0);
    }
    if (v.z) active[pre.z] = bid;
    count_next[bid] = 0;
    pre = add4(pre, v);
  }
  if (tile == 0 && threadIdx.x == 0) count_next[total_blocks] = 0;
  if (tile == ntiles - 1 && threadIdx.x == 0) {
    totals[kTotValid] = (int)excl_sh[0] + tot.x;
    totals[kTotChunks] = (int)excl_sh[1] + tot.y;
    totals[kTotActive] = (int)excl_sh[2] + tot.z;
    totals[kTotPBlocks] = (int)excl_sh[3] + tot.w;
  }
  // flush the histograms; clear next substep's copy
  for (int i = threadIdx.x; i < passes * kRadixBins; i += kThreads) {
    const int h = (&lh[0][0])[i];
    if (h) atomicAdd(&ghist[i], h);
  }
  if (tile == 0)
    for (int i = threadIdx.x; i < kMaxRadixPasses * kRadixBins; i += kThreads) ghist_next[i] = 0;
}

// Tile sums and group sums (zero before) of a window too large for the single
// pass.
template <int D>
__global__ __launch_bounds__(kThreads) void k_bscan_reduce(const Params* __restrict__ scenes,
                                                           const int* __restrict__ count,
                                                           int total_blocks, int chunk,
                                                           int4* __restrict__ tile_sums,
                                                           int4* __restrict__ group_sums) {
  __shared__ int4 wsum[kThreads / 64];
  const Params& P = scenes[0];  // the combined window extents
  int4 acc = make_int4(0, 0, 0, 0);
  const int first = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
#pragma unroll
  for (int k = 0; k < kScanItems; k++)
    if (first + k < total_blocks) acc = add4(acc, block_values<D>(first + k, count, P, chunk));
  int4 tot;
  block_exscan4(acc, &tot, wsum);
  if (threadIdx.x < 4) {
    const int c = threadIdx.x;
    const int v = c == 0 ? tot.x : c == 1 ? tot.y : c == 2 ? tot.z : tot.w;
    reinterpret_cast<int*>(&tile_sums[blockIdx.x])[c] = v;
    if (v) atomicAdd(&reinterpret_cast<int*>(&group_sums[blockIdx.x / kScanGroup])[c], v);
  }
}

// ---------------------------------------------------------------------------
// one pass of the stable LSD radix sort (8-bit digit), single launch.  Each
// wave ranks its own contiguous quarter of the tile with ballots and
// wave-private LDS counters (no workgroup barrier per round); one prefix over
// the four waves gives tile-local stable ranks; decoupled look-back over
// tiles gives the per-digit tile offsets; the digit totals come from the
// histogram k_bscan built.
//
// Up to a few hundred thousand keys a pass is one chain of latencies: the
// keys, ITEMS rounds of ranking, the look-back, the stores.  Smaller tiles
// halve the rounds but lengthen the look-back, whose status words come from
// memory past the L2s: 200k keys, 16 items a thread with a ticket and one
// predecessor at a time 13.0 us; eight predecessors at a time, no ticket and
// 16 / 8 / 4 / 2 items 12.5 / 11.0 / 11.9 / 14.1 us; 32 predecessors at a time
// 13.0 (8 items) and 14.6 (4).
// ---------------------------------------------------------------------------
template <int ITEMS>
__global__ __launch_bounds__(kThreads) void k_onesweep(
    const int* __restrict__ keys_in, const int* __restrict__ vals_in, int* __restrict__ keys_out,
    int* __restrict__ vals_out, int n, int shift, int ntiles, const int* __restrict__ ghist,
    unsigned long long* __restrict__ status, LBState* __restrict__ lbs, int* __restrict__ err) {
  constexpr int WAVES = kThreads / 64;
  constexpr int TILE = kThreads * ITEMS;
  constexpr int PER_WAVE = TILE / WAVES;
  constexpr int ROUNDS = PER_WAVE / 64;
  __shared__ LBTicket tk_sh;
  __shared__ int wcnt[WAVES][kRadixBins];
  __shared__ int gbase[kRadixBins];
  __shared__ int4 wsum[WAVES];
  const LBTicket tk = lb_acquire(lbs, &tk_sh, ntiles);
  const int tile = tk.tile;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const unsigned long long lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  const int i0 = tile * TILE + wave * PER_WAVE + lane;

  int key[ROUNDS], val[ROUNDS], lr[ROUNDS];
#pragma unroll
  for (int r = 0; r < ROUNDS; r++) {
    const int i = i0 + r * 64;
    key[r] = i < n ? keys_in[i] : 0;
    val[r] = i < n ? (vals_in ? vals_in[i] : i) : 0;
  }
#pragma unroll
  for (int w = 0; w < WAVES; w++) wcnt[w][threadIdx.x] = 0;
  int4 gtot;
  // block_exscan4 synchronises, which also publishes the zeroed counters
  const int gex = block_exscan4(make_int4(ghist[threadIdx.x], 0, 0, 0), &gtot, wsum).x;
  int* my = wcnt[wave];
#pragma unroll
  for (int r = 0; r < ROUNDS; r++) {
    const bool valid = i0 + r * 64 < n;
    const int d = (key[r] >> shift) & (kRadixBins - 1);
    unsigned long long peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; b++) {
      const bool bit = (d >> b) & 1;
      const unsigned long long bal = __ballot(bit);
      peers &= bit ? bal : ~bal;
    }
    const int rank = (int)__popcll(peers & lt);
    // every lane reads its digit's counter before the group leader bumps it;
    // a wave's LDS accesses are served in program order
    const int base = my[d];
    __asm__ volatile("" ::: "memory");
    if (valid && rank == 0) my[d] = base + (int)__popcll(peers);
    __asm__ volatile("" ::: "memory");
    lr[r] = base + rank;
  }
  __syncthreads();
  int agg = 0;
#pragma unroll
  for (int w = 0; w < WAVES; w++) {
    const int c = wcnt[w][threadIdx.x];
    wcnt[w][threadIdx.x] = agg;
    agg += c;
  }
  {
    unsigned excl = 0;
    unsigned long long* st = &status[(int64_t)tile * kRadixBins + threadIdx.x];
    if (tile == 0) {
      lb_publish(st, kFlagPre, tk.epoch, (unsigned)agg);
    } else {
      lb_publish(st, kFlagAgg, tk.epoch, (unsigned)agg);
      excl = lb_lookback(status, kRadixBins, tile, threadIdx.x, tk.epoch, err);
      lb_publish(st, kFlagPre, tk.epoch, excl + (unsigned)agg);
    }
    gbase[threadIdx.x] = gex + (int)excl;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ROUNDS; r++) {
    if (i0 + r * 64 < n) {
      const int d = (key[r] >> shift) & (kRadixBins - 1);
      const int pos = gbase[d] + my[d] + lr[r];
      if (pos >= 0 && pos < n) {
        keys_out[pos] = key[r];
        vals_out[pos] = val[r];
      } else {
        atomicOr(err, 4);  // histogram and keys disagree (cannot happen)
      }
    }
  }
  __syncthreads();
  lb_release(lbs, ntiles, tk.epoch);
}

// ---------------------------------------------------------------------------
// The block scan inside p2g.  Every workgroup scans the whole window itself
// (kWindowItems blocks per thread) to find its chunks; the last one, which
// seldom has a chunk, also writes k_bscan's results for the kernels after it.
// Bound, like k_bscan, by round trips to memory, of which this is one instead
// of a kernel's four: taken in 2D by steady-state substeps of windows of up to
// kThreads kWindowItems blocks whose transfer walks the direction lists, where
// each workgroup has about one chunk.  A kernel of 3.9 to 4.7 us and its launch
// go, p2g takes 3 to 4 us longer: a substep of 5000 particles (400 blocks)
// 19.8 -> 17.5 us, 60000 (1369 blocks) 24.1 -> 23.1, 160000 (2025 blocks) 28.5
// -> 27.4.  With the counts read by each thread where it needs them, without
// LDS, p2g took 12 us longer at 1369 blocks.  In 3D the registers spill.
// ---------------------------------------------------------------------------
struct WindowScan {
  const int* count;
  int* count_next;
  int total_blocks, chunk;
  unsigned chunk_inv;  // ceil(2^32 / chunk): x / chunk for x < 2^32 / chunk, chunk > 1
  int *pstart, *pchunk_begin, *pchunk_cnt;
  int4* chunks;
  int *active, *totals, *ghist_next, *step;
};
constexpr int kWindowItems = 9;
constexpr int kWindowGroups = 1024;  // all resident at once

template <int D>
struct ScannedWindow {
  static constexpr int K = kWindowItems;
  int per;                   // blocks per thread: odd, so that its LDS reads conflict with none
  int nchunks, pos, chunk0;  // position and chunk of the thread's first block
  int n[K], nc[K];           // particles and chunks of its blocks

  // lcount: kThreads K words of LDS, free again afterwards.
  __device__ void scan(const WindowScan& A, const Params& P, int* lcount, int4* wsum) {
    per = (A.total_blocks + kThreads - 1) / kThreads | 1;
    int c[K];
#pragma unroll
    for (int k = 0; k < K; k++)
      if (k < per) c[k] = A.count[min(k * kThreads + (int)threadIdx.x, A.total_blocks)];
#pragma unroll
    for (int k = 0; k < K; k++)
      if (k < per) lcount[k * kThreads + threadIdx.x] = c[k];
    lds_barrier();
    const int first = threadIdx.x * per;
    int lb[3] = {0, 0, 0};
    if (first < A.total_blocks) decode_local<D>(first, P, lb);
    int4 v[K], acc = make_int4(0, 0, 0, 0), tot;
#pragma unroll
    for (int k = 0; k < K; k++) {
      v[k] = make_int4(0, 0, 0, 0);
      n[k] = nc[k] = 0;
      if (k >= per) continue;
      // past the window: block 0, read like the others, counts for nothing
      const bool on = first + k < A.total_blocks;
      const int l[3] = {on ? lb[0] : 0, on ? lb[1] : 0, on ? lb[2] : 0};
      v[k] = block_values<D>(on ? first + k : 0, l, lcount, P);
      v[k].y = (int)__umulhi((unsigned)(v[k].x + A.chunk - 1), A.chunk_inv);
      if (!on) v[k] = make_int4(0, 0, 0, 0);
      if (++lb[0] == P.bn[0]) {
        lb[0] = 0;
        if (++lb[1] == P.bn[1]) {
          lb[1] = 0;
          lb[2]++;
        }
      }
      acc = add4(acc, v[k]);
      n[k] = v[k].x;
      nc[k] = v[k].y;
    }
    int4 pre = block_exscan4(acc, &tot, wsum);
    nchunks = tot.y;
    pos = pre.x;
    chunk0 = pre.y;
    if (blockIdx.x != gridDim.x - 1) return;
#pragma unroll
    for (int k = 0; k < K; k++) {
      const int bid = first + k;
      if (k >= per || bid >= A.total_blocks) break;
      A.pstart[bid] = pre.x;
      A.pchunk_begin[bid] = pre.y;
      A.pchunk_cnt[bid] = v[k].y;
      for (int c = 0; c < v[k].y; c++) {
        const int b0 = pre.x + c * A.chunk;
        A.chunks[pre.y + c] = make_int4(bid, b0, min(b0 + A.chunk, pre.x + v[k].x), 0);
      }
      if (v[k].z) A.active[pre.z] = bid;
      A.count_next[bid] = 0;
      pre = add4(pre, v[k]);
    }
    for (int i = threadIdx.x; i < kMaxRadixPasses * kRadixBins; i += kThreads) A.ghist_next[i] = 0;
    if (threadIdx.x == 0) {
      A.count_next[A.total_blocks] = 0;
      A.totals[kTotValid] = tot.x;
      A.totals[kTotChunks] = tot.y;
      A.totals[kTotActive] = tot.z;
      A.totals[kTotPBlocks] = tot.w;
      if (A.step) atomicAdd(A.step, 1);  // the substep counter of the max-velocity slots
    }
  }

  // Chunk c (block, begin, end, the block's first position), from the thread
  // that holds its block; the whole workgroup calls it with a slot that no
  // call without a barrier in between uses.
  __device__ int4 find(int c, int chunk, int4* slot) const {
    int p = pos, c0 = chunk0;
#pragma unroll
    for (int k = 0; k < K; k++) {
      if (c >= c0 && c < c0 + nc[k]) {
        const int b0 = p + (c - c0) * chunk;
        *slot = make_int4(threadIdx.x * per + k, b0, min(b0 + chunk, p + n[k]), p);
      }
      p += n[k];
      c0 += nc[k];
    }
    lds_barrier();
    return *slot;
  }
};

// ---------------------------------------------------------------------------
// P2G (mpm_solver.py:487-584)
//
// One workgroup per chunk (<= kChunkMax particles of one grid block), taken
// kBatch particles at a time through phases 1-3; one node tile per chunk.
//  phase 1  one particle per thread: constitutive update (F, Jp written back)
//           and the particle's affine momentum terms staged in LDS;
//  phase 2  a stable counting sort of the chunk's particles by cell;
//  phase 3  cell-major scatter: lane l of a wave owns cell l of the block
//           (3D: 64 cells = 64 lanes; 2D: 16 cells, four lane groups), so the
//           27 (9) stencil nodes a wave updates in one instruction are
//           distinct and each wave / lane group accumulates into its own LDS
//           tile with plain read-modify-write -- no float atomics;
//  phase 4  the private tiles are summed in a fixed order and the (4+2)^d
//           node tile (momentum, mass) is written to HBM for the grid pass.
// The accumulation order is fixed, so p2g is bitwise reproducible.
// ---------------------------------------------------------------------------
// MODE 0: the forward transfer.  MODE 1: the scatter half of the g2p adjoint
// -- node o of particle p receives w_o (a + c4 Cbar (o - fx)) with
// a = vbar' + dt xbar' and Cbar the adjoint of the new C (gf holds the
// adjoints of the new particle state, same layout as pf); the mass channel
// stays zero.  Both scatter "q + Ad o" per node through the same LDS path.
// At most 128 VGPRs (4 waves per SIMD): the latency of the particle loads
// and of the LDS scatter is hidden better than at 3 waves with no spills
// (measured: 85 -> 75 us per 1M-particle substep, a few spilled registers).
// ORDER: where the chunk's particles come from and what p2g does to their
// order.  kOrderGiven: perm.  kOrderLists: the previous substep's direction
// lists (wave_members); p2g writes perm.  kOrderMove: perm, and the particle
// state moves into the sorted order on the way (position j becomes slot j of
// pf_out / pi_out): p2g reads every field but two integers anyway and is
// bound by the vector ALU and LDS, so the extra writes cost less than a pass
// of their own (1M particles: 76 -> 98 us instead of 76 + 65; 16M: 1.15 ->
// 2.24 ms instead of 1.15 + 1.64).
// SCAN (with kOrderLists): the block scan runs in here (WindowScan).
template <int D, int MODE, bool Q = false, int ORDER = kOrderGiven, bool SCAN = false>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_p2g(
    const Params* __restrict__ scenes, const int* __restrict__ slab, const float* __restrict__ pf,
    const int* __restrict__ pi, int64_t cap, int* __restrict__ perm,
    const int4* __restrict__ chunks, const int* __restrict__ totals, float4* __restrict__ tiles,
    const float* __restrict__ gf, float* __restrict__ pf_out, PrevBinning prev,
    const int* __restrict__ pstart, int* __restrict__ pi_out, int n, int nw,
    int* __restrict__ err, ScanStatus scan, WindowScan window) {
  using L = Layout<D>;
  if (MODE == 0 && !SCAN) scan.clear();
  constexpr int TN = Geo<D>::kTileNodes;
  constexpr int CELLS = Geo<D>::kNodesPerBlock;  // cells of a block (64 / 16)
  constexpr int GROUPS = 64 / CELLS;             // lane groups per wave
  constexpr int WAVES = kThreads / 64;
  constexpr int SUBS = WAVES * GROUPS;           // private tiles
  __shared__ float4 stage[4][kBatch];  // [record part][particle]: lane-contiguous
  __shared__ float4 ptile[SUBS][TN];
  __shared__ int wcnt[WAVES][CELLS];
  __shared__ int cstart[CELLS], ccount[CELLS];
  __shared__ unsigned char order[kBatch];

  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const unsigned long long lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  __shared__ int4 wsum[SCAN ? kThreads / 64 : 1], found[SCAN ? 2 : 1];
  ScannedWindow<D> own;
  if (SCAN) own.scan(window, scenes[0], reinterpret_cast<int*>(&ptile[0][0]), wsum);
  static_assert(!SCAN || sizeof(ptile) >= sizeof(int) * kThreads * kWindowItems, "");
  int turn = 0;
  for (XcdItems it(SCAN ? own.nchunks : totals[kTotChunks], kSpreadChunks); it.valid(); it.next()) {
    const int c = it.c;
    const int4 ck = SCAN ? own.find(c, window.chunk, &found[SCAN ? turn ^= 1 : 0]) : chunks[c];
    int lbc[3], b[3];
    decode_local<D>(ck.x, scenes[0], lbc);
    const Params& P = scenes[scene_of<D>(lbc, slab)];
    int ids[kChunkMax / kThreads];  // slots of this thread's particle of each batch
    if (ORDER == kOrderLists) {
      const int first = SCAN ? ck.w : pstart[ck.x];
      wave_members<D, kChunkMax / kThreads>(lbc, ck.y - first + threadIdx.x, kThreads,
                                            ck.z - first, scenes[0], prev, ids);
#pragma unroll
      for (int k = 0; k < kChunkMax / kThreads; k++) {
        const int j = ck.y + threadIdx.x + k * kThreads;
        if (j >= ck.z) continue;
        if (ids[k] < 0) atomicOr(err, 16);  // counts and lists disagree (cannot happen)
        perm[j] = max(ids[k], 0);
      }
    }
    if (ORDER == kOrderMove)
      for (int j = ck.y + threadIdx.x; j < ck.z; j += kThreads) {
        const int p = perm[j];
        for (int w = 0; w < L::NI; w++) pi_out[(int64_t)w * cap + j] = pi[(int64_t)w * cap + p];
        if (P.skip)  // the scene sits the substep out: its state moves unchanged
          for (int w = 0; w < nw; w++) pf_out[(int64_t)w * cap + j] = pf[(int64_t)w * cap + p];
        if (P.skip) perm[j] = j;
      }
    if (P.skip) continue;  // workgroup-uniform: the whole chunk belongs to one scene
    to_local<D>(lbc, P, b);
#pragma unroll
    for (int a = 0; a < D; a++) b[a] = (b[a] + P.blo[a]) * kBlock;  // first node of the block
    for (int i = threadIdx.x; i < SUBS * TN; i += kThreads)
      (&ptile[0][0])[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    // the chunk's particles, kBatch at a time, all into the same private tiles
    for (int b0 = ck.y; b0 < ck.z; b0 += kBatch) {
      const int nc = min(kBatch, ck.z - b0);
      for (int i = threadIdx.x; i < WAVES * CELLS; i += kThreads) (&wcnt[0][0])[i] = 0;

      // ---- phase 1: constitutive update and staging ----
      const int t = threadIdx.x;
      int p = -1;
      if (ORDER == kOrderLists) {
#pragma unroll
        for (int k = 0; k < kChunkMax / kThreads; k++)
          if (b0 - ck.y == k * kThreads) p = ids[k];
      } else if (t < nc) {
        p = perm[b0 + t];
      }
      const bool valid = p >= 0;
      int cell = 0;
      if (MODE == 1 && valid) {
        const int mat = pi[(int64_t)L::MAT * cap + p];
        float fx[3] = {0.0f, 0.0f, 0.0f};
        int l[3] = {0, 0, 0};
  #pragma unroll
        for (int a = 0; a < D; a++) {
          int base;
          base_fx(pf[(int64_t)(L::X + a) * cap + p], P.inv_dx, base, fx[a]);
          l[a] = min(max(base - b[a], 0), kBlock - 1);
        }
        cell = D == 3 ? l[0] + 4 * (l[1] + 4 * l[2]) : l[0] + 4 * l[1];
        // a stationary particle keeps x, v, C in g2p: no grid adjoint
        const float on = mat == kStationary ? 0.0f : 1.0f;
        float Ad[3][3] = {{0.0f}}, q[3] = {0.0f, 0.0f, 0.0f};
  #pragma unroll
        for (int a = 0; a < D; a++) {
          float s = on * (gf[(int64_t)(L::V + a) * cap + p] + P.dt * gf[(int64_t)(L::X + a) * cap + p]);
  #pragma unroll
          for (int e = 0; e < D; e++) {
            Ad[a][e] = on * P.c4 * gf[(int64_t)(L::C + a * D + e) * cap + p];
            s -= Ad[a][e] * fx[e];
          }
          q[a] = s;
        }
        if (D == 3) {
          stage[0][t] = make_float4(Ad[0][0], Ad[0][1], Ad[0][2], Ad[1][0]);
          stage[1][t] = make_float4(Ad[1][1], Ad[1][2], Ad[2][0], Ad[2][1]);
          stage[2][t] = make_float4(Ad[2][2], q[0], q[1], q[2]);
          stage[3][t] = make_float4(fx[0], fx[1], fx[2], 0.0f);
        } else {
          stage[0][t] = make_float4(Ad[0][0], Ad[0][1], Ad[1][0], Ad[1][1]);
          stage[1][t] = make_float4(q[0], q[1], fx[0], fx[1]);
          stage[2][t] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
      } else if (MODE == 0 && valid) {
        using PS = Particles<D, Q>;
        const int mat = pi[(int64_t)L::MAT * cap + p];
        float xp[3], vp[3], C[3][3], F[3][3], stress[3][3];
        PS::load_x(pf, cap, p, xp);
        PS::load_v(pf, cap, p, vp);
        PS::load_C(pf, cap, p, C);
        PS::load_F(pf, cap, p, F);
        const int po = ORDER == kOrderMove ? b0 + t : p;  // slot of the new state
        if (ORDER == kOrderMove) {
          PS::move_xvC(pf, pf_out, cap, p, po);
          perm[po] = po;
        }
        float Jp = P.plastic ? PS::load_Jp(pf, cap, p) : 1.0f;
        float fx[3] = {0.0f, 0.0f, 0.0f};
        int l[3] = {0, 0, 0};
  #pragma unroll
        for (int a = 0; a < D; a++) {
          int base;
          base_fx(xp[a], P.inv_dx, base, fx[a]);
          // the binning pass put this particle in this block from the same x
          l[a] = min(max(base - b[a], 0), kBlock - 1);
        }
        cell = D == 3 ? l[0] + 4 * (l[1] + 4 * l[2]) : l[0] + 4 * l[1];
        float mu_0 = P.mu_0, lambda_0 = P.lambda_0;
        if (P.youngs) {
          const float E = P.youngs[p];
          mu_0 = E * P.kmu;
          lambda_0 = E * P.kla;
        }
        constitutive<D>(mat, P, mu_0, lambda_0, F, C, Jp, stress);
        PS::store_F(pf_out, cap, po, F);  // the stress already used F before rounding (mpm:567)
        if (P.plastic)
          PS::store_Jp(pf_out, cap, po, Jp);
        else if (!Q && ORDER == kOrderMove)
          PS::store_Jp(pf_out, cap, po, PS::load_Jp(pf, cap, p));
        float mass = P.p_mass;  // mpm_solver.py:571-573
        if (mat == kWater) mass *= P.water_density;
        // contribution to node o: w_o * (mass v + A (o - fx) dx) = w_o * (q + Adx o)
        // with A = stress_scale tau + mass C (mpm_solver.py:569-583)
        float Ad[3][3] = {{0.0f}}, q[3] = {0.0f, 0.0f, 0.0f};
  #pragma unroll
        for (int a = 0; a < D; a++) {
  #pragma unroll
          for (int e = 0; e < D; e++) Ad[a][e] = (P.stress_scale * stress[a][e] + mass * C[a][e]) * P.dx;
          float s = mass * vp[a];
  #pragma unroll
          for (int e = 0; e < D; e++) s -= Ad[a][e] * fx[e];
          q[a] = s;
        }
        if (D == 3) {
          stage[0][t] = make_float4(Ad[0][0], Ad[0][1], Ad[0][2], Ad[1][0]);
          stage[1][t] = make_float4(Ad[1][1], Ad[1][2], Ad[2][0], Ad[2][1]);
          stage[2][t] = make_float4(Ad[2][2], q[0], q[1], q[2]);
          stage[3][t] = make_float4(fx[0], fx[1], fx[2], mass);
        } else {
          stage[0][t] = make_float4(Ad[0][0], Ad[0][1], Ad[1][0], Ad[1][1]);
          stage[1][t] = make_float4(q[0], q[1], fx[0], fx[1]);
          stage[2][t] = make_float4(mass, 0.0f, 0.0f, 0.0f);
        }
      }
      lds_barrier();

      // ---- phase 2: stable counting sort of the chunk by cell ----
      unsigned long long peers = __ballot(valid);
  #pragma unroll
      for (int bit = 0; bit < (D == 3 ? 6 : 4); bit++) {
        const bool on = (cell >> bit) & 1;
        const unsigned long long bal = __ballot(on);
        peers &= on ? bal : ~bal;
      }
      const int rank = (int)__popcll(peers & lt);
      if (valid && rank == 0) wcnt[wave][cell] = (int)__popcll(peers);
      lds_barrier();
      if (threadIdx.x < 64) {  // one wave: per-cell totals and exclusive scan
        int run = 0;
        if (lane < CELLS) {
  #pragma unroll
          for (int w = 0; w < WAVES; w++) {
            const int cnt = wcnt[w][lane];
            wcnt[w][lane] = run;
            run += cnt;
          }
        }
        int inc = run;
  #pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const int y = __shfl_up(inc, off);
          if (lane >= off) inc += y;
        }
        if (lane < CELLS) {
          ccount[lane] = run;
          cstart[lane] = inc - run;
        }
      }
      lds_barrier();
      if (valid) order[cstart[cell] + wcnt[wave][cell] + rank] = (unsigned char)t;
      lds_barrier();

      // ---- phase 3: cell-major scatter into private tiles ----
      {
        const int my_cell = scatter_cell_of_lane<D>(lane);
        const int sub = wave * GROUPS + lane / CELLS;
        const int lc[3] = {my_cell & 3, (my_cell >> 2) & 3, my_cell >> 4};
        const int cbeg = cstart[my_cell], ccnt = ccount[my_cell];
        float4* tp = ptile[sub];
        cell_scatter<D, SUBS>(sub, ccnt, cbeg, order, stage, lc, tp);
      }
      lds_barrier();
    }  // batches of the chunk

    // ---- phase 4: sum the private tiles, write the node tile ----
    float4* out = tiles + (int64_t)c * TN;
    for (int i = threadIdx.x; i < TN; i += kThreads) {
      float4 acc = ptile[0][i];
#pragma unroll
      for (int sdx = 1; sdx < SUBS; sdx++) {
        const float4 v = ptile[sdx][i];
        acc.x += v.x;
        acc.y += v.y;
        acc.z += v.z;
        acc.w += v.w;
      }
      out[i] = acc;
    }
    lds_barrier();
  }
  // particles outside the window (sorted to the end, frozen) move as they are
  if (ORDER == kOrderMove)
    for (int j = totals[kTotValid] + blockIdx.x * kThreads + threadIdx.x; j < n;
         j += gridDim.x * kThreads) {
      const int p = perm[j];
      for (int w = 0; w < nw; w++) pf_out[(int64_t)w * cap + j] = pf[(int64_t)w * cap + p];
      for (int w = 0; w < L::NI; w++) pi_out[(int64_t)w * cap + j] = pi[(int64_t)w * cap + p];
      perm[j] = j;
    }
}

// ---------------------------------------------------------------------------
// grid operator (mpm_solver.py:586-692)
// ---------------------------------------------------------------------------
// Velocity of the node with index I from its p2g sums (momentum, mass):
// normalisation, gravity (mpm_solver.py:591-595) and the post-processes.
template <int D>
__device__ __forceinline__ float4 node_velocity(const Params& P, const int I[3], float4 sum) {
  float p[3] = {sum.x, sum.y, sum.z};
  if (node_has_mass(sum.w)) {
    const float inv = 1.0f / sum.w;
#pragma unroll
    for (int a = 0; a < D; a++) p[a] = inv * p[a];
#pragma unroll
    for (int a = 0; a < D; a++) p[a] += P.dt * P.gravity[a];
  }
  apply_post<D>(P, I, p);
  return make_float4(p[0], p[1], D == 3 ? p[2] : 0.0f, sum.w);
}

// Bounding-box walls zero the outward velocity components near the domain
// faces (mpm_solver.py:600-616); bit a of the result is set when component a
// of v (before the walls) passes unchanged.
// MODE 0: the grid operator (raw != 0: store the p2g sums unnormalised).
// MODE 1: its adjoint -- the tiles hold the g2p-adjoint scatter vbar; with
// the forward's raw sums (p, m) in grid, write (pbar, mbar) to gbar:
// v = post(p / m + dt g) gives vbar' = post^T(vbar) (apply_post_adjoint:
// walls, planes and spheres), pbar = vbar' / m and
// mbar = -sum_a pbar_a p_a / m.
template <int D, int MODE>
__global__ __launch_bounds__(kThreads) void k_grid_op(const Params* __restrict__ scenes,
                                                      const int* __restrict__ slab,
                                                      const int* __restrict__ active,
                                                      const int* __restrict__ totals,
                                                      const int* __restrict__ pchunk_begin,
                                                      const int* __restrict__ pchunk_cnt,
                                                      const float4* __restrict__ tiles,
                                                      float4* __restrict__ grid, int raw,
                                                      float4* __restrict__ gbar,
                                                      float4* __restrict__ raw_out) {
  constexpr int NPB = Geo<D>::kNodesPerBlock, TN = Geo<D>::kTileNodes;
  // A lane per node, so in 3D a wave per block: its source blocks, chunk
  // ranges and scene are the same for every lane, and a load instruction
  // reads the 16-byte nodes of one tile's rows.  Bound by the chain of
  // dependent loads (block, chunk ranges, tiles) at 1M particles, by the
  // tiles' bytes at 16M.  Eight lanes per node, one per source block, spread
  // every load over eight tiles: 1M 20.0 -> 14.0 us, 16M 211 -> 108 us,
  // use_g2p2g 300k 17.8 -> 12.1 us.
  constexpr int SRC = D == 3 ? 8 : 4;
  constexpr int BPW = 64 / NPB;  // blocks per wave
  const int nact = totals[kTotActive];
  const int lane = threadIdx.x & 63, node = lane % NPB;
  const int l[3] = {node & 3, (node >> 2) & 3, node >> 4};
  constexpr int BPG = kThreads / NPB;  // blocks per workgroup
  for (XcdItems it((nact + BPG - 1) / BPG, INT32_MAX); it.valid(); it.next()) {
    const int w = it.c * (kThreads / 64) + (threadIdx.x >> 6);
    const int blk = D == 3 ? __builtin_amdgcn_readfirstlane(w) : w * BPW + lane / NPB;
    if (blk >= nact) continue;
    const int bid = active[blk];
    int lb[3];
    decode_local<D>(bid, scenes[0], lb);
    const Params& P = scenes[scene_of<D>(lb, slab)];
    if (P.skip) continue;
    int first[SRC], left[SRC], tn[SRC];
#pragma unroll
    for (int src = 0; src < SRC; src++) {  // particle block b - d, d in {0, 1}^D
      const int d[3] = {src & 1, (src >> 1) & 1, src >> 2};
      int q[3];
      bool in = true, reach = true;
      tn[src] = 0;
#pragma unroll
      for (int a = D - 1; a >= 0; a--) {
        q[a] = lb[a] - d[a];
        in &= q[a] >= 0;
        reach &= l[a] + kBlock * d[a] < kTile;
        tn[src] = tn[src] * kTile + l[a] + kBlock * d[a];
      }
      first[src] = left[src] = 0;
      if (in) {
        const int nb = encode_local<D>(q, P);
        first[src] = pchunk_begin[nb];
        left[src] = pchunk_cnt[nb];
      }
      if (!reach) left[src] = 0;
    }
    const float4 sum = sum_tiles<SRC, TN, D>(tiles, first, left, tn);
    const float p[3] = {sum.x, sum.y, sum.z};
    if (MODE == 0 && raw_out) raw_out[(int64_t)bid * NPB + node] = sum;
    if (MODE == 1) {
      const float4 f = grid[(int64_t)bid * NPB + node];
      float pb[3] = {0.0f, 0.0f, 0.0f}, mb = 0.0f;
      if (node_has_mass(f.w)) {
        const float inv = 1.0f / f.w;
        const float pf4[3] = {f.x, f.y, f.z};
        float v[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int a = 0; a < D; a++) v[a] = pf4[a] * inv + P.dt * P.gravity[a];
        int I[3], lbl[3];
        to_local<D>(lb, P, lbl);
#pragma unroll
        for (int a = 0; a < D; a++) I[a] = (lbl[a] + P.blo[a]) * kBlock + l[a];
        float vb[3] = {p[0], p[1], p[2]};
        apply_post_adjoint<D>(P, I, v, vb);
#pragma unroll
        for (int a = 0; a < D; a++) {
          pb[a] = vb[a] * inv;
          mb -= pb[a] * (pf4[a] * inv);
        }
      }
      gbar[(int64_t)bid * NPB + node] = make_float4(pb[0], pb[1], D == 3 ? pb[2] : 0.0f, mb);
      continue;
    }
    float4 out = make_float4(p[0], p[1], D == 3 ? p[2] : 0.0f, sum.w);
    if (!raw) {
      int I[3], lbl[3];
      to_local<D>(lb, P, lbl);
#pragma unroll
      for (int a = 0; a < D; a++) I[a] = (lbl[a] + P.blo[a]) * kBlock + l[a];
      out = node_velocity<D>(P, I, sum);
    }
    grid[(int64_t)bid * NPB + node] = out;
  }
}

// ---------------------------------------------------------------------------
// G2P (mpm_solver.py:694-735)
// ---------------------------------------------------------------------------
// W: minimum waves per SIMD the register allocation must allow (1: no
// constraint, 5 waves at its register count; 6: at most 80 registers, more
// grid-tile gathers in flight where each block holds few particles).
// TILES: the grid operator runs in here.  The workgroup sums the p2g tiles
// that reach its (4+2)^d nodes itself, in k_grid_op's order (bitwise the same
// velocities), instead of reading them from the grid: every node is summed by
// up to 2^d workgroups, out of L2, and a kernel, its launch and the grid's
// round trip through memory go.  Taken up to kOneRound particles in up to
// kFewChunks chunks, that is while the workgroups run at once; substeps with
// the grid operator apart and inside: 2D 20k (143 chunks) 21.5 -> 19.0 us; 3D
// 2000 particles 33.6 -> 31.6, 30k 37.7 -> 34.8, 100k (593 chunks) 43.9 ->
// 41.4, 160k (855) 48.7 -> 45.8, 100k in 1872 chunks 52.4 -> 51.9, but 250k
// 64.2 -> 66.8, and spread thinly 50k in 2975 chunks 60.2 -> 61.5, 100k in 8687
// 138 -> 153, in 2D 20k in 10289 chunks 87.6 -> 94.2.
template <int D, bool Q = false, int W = 1, bool TILES = false>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(W))) void k_g2p(const Params* __restrict__ scenes,
                                                  const int* __restrict__ slab,
                                                  float* __restrict__ pf,
                                                  const int* __restrict__ pi, int64_t cap,
                                                  const int* __restrict__ perm,
                                                  const int4* __restrict__ chunks,
                                                  const int* __restrict__ totals,
                                                  const float4* __restrict__ grid,
                                                  unsigned* __restrict__ maxv,
                                                  const int* __restrict__ step, int stride,
                                                  int* __restrict__ members,
                                                  int* __restrict__ dseg,
                                                  int* __restrict__ count_next,
                                                  int* __restrict__ err,
                                                  float* __restrict__ pf_out, int n,
                                                  const int* __restrict__ pchunk_begin,
                                                  const int* __restrict__ pchunk_cnt,
                                                  const float4* __restrict__ tiles) {
  using L = Layout<D>;
  constexpr int NPB = Geo<D>::kNodesPerBlock, TN = Geo<D>::kTileNodes;
  // grid velocity tile as three float arrays: the per-particle gathers hit
  // fewer LDS bank conflicts than with one float4 per node (29 vs 32 us per
  // 1M-particle substep)
  __shared__ float tile_x[TN], tile_y[TN], tile_z[TN];
  __shared__ float red[kThreads / 64];
  __shared__ int dwcnt[kThreads / 64][32];
  __shared__ int dbase[32];  // particles per direction in the chunk's earlier batches
  __shared__ int dstart[32];
  __shared__ int2 nbr[TILES ? 27 : 1];  // chunk ranges of the neighbouring blocks
  // the particles of the earlier batches: direction | rank << 8, slot
  __shared__ int lcode[kChunkMax - kBatch], lid[kChunkMax - kBatch];
  // Packed, and at six waves, registers decide the occupancy: there the thread's
  // index after the particle part is kept out of the compiler's sight, so that
  // what is computed from it is not held through that part (packed 98 -> 90
  // registers, five waves per SIMD instead of four; 3 to 5 spilled at six -> none;
  // substeps of 778k packed, with the resident workgroups that go with it, 111.5
  // -> 106.9 us, 300k 70.1 -> 67.7, 2M 220.3 -> 215.3).  Computing it again
  // costs the others 1 to 2% (2D 400k 51.4 and 52.5, 3D 1M 129.1 and 130.5).
  constexpr bool TIGHT = D == 3 && (Q || W >= 6);
  const int wave0 = threadIdx.x >> 6, lane0 = threadIdx.x & 63;
  const unsigned long long lt0 = lane0 == 0 ? 0ull : (~0ull >> (64 - lane0));
  float vmax = 0.0f;
  for (XcdItems it(totals[kTotChunks], kSpreadChunks); it.valid(); it.next()) {
    const int c = it.c;
    const int4 ck = chunks[c];
    int lb[3], lbl[3];
    decode_local<D>(ck.x, scenes[0], lb);
    const Params& P = scenes[scene_of<D>(lb, slab)];
    to_local<D>(lb, P, lbl);
    // a skipped scene keeps its particles (and so their blocks) unchanged; its
    // grid was not rebuilt and is not read
    const bool skip = P.skip != 0;
    if (threadIdx.x < 32) dbase[threadIdx.x] = 0;
    if (TILES) {
      constexpr int NB = D == 3 ? 27 : 9, SRC = D == 3 ? 8 : 4;
      if (threadIdx.x < NB) {  // chunk ranges of the blocks lb + {-1, 0, 1}^d
        const int q[3] = {lb[0] - 1 + (int)threadIdx.x % 3, lb[1] - 1 + ((int)threadIdx.x / 3) % 3,
                          D == 3 ? lb[2] - 1 + (int)threadIdx.x / 9 : 0};
        bool ok = true;  // below the window there is no block; above it is lb + 1 at most
#pragma unroll
        for (int a = 0; a < D; a++) ok &= q[a] >= 0;
        int2 r = make_int2(0, 0);
        if (ok) {
          const int nb = encode_local<D>(q, P);
          r = make_int2(pchunk_begin[nb], pchunk_cnt[nb]);
        }
        nbr[threadIdx.x] = r;
      }
      lds_barrier();
      for (int i = skip ? TN : threadIdx.x; i < TN; i += kThreads) {
        const int t[3] = {i % kTile, (i / kTile) % kTile, i / (kTile * kTile)};
        // source block lb + hi - d, hi the node's own block, d in {0, 1}^d;
        // its tile holds the node at l + 4 d
        int first[SRC], left[SRC], tn[SRC];
#pragma unroll
        for (int src = 0; src < SRC; src++) {
          const int d[3] = {src & 1, (src >> 1) & 1, src >> 2};
          int nb = 0;
          bool reach = true;
          tn[src] = 0;
#pragma unroll
          for (int a = D - 1; a >= 0; a--) {
            const int x = (t[a] & (kBlock - 1)) + kBlock * d[a];
            reach &= x < kTile;
            tn[src] = tn[src] * kTile + x;
            nb = nb * 3 + (t[a] >= kBlock ? 1 : 0) - d[a] + 1;
          }
          const int2 r = nbr[nb];
          first[src] = r.x;
          left[src] = reach ? r.y : 0;
        }
        const float4 sum = sum_tiles<SRC, TN, D>(tiles, first, left, tn);
        int I[3];
#pragma unroll
        for (int a = 0; a < D; a++) I[a] = (lbl[a] + P.blo[a]) * kBlock + t[a];
        const float4 g = node_velocity<D>(P, I, sum);
        tile_x[i] = g.x;
        tile_y[i] = g.y;
        tile_z[i] = g.z;
      }
    } else {
      for (int i = skip ? TN : threadIdx.x; i < TN; i += kThreads) {
        const int tl[3] = {i % kTile, (i / kTile) % kTile, i / (kTile * kTile)};
        int q[3], ln[3];
#pragma unroll
        for (int a = 0; a < D; a++) {
          const int hi = tl[a] >= kBlock;
          q[a] = lb[a] + hi;
          ln[a] = tl[a] - kBlock * hi;
        }
        const int gb = encode_local<D>(q, P);
        const int node = D == 3 ? ln[0] + 4 * (ln[1] + 4 * ln[2]) : ln[0] + 4 * ln[1];
        const float4 g = grid[(int64_t)gb * NPB + node];
        tile_x[i] = g.x;
        tile_y[i] = g.y;
        tile_z[i] = g.z;
      }
    }
    lds_barrier();
    int b[3];
#pragma unroll
    for (int a = 0; a < D; a++) b[a] = (lbl[a] + P.blo[a]) * kBlock;
    // one particle per thread, kBatch particles of the chunk at a time
    for (int b0 = ck.y; b0 < ck.z; b0 += kBatch) {
      const int j = b0 + threadIdx.x;
      const bool live = j < ck.z;
      int dir = 13;  // block offset of the particle after advection, (dz+1)*9 + (dy+1)*3 + (dx+1)
      const int p = live ? perm[j] : 0;
      if (live) {
        using PS = Particles<D, Q>;
        const int mat = pi[(int64_t)L::MAT * cap + p];
        float xp[3] = {0.0f, 0.0f, 0.0f}, fx[3], w[3][3];
        int l[3];
        bool inside = true;
        PS::load_x(pf, cap, p, xp);
  #pragma unroll
        for (int a = 0; a < D; a++) {
          int base;
          base_fx(xp[a], P.inv_dx, base, fx[a]);
          bspline(fx[a], w[a]);
          l[a] = base - b[a];
          inside &= (l[a] >= 0) & (l[a] < kBlock);
        }
        // v = sum_o w_o g_o and C = 4 inv_dx sum_o w_o g_o (o - fx)^T
        // (mpm_solver.py:714-721), evaluated through the tensor-product
        // weights w_o = wx[ox] wy[oy] wz[oz]: P_e = sum_o w_o g_o (o_e - fx_e)
        // with the factor (o_e - fx_e) folded into axis e's weights (wd), so
        // C = 4 inv_dx P needs no subtraction of two nearly equal sums.  One
        // pass over the 27 nodes, per-axis partial sums instead of a 3x3 outer
        // product per node.
        float nv[3] = {0.0f, 0.0f, 0.0f}, pe[3][3] = {{0.0f}}, nC[3][3];
        float wd[3][3];
  #pragma unroll
        for (int a = 0; a < 3; a++)
  #pragma unroll
          for (int k = 0; k < 3; k++) wd[a][k] = a < D ? ((float)k - fx[a]) * w[a][k] : 0.0f;
        if (inside && !skip) {
  #pragma unroll
          for (int oz = 0; oz < (D == 3 ? 3 : 1); oz++) {
            float b0[3] = {0.0f, 0.0f, 0.0f}, bx[3] = {0.0f, 0.0f, 0.0f}, by[3] = {0.0f, 0.0f, 0.0f};
  #pragma unroll
            for (int oy = 0; oy < 3; oy++) {
              float a0[3] = {0.0f, 0.0f, 0.0f}, ax[3] = {0.0f, 0.0f, 0.0f};
  #pragma unroll
              for (int ox = 0; ox < 3; ox++) {
                const int node = D == 3 ? (l[0] + ox) + kTile * ((l[1] + oy) + kTile * (l[2] + oz))
                                        : (l[0] + ox) + kTile * (l[1] + oy);
                const float gg[3] = {tile_x[node], tile_y[node], D == 3 ? tile_z[node] : 0.0f};
  #pragma unroll
                for (int c = 0; c < D; c++) {
                  const float g = gg[c];
                  a0[c] += w[0][ox] * g;
                  ax[c] += wd[0][ox] * g;
                }
              }
  #pragma unroll
              for (int c = 0; c < D; c++) {
                b0[c] += w[1][oy] * a0[c];
                bx[c] += w[1][oy] * ax[c];
                by[c] += wd[1][oy] * a0[c];
              }
            }
            const float wz = D == 3 ? w[2][oz] : 1.0f;
  #pragma unroll
            for (int c = 0; c < D; c++) {
              nv[c] += wz * b0[c];
              pe[c][0] += wz * bx[c];
              pe[c][1] += wz * by[c];
              if (D == 3) pe[c][2] += wd[2][oz] * b0[c];
            }
          }
        }
  #pragma unroll
        for (int c = 0; c < D; c++)
  #pragma unroll
          for (int e = 0; e < D; e++) nC[c][e] = P.c4 * pe[c][e];
        float xn[3] = {xp[0], xp[1], xp[2]};
        if (skip) {
        } else if (mat != kStationary) {  // mpm_solver.py:722-724
          PS::store_v(pf_out, cap, p, nv);  // x advances by the stored v
  #pragma unroll
          for (int a = 0; a < D; a++) {
            xn[a] = xp[a] + P.dt * nv[a];
            vmax = fmaxf(vmax, fabsf(nv[a]));
          }
          PS::store_x(pf_out, cap, p, xn);  // xn: the stored x (binned next)
          PS::store_C(pf_out, cap, p, nC);
        } else {
          float vs[3];
          PS::load_v(pf, cap, p, vs);
  #pragma unroll
          for (int a = 0; a < D; a++) {
            const float va = vs[a];
            vmax = fmaxf(vmax, fabsf(va));
            if (!Q && pf_out != pf) {  // out of place: a stationary particle keeps x, v, C
              pf_out[(int64_t)(L::V + a) * cap + p] = va;
              pf_out[(int64_t)(L::X + a) * cap + p] = xp[a];
  #pragma unroll
              for (int e = 0; e < D; e++)
                pf_out[(int64_t)(L::C + a * D + e) * cap + p] = pf[(int64_t)(L::C + a * D + e) * cap + p];
            }
          }
        }
        // block of the new position for the next substep's binning
        // (build_pid, mpm_solver.py:357-361); particles move less than one block
        // per substep under any sane CFL number
        int dd[3] = {0, 0, 0}, q[3] = {0, 0, 0};
        bool near = true;
  #pragma unroll
        for (int a = 0; a < D; a++) {
          int base;
          float f;
          base_fx(xn[a], P.inv_dx, base, f);
          q[a] = (base >> 2) - P.blo[a];  // scene-local block
          dd[a] = q[a] - lbl[a];
          near &= (dd[a] >= -1) & (dd[a] <= 1) & (q[a] >= 0) & (q[a] < P.bnl[a] - 1);
        }
        if (near) {
          dir = (dd[2] + 1) * 9 + (dd[1] + 1) * 3 + (dd[0] + 1);
        } else {
          // left the window (bit 0) or moved more than one block (bit 3): the
          // particle stays binned in its old block and the caller is told
          atomicOr(err, (q[0] < 0 || q[0] >= P.bnl[0] - 1 || q[1] < 0 || q[1] >= P.bnl[1] - 1 ||
                         (D == 3 && (q[2] < 0 || q[2] >= P.bnl[2] - 1)))
                            ? 1
                            : 8);
        }
      }
      if (!members) continue;  // no binning follows from this substep
      int tid = threadIdx.x;
      if (TIGHT) __asm__ volatile("" : "+v"(tid));
      const int wave = TIGHT ? tid >> 6 : wave0, lane = TIGHT ? tid & 63 : lane0;
      // stable rank of the particle among the chunk's particles with the same
      // direction
      if (lane < 32) dwcnt[wave][lane] = 0;  // the wave's own row, in program order
      unsigned long long peers = __ballot(live);
  #pragma unroll
      for (int bit = 0; bit < 5; bit++) {
        const bool on = (dir >> bit) & 1;
        const unsigned long long bal = __ballot(on);
        peers &= on ? bal : ~bal;
      }
      const int rank = TIGHT ? lanes_before(peers) : (int)__popcll(peers & lt0);
      if (live && rank == 0) dwcnt[wave][dir] = (int)__popcll(peers);
      lds_barrier();
      const bool last = b0 + kBatch >= ck.z;
      if (tid < 64) {
        int run = 0;
        if (lane < 27) {
          run = dbase[lane];
  #pragma unroll
          for (int w = 0; w < kThreads / 64; w++) {
            const int cnt = dwcnt[w][lane];
            dwcnt[w][lane] = run;
            run += cnt;
          }
          dbase[lane] = run;
        }
        if (last) write_groups<D>(c, lb, P, run, dstart, dseg, count_next);
      }
      lds_barrier();
      if (live) {
        const int r = dwcnt[wave][dir] + rank;
        if (last) {
          members[ck.y + dstart[dir] + r] = p;
        } else {
          const int i = TIGHT ? b0 - ck.y + tid : j - ck.y;
          lcode[i] = dir | (r << 8);
          lid[i] = p;
        }
      }
      if (last)  // the earlier batches' particles (this thread's own entries)
        for (int i = tid; i < b0 - ck.y; i += kThreads)
          members[ck.y + dstart[lcode[i] & 255] + (lcode[i] >> 8)] = lid[i];
      lds_barrier();
    }  // batches of the chunk
    if (!members) lds_barrier();  // the node tile is rewritten for the next chunk
  }
  // out of place: particles outside every chunk (escaped the window; sorted
  // to the end) keep their whole state
  if (!Q && pf_out != pf) {
    for (int j = totals[kTotValid] + blockIdx.x * kThreads + threadIdx.x; j < n;
         j += gridDim.x * kThreads) {
      const int p = perm[j];
      for (int c = 0; c < L::NF; c++) pf_out[(int64_t)c * cap + p] = pf[(int64_t)c * cap + p];
    }
  }
  // compute_max_velocity (mpm_solver.py:726-735): non-negative floats order
  // like their bit patterns.
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) vmax = fmaxf(vmax, __shfl_xor(vmax, off));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = vmax;
  lds_barrier();
  if (threadIdx.x == 0) {
    float m = red[0];
#pragma unroll
    for (int w = 1; w < kThreads / 64; w++) m = fmaxf(m, red[w]);
    // one partial maximum per workgroup, reduced by the reader: a single
    // device-wide atomic serialised thousands of workgroups
    maxv[(int64_t)(step ? *step : 0) * stride + blockIdx.x] = __float_as_uint(m);
  }
}

// ---------------------------------------------------------------------------
// particle bookkeeping kernels
// ---------------------------------------------------------------------------
// Block keys in sorted order, from the chunks (mpm_read_binning).
__global__ __launch_bounds__(kThreads) void k_sorted_keys(const int4* __restrict__ chunks,
                                                          const int* __restrict__ totals, int n,
                                                          int total_blocks,
                                                          int* __restrict__ keys) {
  for (int c = blockIdx.x; c < totals[kTotChunks]; c += gridDim.x) {
    const int4 ck = chunks[c];
    for (int j = ck.y + threadIdx.x; j < ck.z; j += kThreads) keys[j] = ck.x;
  }
  for (int j = totals[kTotValid] + blockIdx.x * kThreads + threadIdx.x; j < n;
       j += gridDim.x * kThreads)
    keys[j] = total_blocks;
}

// New particles: seed_particle (mpm_solver.py:823-838).
template <int D, bool Q, bool G>
__global__ __launch_bounds__(kThreads) void k_append(const float* __restrict__ x,
                                                     const float* __restrict__ v,
                                                     const int* __restrict__ mat, int k,
                                                     int n_old, int scene, int plastic,
                                                     float* __restrict__ pf,
                                                     int* __restrict__ pi, int64_t cap) {
  using L = Layout<D>;
  using PS = Particles<D, Q, G>;
  const int t = blockIdx.x * kThreads + threadIdx.x;
  if (t >= k) return;
  const int s = n_old + t;
  const int m = mat[t];
  float xs[3] = {0.0f, 0.0f, 0.0f}, vs[3] = {0.0f, 0.0f, 0.0f}, C[3][3], F[3][3];
#pragma unroll
  for (int a = 0; a < D; a++) {
    xs[a] = x[(int64_t)t * D + a];
    vs[a] = v ? v[(int64_t)t * D + a] : 0.0f;
#pragma unroll
    for (int e = 0; e < D; e++) {
      C[a][e] = 0.0f;
      F[a][e] = a == e ? 1.0f : 0.0f;
    }
  }
  PS::store_x(pf, cap, s, xs);
  PS::store_v(pf, cap, s, vs);
  PS::store_C(pf, cap, s, C);
  PS::store_F(pf, cap, s, F);
  if (!Q || plastic) PS::store_Jp(pf, cap, s, m == kSand ? 0.0f : 1.0f);  // mpm_solver.py:831-835
  pi[(int64_t)L::MAT * cap + s] = m;
  pi[(int64_t)L::ORIG * cap + s] = s;
  pi[(int64_t)L::SCENE * cap + s] = scene;
}

template <int D, bool G>
__global__ __launch_bounds__(kThreads) void k_unpack(const float* __restrict__ packed,
                                                     float* __restrict__ flt, int n, int64_t cap,
                                                     int plastic) {
  using PQ = Particles<D, true, G>;
  using PF = Particles<D, false>;
  for (int p = blockIdx.x * kThreads + threadIdx.x; p < n; p += gridDim.x * kThreads) {
    float x[3], v[3], C[3][3], F[3][3];
    PQ::load_x(packed, cap, p, x);
    PQ::load_v(packed, cap, p, v);
    PQ::load_C(packed, cap, p, C);
    PQ::load_F(packed, cap, p, F);
    PF::store_x(flt, cap, p, x);
    PF::store_v(flt, cap, p, v);
    PF::store_C(flt, cap, p, C);
    PF::store_F(flt, cap, p, F);
    PF::store_Jp(flt, cap, p, plastic ? PQ::load_Jp(packed, cap, p) : 1.0f);
  }
}

template <int D, bool G>
__global__ __launch_bounds__(kThreads) void k_pack(const float* __restrict__ flt,
                                                   float* __restrict__ packed, int n, int64_t cap,
                                                   int plastic) {
  using PQ = Particles<D, true, G>;
  using PF = Particles<D, false>;
  for (int p = blockIdx.x * kThreads + threadIdx.x; p < n; p += gridDim.x * kThreads) {
    float x[3], v[3], C[3][3], F[3][3];
    PF::load_x(flt, cap, p, x);
    PF::load_v(flt, cap, p, v);
    PF::load_C(flt, cap, p, C);
    PF::load_F(flt, cap, p, F);
    PQ::store_x(packed, cap, p, x);
    PQ::store_v(packed, cap, p, v);
    PQ::store_C(packed, cap, p, C);
    PQ::store_F(packed, cap, p, F);
    if (plastic) PQ::store_Jp(packed, cap, p, PF::load_Jp(flt, cap, p));
  }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void k_gather(const T* __restrict__ src, int64_t cap,
                                                     int ncomp, const int* __restrict__ orig,
                                                     int n, T* __restrict__ dst) {
  for (int j = blockIdx.x * kThreads + threadIdx.x; j < n; j += gridDim.x * kThreads) {
    const int o = orig[j];
    for (int c = 0; c < ncomp; c++) dst[(int64_t)o * ncomp + c] = src[(int64_t)c * cap + j];
  }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void k_scatter(const T* __restrict__ src, int64_t cap,
                                                      int ncomp, const int* __restrict__ orig,
                                                      int n, T* __restrict__ dst) {
  for (int j = blockIdx.x * kThreads + threadIdx.x; j < n; j += gridDim.x * kThreads) {
    const int o = orig[j];
    for (int c = 0; c < ncomp; c++) dst[(int64_t)c * cap + j] = src[(int64_t)o * ncomp + c];
  }
}

// particle_info (mpm_solver.py:1172-1191): x, v (n, D) and material in
// insertion order, from either layout (null: not wanted).
template <int D, bool Q, bool G>
__global__ __launch_bounds__(kThreads) void k_particle_info(const float* __restrict__ pf,
                                                            const int* __restrict__ pi,
                                                            int64_t cap, int n,
                                                            float* __restrict__ x,
                                                            float* __restrict__ v,
                                                            int* __restrict__ mat) {
  using L = Layout<D>;
  using PS = Particles<D, Q, G>;
  for (int j = blockIdx.x * kThreads + threadIdx.x; j < n; j += gridDim.x * kThreads) {
    const int64_t o = pi[(int64_t)L::ORIG * cap + j];
    float a[3];
    if (x) {
      PS::load_x(pf, cap, j, a);
#pragma unroll
      for (int c = 0; c < D; c++) x[o * D + c] = a[c];
    }
    if (v) {
      PS::load_v(pf, cap, j, a);
#pragma unroll
      for (int c = 0; c < D; c++) v[o * D + c] = a[c];
    }
    if (mat) mat[o] = pi[(int64_t)L::MAT * cap + j];
  }
}

// Largest |v| of each substep (one workgroup) from its per-workgroup maxima
// (float bits); the last workgroup copies the error bits and the number of
// chunks behind them.  out is pinned host memory.
__global__ __launch_bounds__(kThreads) void k_max_rows(const unsigned* __restrict__ part,
                                                       int stride, const int* __restrict__ err,
                                                       const int* __restrict__ totals,
                                                       unsigned* __restrict__ out) {
  if (blockIdx.x == gridDim.x - 1) {
    if (threadIdx.x == 0) {
      out[blockIdx.x] = (unsigned)*err;
      out[blockIdx.x + 1] = (unsigned)totals[kTotChunks];
    }
    return;
  }
  __shared__ unsigned red[kThreads / 64];
  unsigned m = 0;
  for (int i = threadIdx.x; i < stride; i += kThreads)
    m = max(m, part[(int64_t)blockIdx.x * stride + i]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, off));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kThreads / 64; w++) m = max(m, red[w]);
    out[blockIdx.x] = m;
  }
}

__global__ __launch_bounds__(kThreads) void k_copy_segments(CopySegments S) {
  for (int s = 0; s < S.count; s++)
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < S.n[s];
         i += (int64_t)gridDim.x * kThreads)
      S.dst[s][i] = S.src[s][i];
}

// dst[r][i] = src[r][index[i]]: a particle state into or out of the sorted
// order, and its gradient back.  Bound by the gathered four-byte reads, each
// of a cache line of its own when the two orders have nothing in common, so
// the rows are dealt out to the XCDs (workgroups go round-robin over them):
// each row's lines are fetched into one L2 and reused there by its other
// columns.  The last rows % 8 rows are shared by all.  Against torch's
// indexing: state and E in and the state out (25 + 1 + 25 rows of 200k) 110 ->
// 49 us; the backward of the same at 150k, which sorted the indices, 420 -> 38.
__global__ __launch_bounds__(kThreads) void k_take_columns(
    const float* __restrict__ src, int64_t row_stride, int64_t col_stride,
    const int64_t* __restrict__ index, float* __restrict__ dst, int rows, int64_t n) {
  constexpr int X = XcdItems::kXcds;
  const int own = rows / X * X;
  const int64_t step = (int64_t)(gridDim.x / X) * kThreads;
  for (int64_t i = (int64_t)(blockIdx.x / X) * kThreads + threadIdx.x; i < n; i += step) {
    const float* s = src + index[i] * col_stride;
#pragma unroll 4
    for (int r = blockIdx.x % X; r < own; r += X) dst[r * n + i] = s[r * row_stride];
  }
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kThreads) {
    const float* s = src + index[i] * col_stride;
    for (int r = own; r < rows; r++) dst[r * n + i] = s[r * row_stride];
  }
}

// Start of a call of substeps: the scene table out of pinned host memory, the
// max-velocity slots cleared, the substep counter before its first slot.  One
// launch in place of two fills and a copy, 10 us of a call on the device.
__global__ __launch_bounds__(kThreads) void k_begin_call(const unsigned* __restrict__ host_table,
                                                         unsigned* __restrict__ table, int words,
                                                         unsigned* __restrict__ maxv, int64_t n,
                                                         int* __restrict__ step) {
  const int64_t first = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * kThreads;
  for (int64_t i = first; i < words; i += stride) table[i] = host_table[i];
  for (int64_t i = first; i < n; i += stride) maxv[i] = 0u;
  if (first == 0) *step = -1;
}

__global__ __launch_bounds__(kThreads) void k_fill_u32(unsigned* __restrict__ p, unsigned v,
                                                       int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kThreads)
    p[i] = v;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static inline int div_up(int64_t a, int64_t b) { return (int)((a + b - 1) / b); }
static inline int clamp_groups(int64_t g, int cap) {
  return (int)std::max<int64_t>(1, std::min<int64_t>(g, cap));
}
// the same, a multiple of the eight XCDs (XcdItems)
static inline int xcd_groups(int64_t g, int cap) {
  return (int)std::min<int64_t>((std::max<int64_t>(g, 1) + 7) & ~7, cap & ~7);
}

// Workgroups of a kernel that the device holds at once.
static int resident_groups(const void* kern) {
  static std::mutex mu;
  static std::map<const void*, int> known;
  std::lock_guard<std::mutex> lock(mu);
  const auto it = known.find(kern);
  if (it != known.end()) return it->second;
  int dev = 0, cus = 0, per_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kThreads, 0) != hipSuccess ||
      cus * per_cu < 8) {
    (void)hipGetLastError();
    return 1024;
  }
  return known[kern] = cus * per_cu;
}

// Workgroups of the grid operators: a lane per node of the active blocks (at
// most the window's, and 2^D per particle), as many as are resident at once.
template <int D>
static int grid_op_groups(const SubstepBuffers& B) {
  const int64_t blocks = std::min<int64_t>(B.total_blocks, (int64_t)B.n * (D == 3 ? 8 : 4));
  return xcd_groups(div_up(blocks * Geo<D>::kNodesPerBlock, kThreads), 2048);
}

struct TimerScope {
  Timer* t;
  hipStream_t st;
  TimerScope(Timer* t_, const char* name, hipStream_t s) : t(t_), st(s) {
    if (t) t->begin(name, st);
  }
  ~TimerScope() {
    if (t) t->end(st);
  }
};

// The previous substep's direction lists.
static PrevBinning prev_binning(const SubstepBuffers& B) {
  PrevBinning p{};
  p.pchunk_begin = B.pchunk_begin_prev;
  p.pchunk_cnt = B.pchunk_cnt_prev;
  p.chunks = B.chunks_prev;
  p.dseg = B.dseg_prev;
  p.members = B.members_prev;
  return p;
}

// Whether the transfer walks the direction lists itself (mpm_binning.h says
// what each way costs).  A substep that moves the particles takes the given
// order.
static bool order_in_transfer(const SubstepBuffers& B) {
  return !B.full_sort && !B.move && B.few_chunks &&
         B.n <= (B.g2p2g ? kOneRound : kListsInTransfer);
}

// Whether p2g scans the block window itself (WindowScan says why there).  Its
// division by the chunk size is a multiplication by ceil(2^32 / chunk), which
// for chunks of one particle does not fit 32 bits: those take k_bscan.
template <int D>
static bool scan_in_p2g(const SubstepBuffers& B) {
  return D == 2 && order_in_transfer(B) && !B.g2p2g && B.chunk > 1 &&
         B.total_blocks <= kThreads * kWindowItems;
}

// binning of one substep: block counts, the dense-window scan (chunks,
// active blocks) and the sorted order
template <int D>
static void launch_binning(const Params* P, SubstepBuffers& B, hipStream_t st, Timer* tm) {
  const int n = B.n;
  if (n == 0) return;
  const int nparts = div_up(B.total_blocks, kScanTile);
  const int passes = (B.key_bits + 7) / 8;
  int* ghist = B.ghist + (B.parity & 1) * kMaxRadixPasses * kRadixBins;
  int* ghist_next = B.ghist + ((B.parity & 1) ^ 1) * kMaxRadixPasses * kRadixBins;
  if (B.full_sort) {
    // first substep (or positions changed from the host): block counts from
    // scratch, then a stable radix sort of the slots
    TimerScope ts(tm, "k_keys", st);
    if (!B.count_zeroed) launch_fill_u32((unsigned*)B.count, 0u, B.total_blocks + 1, st);
    if (B.quant)
      k_keys<D, true><<<clamp_groups(div_up(n, kThreads), 8192), kThreads, 0, st>>>(
          P, B.pf, B.pi, B.cap, n, B.total_blocks, B.keys, B.count, B.err);
    else
      k_keys<D, false><<<clamp_groups(div_up(n, kThreads), 8192), kThreads, 0, st>>>(
          P, B.pf, B.pi, B.cap, n, B.total_blocks, B.keys, B.count, B.err);
  }
  if (!scan_in_p2g<D>(B)) {
    TimerScope ts(tm, "k_bscan", st);
    const bool two_level = nparts > kScanTilesOnePass;
    int4* group_sums = two_level ? reinterpret_cast<int4*>(B.scan_status) : nullptr;
    if (two_level) {
      k_bscan_reduce<D><<<nparts, kThreads, 0, st>>>(P, B.count, B.total_blocks, B.chunk,
                                                     B.tile_sums, group_sums);
    }
    k_bscan<D><<<nparts, kThreads, 0, st>>>(
        P, B.count, B.count_next, B.total_blocks, B.chunk, nparts, B.full_sort ? passes : 0,
        B.pstart, B.pchunk_begin, B.pchunk_cnt, B.chunks, B.active, B.totals, ghist, ghist_next,
        B.scan_status, two_level ? B.tile_sums : nullptr, group_sums, B.err, B.step);
  }
  if (B.full_sort) {
    TimerScope ts(tm, "k_radix", st);
    const int small = div_up(n, kRadixSmallTile);
    const bool use_small = small <= kRadixSmallTiles && small <= B.radix_cap;
    const int ntiles = use_small ? small : div_up(n, kRadixTile);
    auto kern = use_small ? k_onesweep<kRadixSmallItems> : k_onesweep<kRadixItems>;
    const int* kin = B.keys;
    const int* vin = nullptr;
    int* kbuf[2] = {B.keys_alt, B.keys_alt + B.cap};
    int* vbuf[2] = {B.perm, B.perm_alt};
    for (int pass = 0; pass < passes; pass++) {
      kern<<<ntiles, kThreads, 0, st>>>(kin, vin, kbuf[pass & 1], vbuf[pass & 1], n,
                                               pass * 8, ntiles, ghist + pass * kRadixBins,
                                               B.lb_status_radix, B.lbs, B.err);
      kin = kbuf[pass & 1];
      vin = vbuf[pass & 1];
    }
    if (vin != B.perm) std::swap(B.perm, B.perm_alt);
  } else if (!order_in_transfer(B)) {
    TimerScope ts(tm, "k_members", st);
    const int chunk_bound = std::min(B.total_blocks, n) + div_up(n, B.chunk);
    k_members<D><<<clamp_groups(div_up(chunk_bound, kThreads / 64), 4096), kThreads, 0, st>>>(
        P, B.chunks, B.totals, B.pstart, prev_binning(B), B.perm, B.err);
  }
}

// The block scan's published tile sums, or the group sums of a larger window
// (in the same array, two words each), for the transfer after it to clear.
static ScanStatus scan_status(const SubstepBuffers& B) {
  const int tiles = div_up(B.total_blocks, kScanTile);
  return {B.scan_status, tiles <= kScanTilesOnePass ? 4 * tiles : 2 * div_up(tiles, kScanGroup)};
}

static WindowScan window_scan(const SubstepBuffers& B) {
  const unsigned inv = (unsigned)(((1ull << 32) + B.chunk - 1) / B.chunk);
  return {B.count, B.count_next, B.total_blocks, B.chunk, inv, B.pstart, B.pchunk_begin,
          B.pchunk_cnt, B.chunks, B.active, B.totals,
          B.ghist + ((B.parity & 1) ^ 1) * kMaxRadixPasses * kRadixBins, B.step};
}

// The slots were rewritten in sorted order by the transfer just launched.
static void take_moved(SubstepBuffers& B) {
  std::swap(B.pf, B.pf_alt);
  std::swap(B.pi, B.pi_alt);
  B.pf_out = B.pf;
  B.move = false;
}

// binning, p2g and the grid operator of one substep
template <int D>
void launch_front(const Params* P, const int* slab, SubstepBuffers& B, int raw, hipStream_t st,
                  Timer* tm) {
  launch_binning<D>(P, B, st, tm);
  launch_transfer<D>(P, slab, B, raw, st, tm);
}

// one substep of the use_g2p2g mode: binning, the fused transfer from
// B.grid_in, and the grid operator into B.grid
template <int D>
static void launch_g2p2g(const Params* P, const int* slab, SubstepBuffers& B, int s_index,
                         hipStream_t st, Timer* tm) {
  const int n = B.n;
  const int G = B.persistent_groups;
  if (n == 0) return;
  launch_binning<D>(P, B, st, tm);
  const int chunk_bound = std::min(B.total_blocks, n) + div_up(n, B.chunk);
  {
    TimerScope ts(tm, "k_g2p2g", st);
    auto kern = B.quant ? k_g2p2g<D, true> : k_g2p2g<D, false>;
    if (order_in_transfer(B))
      kern = B.quant ? k_g2p2g<D, true, kOrderLists> : k_g2p2g<D, false, kOrderLists>;
    if (B.move) kern = B.quant ? k_g2p2g<D, true, kOrderMove> : k_g2p2g<D, false, kOrderMove>;
    // In 3D no more workgroups than are resident at once (three per CU, by LDS)
    // while each takes a few chunks: the rest would start in a second, uneven
    // round (2048 and 768: 300k 68.4 and 66.3 us a substep, 600k thinly spread
    // 101.8 and 98.7, 1M 132.3 and 132.6, with 4096 asked for 134 and 137).
    const int resident = D == 3 && n <= 768 * 1024 ? std::min(G, 768) : G;
    kern<<<xcd_groups(chunk_bound, resident), kThreads, 0, st>>>(
        P, slab, B.pf, B.pi, B.cap, B.perm, B.chunks, B.totals, B.grid_in, B.tiles, B.n_final,
        B.maxv, B.step, B.persistent_groups, B.members, B.dseg, B.count_next, B.err,
        prev_binning(B), B.pstart, B.move ? B.pf_alt : B.pf, B.move ? B.pi_alt : nullptr, n, B.nw,
        scan_status(B));
    if (B.move) take_moved(B);
  }
  {
    TimerScope ts(tm, "k_grid_op", st);
    k_grid_op_g2p2g<D><<<grid_op_groups<D>(B), kThreads, 0, st>>>(
        P, slab, B.active, B.totals, B.pchunk_begin, B.pchunk_cnt, B.tiles, B.grid);
  }
  std::swap(B.count, B.count_next);
}

template <int D>
void launch_grid_op(const Params* P, const int* slab, const SubstepBuffers& B, int raw,
                    hipStream_t st, Timer* tm) {
  TimerScope ts(tm, "k_grid_op", st);
  k_grid_op<D, 0><<<grid_op_groups<D>(B), kThreads, 0, st>>>(
      P, slab, B.active, B.totals, B.pchunk_begin, B.pchunk_cnt, B.tiles, B.grid, raw, nullptr,
      B.raw_out);
}

// p2g and the grid operator on an existing binning
template <int D>
void launch_transfer(const Params* P, const int* slab, SubstepBuffers& B, int raw, hipStream_t st,
                     Timer* tm) {
  const int n = B.n;
  const int G = B.persistent_groups;
  if (n == 0) return;
  const int chunk_bound = std::min(B.total_blocks, n) + div_up(n, B.chunk);
  {
    TimerScope ts(tm, "k_p2g", st);
    auto kern = B.quant ? k_p2g<D, 0, true> : k_p2g<D, 0, false>;
    if (order_in_transfer(B))
      kern = B.quant ? k_p2g<D, 0, true, kOrderLists> : k_p2g<D, 0, false, kOrderLists>;
    // Past kOneRound particles four times the workgroups of the other transfer:
    // with one or two chunks each, the hardware evens out chunks that differ by
    // material and size, and p2g has little to set up per workgroup (2048 and
    // 8192: 1M 74.6 and 72.5 us, 2D 400k 21.2 and 19.4, a batch of 1.1M 86.5
    // and 82.4, 16M 1258 and 1219).
    int groups = xcd_groups(chunk_bound, n > kOneRound ? 4 * G : G);
    if constexpr (D == 2)
      if (scan_in_p2g<D>(B)) {
        groups = std::min(groups, kWindowGroups);
        kern = B.quant ? k_p2g<D, 0, true, kOrderLists, true> : k_p2g<D, 0, false, kOrderLists, true>;
      }
    if (B.move) kern = B.quant ? k_p2g<D, 0, true, kOrderMove> : k_p2g<D, 0, false, kOrderMove>;
    kern<<<groups, kThreads, 0, st>>>(
        P, slab, B.pf, B.pi, B.cap, B.perm, B.chunks, B.totals, B.tiles, nullptr,
        B.move ? B.pf_alt : B.pf_out, prev_binning(B), B.pstart, B.move ? B.pi_alt : nullptr, n,
        B.nw, B.err, scan_status(B), window_scan(B));
    if (B.move) take_moved(B);
  }
  if (!B.grid_in_g2p) launch_grid_op<D>(P, slab, B, raw, st, tm);
}

// g2p of one substep (after launch_front); the max-velocity slot is the
// device substep counter B.step (s_index is kept for the interface)
template <int D>
void launch_g2p(const Params* P, const int* slab, SubstepBuffers& B, int s_index, hipStream_t st,
                Timer* tm) {
  const int n = B.n;
  const int G = B.persistent_groups;
  if (n == 0) return;
  const int chunk_bound = std::min(B.total_blocks, n) + div_up(n, B.chunk);
  {
    TimerScope ts(tm, "k_g2p", st);
    auto kern = B.g2p_waves >= 6 ? (B.quant ? k_g2p<D, true, 6> : k_g2p<D, false, 6>)
                                 : (B.quant ? k_g2p<D, true, 1> : k_g2p<D, false, 1>);
    if (B.grid_in_g2p) kern = B.quant ? k_g2p<D, true, 1, true> : k_g2p<D, false, 1, true>;
    // In 3D no more workgroups than are resident at once (1280): with more, the
    // ones that start in a second round leave the device uneven (2048 and 1280:
    // substeps of 300k 66.6 and 65.0 us, 1M 117.5 and 116.3, 4M 419 and 405; 16M
    // g2p 645 and 568; packed 778k 109.9 and 106.9).  No gain in 2D (60.8 and 61.8
    // us at 400k).
    const int resident = D == 2 || B.grid_in_g2p
                             ? G
                             : std::min(G, resident_groups((const void*)kern));
    kern<<<xcd_groups(chunk_bound, resident), kThreads, 0, st>>>(
        P, slab, B.pf, B.pi, B.cap, B.perm, B.chunks, B.totals, B.grid,
        B.maxv, B.step, B.persistent_groups, B.members, B.dseg, B.count_next, B.err,
        B.pf_out, n, B.pchunk_begin, B.pchunk_cnt, B.tiles);
  }
  std::swap(B.count, B.count_next);
}

template <int D>
void launch_substep(const Params* P, const int* slab, SubstepBuffers& B, int s_index, int raw,
                    hipStream_t st, Timer* tm) {
  if (B.g2p2g) {
    launch_g2p2g<D>(P, slab, B, s_index, st, tm);
    return;
  }
  launch_front<D>(P, slab, B, raw, st, tm);
  launch_g2p<D>(P, slab, B, s_index, st, tm);
}

template <int D>
void launch_substep_half(const Params* P, const int* slab, SubstepBuffers& B, int s_index,
                         int half, hipStream_t st, Timer* tm) {
  if (B.g2p2g) {
    if (half == 0) launch_g2p2g<D>(P, slab, B, s_index, st, tm);
    return;
  }
  if (half == 0)
    launch_front<D>(P, slab, B, 0, st, tm);
  else
    launch_g2p<D>(P, slab, B, s_index, st, tm);
}

template <int D>
void launch_adjoint(const Params* P, const int* slab, SubstepBuffers& B, const float* pf_in,
                    const float* gout, float* gin, float* gE, float4* gbar,
                    float* nu_part, float* gnu, hipStream_t st, Timer* tm) {
  const int n = B.n;
  const int G = B.persistent_groups;
  const int chunk_bound = n > 0 ? std::min(B.total_blocks, n) + div_up(n, B.chunk) : 1;
  const int groups = xcd_groups(chunk_bound, G);
  if (n > 0) {
    {
      TimerScope ts(tm, "k_g2p_adj_scatter", st);
      k_p2g<D, 1><<<groups, kThreads, 0, st>>>(P, slab, pf_in, B.pi, B.cap, B.perm, B.chunks,
                                               B.totals, B.tiles, gout, nullptr, PrevBinning{},
                                               nullptr, nullptr, n, 0, nullptr, ScanStatus{},
                                               WindowScan{});
    }
    {
      TimerScope ts(tm, "k_grid_op_adj", st);
      k_grid_op<D, 1><<<grid_op_groups<D>(B), kThreads, 0, st>>>(
          P, slab, B.active, B.totals, B.pchunk_begin, B.pchunk_cnt, B.tiles, B.grid, 0, gbar,
          nullptr);
    }
    {
      TimerScope ts(tm, "k_p2g_adj", st);
      k_p2g_adj<D><<<groups, kThreads, 0, st>>>(P, slab, pf_in, B.pi, B.cap, B.perm, B.chunks,
                                                B.totals, B.grid, gbar, gout, gin, gE, nu_part, n);
    }
  } else {
    launch_fill_u32((unsigned*)nu_part, 0u, groups, st);
  }
  k_sum_partials<<<1, kThreads, 0, st>>>(nu_part, groups, gnu);
}

void launch_sorted_keys(const int4* chunks, const int* totals, int n, int total_blocks, int* keys,
                        hipStream_t st) {
  if (n > 0)
    k_sorted_keys<<<clamp_groups(div_up(n, kThreads), 2048), kThreads, 0, st>>>(
        chunks, totals, n, total_blocks, keys);
}

template <int D>
void launch_append(SubstepBuffers& B, const float* x, const float* v, const int* mat, int k,
                   int n_old, int scene, int plastic, hipStream_t st) {
  if (k <= 0) return;
  const int g = div_up(k, kThreads);
  if (!B.quant)
    k_append<D, false, false><<<g, kThreads, 0, st>>>(x, v, mat, k, n_old, scene, plastic, B.pf,
                                                       B.pi, B.cap);
  else if (B.g2p2g)
    k_append<D, true, true><<<g, kThreads, 0, st>>>(x, v, mat, k, n_old, scene, plastic, B.pf,
                                                     B.pi, B.cap);
  else
    k_append<D, true, false><<<g, kThreads, 0, st>>>(x, v, mat, k, n_old, scene, plastic, B.pf,
                                                      B.pi, B.cap);
}

template <int D>
void launch_unpack(const float* packed, float* flt, int n, int64_t cap, bool g2p2g, bool plastic,
                   hipStream_t st) {
  if (n <= 0) return;
  const int g = clamp_groups(div_up(n, kThreads), 8192);
  if (g2p2g)
    k_unpack<D, true><<<g, kThreads, 0, st>>>(packed, flt, n, cap, plastic);
  else
    k_unpack<D, false><<<g, kThreads, 0, st>>>(packed, flt, n, cap, plastic);
}

template <int D>
void launch_pack(const float* flt, float* packed, int n, int64_t cap, bool g2p2g, bool plastic,
                 hipStream_t st) {
  if (n <= 0) return;
  const int g = clamp_groups(div_up(n, kThreads), 8192);
  if (g2p2g)
    k_pack<D, true><<<g, kThreads, 0, st>>>(flt, packed, n, cap, plastic);
  else
    k_pack<D, false><<<g, kThreads, 0, st>>>(flt, packed, n, cap, plastic);
}

void launch_gather_f(const float* src, int64_t cap, int ncomp, const int* orig, int n,
                     float* dst, hipStream_t st) {
  if (n > 0)
    k_gather<float><<<clamp_groups(div_up(n, kThreads), 8192), kThreads, 0, st>>>(src, cap, ncomp,
                                                                                 orig, n, dst);
}
void launch_gather_i(const int* src, int64_t cap, int ncomp, const int* orig, int n, int* dst,
                     hipStream_t st) {
  if (n > 0)
    k_gather<int><<<clamp_groups(div_up(n, kThreads), 8192), kThreads, 0, st>>>(src, cap, ncomp,
                                                                             orig, n, dst);
}
void launch_scatter_f(const float* src, int64_t cap, int ncomp, const int* orig, int n,
                      float* dst, hipStream_t st) {
  if (n > 0)
    k_scatter<float><<<clamp_groups(div_up(n, kThreads), 8192), kThreads, 0, st>>>(src, cap, ncomp,
                                                                                  orig, n, dst);
}
void launch_scatter_i(const int* src, int64_t cap, int ncomp, const int* orig, int n, int* dst,
                      hipStream_t st) {
  if (n > 0)
    k_scatter<int><<<clamp_groups(div_up(n, kThreads), 8192), kThreads, 0, st>>>(src, cap, ncomp,
                                                                              orig, n, dst);
}
void launch_particle_info(int D, bool quant, bool g2p2g, const float* pf, const int* pi,
                          int64_t cap, int n, float* x, float* v, int* mat, hipStream_t st) {
  if (n <= 0) return;
  auto kern = D == 3 ? (quant ? (g2p2g ? k_particle_info<3, true, true> : k_particle_info<3, true, false>)
                              : k_particle_info<3, false, false>)
                     : (quant ? (g2p2g ? k_particle_info<2, true, true> : k_particle_info<2, true, false>)
                              : k_particle_info<2, false, false>);
  kern<<<clamp_groups(div_up(n, kThreads), 8192), kThreads, 0, st>>>(pf, pi, cap, n, x, v, mat);
}
void launch_max_rows(const unsigned* part, int rows, int stride, const int* err,
                     const int* totals, unsigned* out, hipStream_t st) {
  k_max_rows<<<rows + 1, kThreads, 0, st>>>(part, stride, err, totals, out);
}
void launch_copy_segments(const CopySegments& S, hipStream_t st) {
  int64_t most = 0;
  for (int s = 0; s < S.count; s++) most = std::max(most, S.n[s]);
  if (most > 0)
    k_copy_segments<<<clamp_groups(div_up(most, kThreads), 2048), kThreads, 0, st>>>(S);
}
void launch_begin_call(const Params* host_table, Params* table, int scenes, unsigned* maxv,
                       int64_t n, int* step, hipStream_t st) {
  static_assert(sizeof(Params) % sizeof(unsigned) == 0, "copied by words");
  const int words = (int)(sizeof(Params) / sizeof(unsigned)) * scenes;
  k_begin_call<<<clamp_groups(div_up(std::max<int64_t>(n, words), kThreads), 1024), kThreads, 0,
                 st>>>(reinterpret_cast<const unsigned*>(host_table),
                       reinterpret_cast<unsigned*>(table), words, maxv, n, step);
}
void launch_take_columns(const float* src, int64_t row_stride, int64_t col_stride,
                         const int64_t* index, float* dst, int rows, int64_t n, hipStream_t st) {
  if (n > 0 && rows > 0)
    k_take_columns<<<XcdItems::kXcds * clamp_groups(div_up(n, kThreads), 1024), kThreads, 0, st>>>(
        src, row_stride, col_stride, index, dst, rows, n);
}

// The device SVD (svd3 / svd2, the replacement of ti.svd) on n matrices,
// for tests: A, U, V (n, dim, dim) row-major, sig (n, dim).
__global__ __launch_bounds__(kThreads) void k_svd_batch(int dim, const float* __restrict__ A,
                                                        float* __restrict__ U,
                                                        float* __restrict__ sig,
                                                        float* __restrict__ V, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kThreads) {
    float a[3][3] = {{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}};
    float u[3][3], v[3][3], s3[3] = {0.0f, 0.0f, 0.0f};
    const int dd = dim * dim;
    for (int r = 0; r < dim; r++)
      for (int c = 0; c < dim; c++) a[r][c] = A[i * dd + r * dim + c];
    if (dim == 3)
      svd3(a, u, s3, v);
    else
      svd2(a, u, s3, v);
    for (int r = 0; r < dim; r++) {
      sig[i * dim + r] = s3[r];
      for (int c = 0; c < dim; c++) {
        U[i * dd + r * dim + c] = u[r][c];
        V[i * dd + r * dim + c] = v[r][c];
      }
    }
  }
}

void launch_svd_batch(int dim, const float* A, float* U, float* sig, float* V, int64_t n,
                      hipStream_t st) {
  if (n > 0)
    k_svd_batch<<<clamp_groups(div_up(n, kThreads), 4096), kThreads, 0, st>>>(dim, A, U, sig, V,
                                                                            n);
}

void launch_fill_u32(unsigned* p, unsigned v, int64_t n, hipStream_t st) {
  if (n > 0)
    k_fill_u32<<<clamp_groups(div_up(n, kThreads), 4096), kThreads, 0, st>>>(p, v, n);
}

// Per-workgroup bounding box of the particle positions: partial[g * 6 + 2a]
// = min, partial[g * 6 + 2a + 1] = max of x_a (workgroup g).
template <int D, bool Q>
__global__ __launch_bounds__(kThreads) void k_aabb(const float* __restrict__ pf, int64_t cap,
                                                   int n, float* __restrict__ partial) {
  __shared__ float red[kThreads / 64][6];
  float lo[3] = {3.4e38f, 3.4e38f, 3.4e38f}, hi[3] = {-3.4e38f, -3.4e38f, -3.4e38f};
  for (int p = blockIdx.x * kThreads + threadIdx.x; p < n; p += gridDim.x * kThreads) {
    float x[3] = {0.0f, 0.0f, 0.0f};
    Particles<D, Q>::load_x(pf, cap, p, x);
#pragma unroll
    for (int a = 0; a < D; a++) {
      lo[a] = fminf(lo[a], x[a]);
      hi[a] = fmaxf(hi[a], x[a]);
    }
  }
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      lo[a] = fminf(lo[a], __shfl_xor(lo[a], off));
      hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], off));
    }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int a = 0; a < 3; a++) {
      red[wave][2 * a] = lo[a];
      red[wave][2 * a + 1] = hi[a];
    }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int c = threadIdx.x;
    float v = red[0][c];
#pragma unroll
    for (int w = 1; w < kThreads / 64; w++) v = (c & 1) ? fmaxf(v, red[w][c]) : fminf(v, red[w][c]);
    partial[(int64_t)blockIdx.x * 6 + c] = v;
  }
}

void launch_aabb(int D, bool quant, const float* pf, int64_t cap, int n, float* partial,
                 int groups, hipStream_t st) {
  if (D == 3)
    (quant ? k_aabb<3, true> : k_aabb<3, false>)<<<groups, kThreads, 0, st>>>(pf, cap, n, partial);
  else
    (quant ? k_aabb<2, true> : k_aabb<2, false>)<<<groups, kThreads, 0, st>>>(pf, cap, n, partial);
}

// Grid contents carried into a moved block window: node i of new block b
// takes node i of the same global block in the old window, or zero.
__global__ __launch_bounds__(kThreads) void k_remap_grid(const float4* __restrict__ old_grid,
                                                         float4* __restrict__ new_grid,
                                                         WindowMap m, int64_t nodes, int npb) {
  for (int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x; t < nodes;
       t += (int64_t)gridDim.x * kThreads) {
    const int64_t b = t / npb;
    const int node = (int)(t % npb);
    int64_t r = b;
    int64_t ob = 0, stride = 1;
    bool in = true;
    for (int a = 0; a < 3; a++) {
      const int c = (int)(r % m.new_bn[a]);
      r /= m.new_bn[a];
      const int oc = c + m.new_blo[a] - m.old_blo[a];
      in &= (oc >= 0) & (oc < m.old_bn[a]);
      ob += (int64_t)oc * stride;
      stride *= m.old_bn[a];
    }
    new_grid[t] = in ? old_grid[ob * npb + node] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
}

void launch_remap_grid(const float4* old_grid, float4* new_grid, const WindowMap& m,
                       int64_t nodes, int npb, hipStream_t st) {
  if (nodes > 0)
    k_remap_grid<<<clamp_groups(div_up(nodes, kThreads), 8192), kThreads, 0, st>>>(
        old_grid, new_grid, m, nodes, npb);
}

// compute_max_grid_velocity (mpm_solver.py:737-746): the largest velocity
// component magnitude on the grid after the last grid operator.  Nodes of
// active blocks without mass hold zero velocity, as the reference's
// freshly activated nodes do.  Non-negative floats order like their bits.
template <int D>
__global__ __launch_bounds__(kThreads) void k_grid_vmax(const float4* __restrict__ grid,
                                                        const int* __restrict__ active,
                                                        const int* __restrict__ totals,
                                                        unsigned* __restrict__ out) {
  constexpr int NPB = Geo<D>::kNodesPerBlock;
  const int64_t nodes = (int64_t)totals[kTotActive] * NPB;
  float m = 0.0f;
  for (int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x; t < nodes;
       t += (int64_t)gridDim.x * kThreads) {
    const float4 g = grid[(int64_t)active[t / NPB] * NPB + t % NPB];
    m = fmaxf(m, fmaxf(fabsf(g.x), fabsf(g.y)));
    if (D == 3) m = fmaxf(m, fabsf(g.z));
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  if ((threadIdx.x & 63) == 0) atomicMax(out, __float_as_uint(m));
}

void launch_grid_vmax(int D, const float4* grid, const int* active, const int* totals,
                      int64_t total_blocks, unsigned* out, hipStream_t st) {
  launch_fill_u32(out, 0u, 1, st);
  const int npb = D == 3 ? Geo<3>::kNodesPerBlock : Geo<2>::kNodesPerBlock;
  const int groups = clamp_groups(div_up(total_blocks * npb, kThreads), 2048);
  if (D == 3)
    k_grid_vmax<3><<<groups, kThreads, 0, st>>>(grid, active, totals, out);
  else
    k_grid_vmax<2><<<groups, kThreads, 0, st>>>(grid, active, totals, out);
}

template <int D>
__global__ __launch_bounds__(kThreads) void k_grid_gather(const float4* __restrict__ grid,
                                                         const int* __restrict__ active,
                                                         int64_t count, NodeWindow w,
                                                         int* __restrict__ coords,
                                                         float* __restrict__ v,
                                                         float* __restrict__ m) {
  constexpr int NPB = Geo<D>::kNodesPerBlock;
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < count;
       i += (int64_t)gridDim.x * kThreads) {
    const int bid = active[i / NPB], l = (int)(i % NPB);
    const float4 g = grid[(int64_t)bid * NPB + l];
    const int lb0 = bid % w.bn[0];
    const int lb1 = D == 3 ? (bid / w.bn[0]) % w.bn[1] : bid / w.bn[0] - w.zoff;
    coords[i * D + 0] = 4 * (w.blo[0] + lb0) + (l & 3);
    coords[i * D + 1] = 4 * (w.blo[1] + lb1) + ((l >> 2) & 3);
    v[i * D + 0] = g.x;
    v[i * D + 1] = g.y;
    if (D == 3) {
      const int lb2 = bid / (w.bn[0] * w.bn[1]) - w.zoff;
      coords[i * D + 2] = 4 * (w.blo[2] + lb2) + (l >> 4);
      v[i * D + 2] = g.z;
    }
    m[i] = g.w;
  }
}

template <int D>
__global__ __launch_bounds__(kThreads) void k_grid_scatter(float4* __restrict__ grid,
                                                          const int* __restrict__ active,
                                                          int64_t count,
                                                          const float* __restrict__ v) {
  constexpr int NPB = Geo<D>::kNodesPerBlock;
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < count;
       i += (int64_t)gridDim.x * kThreads) {
    float4* g = &grid[(int64_t)active[i / NPB] * NPB + i % NPB];
    g->x = v[i * D + 0];
    g->y = v[i * D + 1];
    if (D == 3) g->z = v[i * D + 2];
  }
}

void launch_grid_gather(int D, const float4* grid, const int* active, int64_t count,
                        const NodeWindow& w, int* coords, float* v, float* m, hipStream_t st) {
  if (count <= 0) return;
  const int groups = clamp_groups(div_up(count, kThreads), 4096);
  if (D == 3)
    k_grid_gather<3><<<groups, kThreads, 0, st>>>(grid, active, count, w, coords, v, m);
  else
    k_grid_gather<2><<<groups, kThreads, 0, st>>>(grid, active, count, w, coords, v, m);
}

void launch_grid_scatter(int D, float4* grid, const int* active, int64_t count, const float* v,
                         hipStream_t st) {
  if (count <= 0) return;
  const int groups = clamp_groups(div_up(count, kThreads), 4096);
  if (D == 3)
    k_grid_scatter<3><<<groups, kThreads, 0, st>>>(grid, active, count, v);
  else
    k_grid_scatter<2><<<groups, kThreads, 0, st>>>(grid, active, count, v);
}

template void launch_transfer<2>(const Params*, const int*, SubstepBuffers&, int, hipStream_t,
                                 Timer*);
template void launch_transfer<3>(const Params*, const int*, SubstepBuffers&, int, hipStream_t,
                                 Timer*);
template void launch_grid_op<2>(const Params*, const int*, const SubstepBuffers&, int, hipStream_t,
                                Timer*);
template void launch_grid_op<3>(const Params*, const int*, const SubstepBuffers&, int, hipStream_t,
                                Timer*);
template void launch_front<2>(const Params*, const int*, SubstepBuffers&, int, hipStream_t,
                              Timer*);
template void launch_front<3>(const Params*, const int*, SubstepBuffers&, int, hipStream_t,
                              Timer*);
template void launch_adjoint<2>(const Params*, const int*, SubstepBuffers&, const float*,
                                const float*, float*, float*, float4*, float*, float*, hipStream_t,
                                Timer*);
template void launch_adjoint<3>(const Params*, const int*, SubstepBuffers&, const float*,
                                const float*, float*, float*, float4*, float*, float*, hipStream_t,
                                Timer*);
template void launch_substep<2>(const Params*, const int*, SubstepBuffers&, int, int, hipStream_t,
                                Timer*);
template void launch_substep<3>(const Params*, const int*, SubstepBuffers&, int, int, hipStream_t,
                                Timer*);
template void launch_substep_half<2>(const Params*, const int*, SubstepBuffers&, int, int,
                                     hipStream_t, Timer*);
template void launch_substep_half<3>(const Params*, const int*, SubstepBuffers&, int, int,
                                     hipStream_t, Timer*);
template void launch_append<2>(SubstepBuffers&, const float*, const float*, const int*, int, int,
                               int, int, hipStream_t);
template void launch_append<3>(SubstepBuffers&, const float*, const float*, const int*, int, int,
                               int, int, hipStream_t);
template void launch_unpack<2>(const float*, float*, int, int64_t, bool, bool, hipStream_t);
template void launch_unpack<3>(const float*, float*, int, int64_t, bool, bool, hipStream_t);
template void launch_pack<2>(const float*, float*, int, int64_t, bool, bool, hipStream_t);
template void launch_pack<3>(const float*, float*, int, int64_t, bool, bool, hipStream_t);

}  // namespace mpm
