// Steady-state binning: the particles of a chunk found from the previous
// substep's direction lists (device code shared by k_p2g and k_g2p2g).
//
// The order of a substep is the previous order stably sorted by the new
// block key.  Particles move less than one block per substep, so the members
// of new block b come from its 3^d old neighbours b - dir; in the previous
// order they are grouped by old block (ascending key), then by old chunk,
// then by position.  g2p leaves each old chunk's particles grouped by
// direction (members, at the chunk's own range) with the count and start of
// each group (dseg).  The next substep walks, for each new chunk, the groups
// that point at its block in that order and takes its share of them
// (wave_members): either the transfer that opens the substep does so itself,
// or k_members does it for all chunks first.
//
// Which of the two: the walk is three dependent round trips to memory, ~2 us
// a chunk.  Inside p2g (four waves per SIMD, every workgroup waiting for its
// own list) they add up over the chunks a workgroup takes one after the
// other: 76 -> 89 us at 4567 chunks (3D, 1M particles), 21.6 -> 33 us at
// 4601 chunks (2D).  With about one chunk per workgroup they cost less than
// a kernel: 5.7 -> 8.6 us at 143 chunks (2D, 20k particles) and 19.6 -> 22.4
// us at 632 (3D, 100k).  A kernel of its own hides them behind eight waves
// per SIMD: 8.9 us at 4567 chunks, 6.3 us at 4601 (2D), 95 us at 86.8k (16M
// particles).  It takes the place of an offsets kernel over the blocks and a
// scatter over the particles (6.4 + 6.5, 4.9 + 5.3 and 65 + 125 us), with the
// key and code arrays between them; a workgroup per chunk instead of a wave
// took 13.2, 10.6 and 151 us.  The line lies at kListsInTransfer particles
// (kOneRound for the fused transfer) in kFewChunks chunks, as far as the
// number is known: substeps with the lists walked by k_members and inside p2g
// take 56.2 and 54.6 us at 200k particles in 1117 chunks (3D), 63.9 and 62.3 at
// 250k in 1390, 84.3 and 84.9 at 500k in 2686; 38.1 and 37.0 at 250k in 2116
// (2D), 51.7 and 55.1 at 400k in 4225; spread thinly 59.6 and 60.5 at 50k in
// 2975 chunks, 129 and 138 at 100k in 8687, in 2D 38.0 and 42.2 at 60k in 3385,
// 285 and 354 at 100k in 45096.
#pragma once

#include "mpm_device.h"

namespace mpm {

// The previous substep's chunks, per-block chunk ranges and direction lists.
// members == nullptr: the order comes from a full sort (perm).
struct PrevBinning {
  const int* pchunk_begin;
  const int* pchunk_cnt;
  const int4* chunks;
  const int* dseg;     // [chunk][27]: count | start << 16
  const int* members;  // particle slots, each old chunk's range grouped by direction
};

__device__ __forceinline__ int wave_scan_inclusive(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(v, off);
    if (lane >= off) v += y;
  }
  return v;
}

// id[k] = slot of the particle at position r0 + k * stride of block lb, for
// positions below r1; -1 beyond, and for a position no group covers (the
// counts and the lists disagree: cannot happen).  A whole wave calls it, each
// lane with its own r0.  The wave holds 64 groups at a time, one per lane
// (27 or 9 neighbours with usually one to three chunks each: one or two
// rounds, but as many as there are groups), and a lane finds its position's
// group by a binary search through shuffles: no LDS, no barrier.
template <int D, int K>
__device__ __forceinline__ void wave_members(const int lb[3], int r0, int stride, int r1,
                                             const Params& W, const PrevBinning& prev,
                                             int id[K]) {
  constexpr int NB = D == 3 ? 27 : 9;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < K; k++) id[k] = -1;
  int c0 = 0, cn = 0;
  if (lane < NB) {
    // ascending old key <=> descending offset (dz, dy, dx) in lexicographic order
    const int q[3] = {lb[0] - 1 + lane % 3, lb[1] - 1 + (lane / 3) % 3,
                      D == 3 ? lb[2] - 1 + lane / 9 : 0};
    if (q[0] >= 0 && q[0] < W.bn[0] && q[1] >= 0 && q[1] < W.bn[1] &&
        (D == 2 || (q[2] >= 0 && q[2] < W.bn[2]))) {
      const int ob = encode_local<D>(q, W);
      c0 = prev.pchunk_begin[ob];
      cn = prev.pchunk_cnt[ob];
    }
  }
  const int cinc = wave_scan_inclusive(cn);
  const int total = __shfl(cinc, 63);
  for (int s0 = 0, base = 0; s0 < total && base < r1; s0 += 64) {
    const int s = s0 + lane;
    // neighbour of group s: the first whose inclusive chunk count exceeds s
    int t = 0;
#pragma unroll
    for (int step = 32; step > 0; step >>= 1) {
      const int y = __shfl(cinc, min(t + step - 1, 63));
      if (t + step <= 63 && y <= s) t += step;
    }
    const int oc = __shfl(c0 + cn - cinc, t) + s;
    int cnt = 0, src = 0;
    if (s < total) {
      const int dx = 1 - t % 3, dy = 1 - (t / 3) % 3, dz = D == 3 ? 1 - t / 9 : 0;
      const int w = prev.dseg[(int64_t)oc * 27 + (dz + 1) * 9 + (dy + 1) * 3 + (dx + 1)];
      cnt = w & 0xffff;
      src = prev.chunks[oc].y + (w >> 16);
    }
    const int inc = wave_scan_inclusive(cnt);
    const int off = base + inc - cnt;
    const int end = base + __shfl(inc, 63);
    src -= off;
#pragma unroll
    for (int k = 0; k < K; k++) {
      const int r = r0 + k * stride;
      const bool in = r < r1 && r >= base && r < end;
      if (!__any(in)) continue;
      int g = 0;  // the last group that starts at or before r (empty ones share a start)
#pragma unroll
      for (int step = 32; step > 0; step >>= 1)
        if (__shfl(off, g + step) <= r) g += step;
      const int at = __shfl(src, g) + r;
      if (in) id[k] = prev.members[at];
    }
    base = end;
  }
}

// The particle order of a steady-state substep, one wave per chunk.
template <int D>
__global__ __launch_bounds__(kThreads) void k_members(const Params* __restrict__ scenes,
                                                      const int4* __restrict__ chunks,
                                                      const int* __restrict__ totals,
                                                      const int* __restrict__ pstart,
                                                      PrevBinning prev, int* __restrict__ perm,
                                                      int* __restrict__ err) {
  constexpr int K = 4;
  const Params& W = scenes[0];  // the combined window extents
  const int nchunks = totals[kTotChunks], lane = threadIdx.x & 63;
  for (int c = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6); c < nchunks;
       c += gridDim.x * (kThreads / 64)) {
    const int4 ck = chunks[c];
    int lb[3], id[K];
    decode_local<D>(ck.x, W, lb);
    const int first = pstart[ck.x];
    for (int b0 = ck.y; b0 < ck.z; b0 += 64 * K) {
      wave_members<D, K>(lb, b0 - first + lane, 64, ck.z - first, W, prev, id);
#pragma unroll
      for (int k = 0; k < K; k++) {
        const int j = b0 + lane + 64 * k;
        if (j >= ck.z) continue;
        if (id[k] < 0) atomicOr(err, 16);  // counts and lists disagree (cannot happen)
        perm[j] = max(id[k], 0);
      }
    }
  }
}

// The direction groups of a chunk, by its first wave: lane d < 27 gives the
// chunk's particles of direction d (0 from the others); their counts and
// starts go to dseg and dstart and are added to the block counts of the next
// substep.
template <int D>
__device__ __forceinline__ void write_groups(int c, const int lb[3], const Params& W, int cnt,
                                             int* dstart, int* dseg, int* count_next) {
  const int d = threadIdx.x & 63;
  const int start = wave_scan_inclusive(cnt) - cnt;
  if (d < 27) {
    dstart[d] = start;
    dseg[(int64_t)c * 27 + d] = cnt | (start << 16);
    if (cnt > 0) {
      const int q[3] = {lb[0] + d % 3 - 1, lb[1] + (d / 3) % 3 - 1, lb[2] + d / 9 - 1};
      atomicAdd(&count_next[encode_local<D>(q, W)], cnt);
    }
  }
}

}  // namespace mpm
