// Tile machinery shared by the pair loops (tsph_pairs.hip, tsph_ale.hip):
// one wavefront per run of `rows` cells of a grid column, persistent waves that
// walk XCD-banded slices of the list of non-empty tiles, the cell-offset table
// of the three neighbour slices in LDS, and the lane-private neighbour lists.
#pragma once

#include <algorithm>
#include <climits>

#include "tsph_internal.h"
#include "tsph_physics.h"

namespace tsph {
namespace tiles {

constexpr int kWave = 64;          // one wavefront per tile
constexpr int kCellCap = 11;       // LDS records budgeted per cell of the slices
constexpr int kLdsGranule = 1280;  // LDS bytes are allocated in units of
constexpr int kList = 32;          // per-lane neighbour list entries in LDS
constexpr int kGroup = 8;          // candidates tested together in the mixed pair loop
constexpr int kStageU = 4;         // staged slots per lane whose loads are in flight together
constexpr float kFar32 = 1e30f;    // coordinate of the mixed loop's sentinel slots

// adds the wavefront's counts to its own slots (kWaveCtr0 + 4 w, w: the
// wavefront's index in the launch); no two wavefronts of a launch share a slot
__device__ __forceinline__ void wave_count(unsigned pairs, unsigned cand, unsigned act,
                                           unsigned long long *counters) {
  unsigned long long a = pairs, b = cand, c = act;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b += __shfl_xor(b, o, 64);
    c += __shfl_xor(c, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    const int w = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    unsigned long long *p = counters + kWaveCtr0 + 4 * w;
    p[0] += a;
    p[1] += b;
    p[2] += c;
  }
}

// --------------------------------------------------------------------------
// tiles: one workgroup = one wavefront = one run of `rows` cells of a column
// --------------------------------------------------------------------------
// Dynamic LDS layout: int tab[3 * (kMaxTileRows + 3)] (cell_start of the rows
// of the three neighbour slices), the staged neighbour records, the lane lists.
constexpr int kTabInts = 3 * (kMaxTileRows + 3);
constexpr int kTabBytes = ((kTabInts * 4 + 15) / 16) * 16;

struct Tile {
  int cx, cy0, cy1, row_lo, nrows, w;
  int own0, own1;   // particle range of the tile
  int lq[4];        // LDS start of slice q (lq[3] = records staged)
  int base[3];      // LDS index - global index, per slice
};

// element q of a 3-array held in registers, without dynamic indexing (which
// would place the array in scratch memory)
__device__ __forceinline__ int sel3(const int (&a)[3], int q) {
  return q == 0 ? a[0] : (q == 1 ? a[1] : a[2]);
}

// Each wavefront of a tile kernel works on its own tile with its own LDS area;
// a workgroup holds one wavefront (static walk) or up to kPoolWaves of them
// (pooled walk), which share nothing but the pool's counter and tile order.
// LDS layout: pool_hdr(DYN) bytes (the pooled walk's counter, then kPoolSort
// tile positions), then one area of lds_wave bytes per wavefront.
constexpr int kPoolWaves = 4;
constexpr int kPoolSort = 64;  // chunks of at most this many tiles go in decreasing cost
constexpr int kPoolHdr = 16 + 4 * kPoolSort;
constexpr int kStaticHdr = 16;
constexpr int pool_hdr(bool pooled) { return pooled ? kPoolHdr : kStaticHdr; }

__device__ __forceinline__ int tile_lane() { return threadIdx.x & (kWave - 1); }

template <bool DYN>
__device__ __forceinline__ unsigned char *wave_lds(unsigned char *smem, int lds_wave) {
  return smem + pool_hdr(DYN) + (threadIdx.x >> 6) * lds_wave;
}

// Hand-over between the lanes of one wavefront through LDS (staged records,
// lists): a wavefront's LDS instructions execute in issue order, so only the
// compiler has to be kept from moving accesses across this point.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Persistent waves over the list of non-empty tiles (tile order).  Workgroup
// b runs on XCD b % 8.  Two walks:
//   * static (DYN = false, one wavefront per workgroup): the list is cut into
//     8 contiguous bands and the waves of XCD x stride through band x, so
//     tiles that are neighbours in the list, which share slices, are staged
//     from the same L2;
//   * pooled (DYN = true): the list is cut into one chunk per workgroup of
//     about equal cost, by the times the tiles took in the previous pass
//     (chunk bounds written by k_cut_chunks), the chunks of XCD x again
//     contiguous; the workgroup's wavefronts take the tiles of their chunk
//     from a counter in LDS, the costliest first (a chunk of up to kPoolSort
//     tiles is sorted by recorded cost when the workgroup starts), so that
//     the tiles left for the end are the cheap ones.  Waves of one compute
//     unit thereby balance each other, and the compute units each other
//     through the costs, without any device-wide atomic (those serialise
//     across the XCDs).
// The pooled walk records each tile's time (tq_mark) for the next cut.
struct TileQueue {
  int ntl;   // static: tiles in the list
  int band;  // static: band of the wave
  int nwb;   // static: waves per band
  int wb;    // static: this wave's rank in its band
  int j;     // static: round of the current tile
  int lo, hi;   // pooled: the chunk
  int *ctr;     // pooled: the chunk's next tile (LDS)
  int *order;   // pooled, sorted chunk: list positions in decreasing cost (LDS)
  bool sorted;  // pooled: the chunk is taken in the order of `order`
  int *cost; // per-tile costs of the wave's table (tile t at cost[kCostTables t])
  int cur;   // global tile being timed (-1: none)
  int old;   // its recorded cost (lane 0)
  unsigned long long t0;  // its start
};

__device__ __forceinline__ int band_lo(int ntl, int b) { return (int)(((long long)ntl * b) >> 3); }

template <bool DYN>
__device__ __forceinline__ TileQueue tq_begin(int *__restrict__ scal, const int *__restrict__ bound,
                                              const int *__restrict__ tile_list,
                                              unsigned char *smem, int table = 0,
                                              int groups = 0) {  // 0: the whole launch
  TileQueue tq;
  tq.ntl = 0;
  tq.band = blockIdx.x & 7;
  tq.nwb = (groups ? groups : (int)gridDim.x) >> 3;
  tq.wb = blockIdx.x >> 3;
  tq.j = -1;
  tq.lo = tq.hi = 0;
  tq.ctr = reinterpret_cast<int *>(smem);
  tq.order = reinterpret_cast<int *>(smem + 16);
  tq.sorted = false;
  tq.cost = scal + S_NSCAL + table;
  tq.cur = -1;
  tq.old = 0;
  tq.t0 = 0;
  if (!DYN) {
    tq.ntl = scal[S_NTILES];
  } else {
    const int chunk = tq.band * tq.nwb + tq.wb;
    tq.lo = bound[chunk];
    tq.hi = bound[chunk + 1];
    tq.sorted = tq.hi - tq.lo <= kPoolSort;
    if (threadIdx.x == 0) *tq.ctr = tq.lo;
    if (tq.sorted && threadIdx.x < kWave) {
      // bitonic sort of (cost, position) over the first wavefront's lanes,
      // decreasing cost, ties in list order; unused lanes sort last
      const int l = threadIdx.x;
      int key = -1, idx = l;
      if (tq.lo + l < tq.hi) key = tq.cost[kCostTables * tile_list[tq.lo + l]];
      for (int k = 2; k <= kWave; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
          const int ok = __shfl_xor(key, j, kWave), oi = __shfl_xor(idx, j, kWave);
          const bool first = ok > key || (ok == key && oi < idx);  // the other ranks first
          const bool keep_first = ((l & k) == 0) == ((l & j) == 0);
          if (keep_first == first) {
            key = ok;
            idx = oi;
          }
        }
      tq.order[l] = tq.lo + idx;
    }
    __syncthreads();
  }
  return tq;
}

// Records the wave's current tile's cost (the time since it began, in 10 ns
// ticks of the device's constant clock, averaged with the tile's recorded
// cost if it has one) and begins global tile `tile` (-1: none, after the
// last tile).
__device__ __forceinline__ void tq_mark(TileQueue &tq, int tile) {
  const unsigned long long now = wall_clock64();
  if (tile_lane() == 0) {
    if (tq.cur >= 0) {
      const unsigned long long u = now - tq.t0;
      int w = u < 1 ? 1 : (u > (1u << 24) ? (1 << 24) : (int)u);
      if (tq.old > 0) w = (tq.old + w + 1) >> 1;
      tq.cost[kCostTables * tq.cur] = w;
    }
    // the new tile's record, read now and used when it ends
    tq.old = tile >= 0 ? tq.cost[kCostTables * tile] : 0;
  }
  tq.cur = tile;
  tq.t0 = now;
}

// pooled walk: lane 0 takes the next tile of the chunk (read with tq_take)
template <bool DYN>
__device__ __forceinline__ int tq_ticket(const TileQueue &tq) {
  int t = 0;
  if (DYN && tile_lane() == 0) t = atomicAdd(tq.ctr, 1);
  return t;
}

// list index of the wave's next tile (raw: the value from tq_ticket), or -1
template <bool DYN>
__device__ __forceinline__ int tq_take(TileQueue &tq, int raw) {
  if (!DYN) {
    const int idx = band_lo(tq.ntl, tq.band) + tq.wb + (++tq.j) * tq.nwb;
    return idx < band_lo(tq.ntl, tq.band + 1) ? idx : -1;
  }
  const int v = __builtin_amdgcn_readfirstlane(raw);
  if (v >= tq.hi) return -1;
  return tq.sorted ? tq.order[v - tq.lo] : v;
}

// Loads the cell offsets of the three slices (one global load per lane, all in
// flight together) and derives the tile ranges.  False for an empty tile.
__device__ __forceinline__ bool tile_begin(const Consts &k, const int *__restrict__ cell_start,
                                           int cx, int cy0, int cy1, int *tab, Tile &t) {
  t.cx = cx;
  t.cy0 = cy0;
  t.cy1 = cy1;
  t.row_lo = max(t.cy0 - 1, 0);
  t.nrows = min(t.cy1 + 1, k.ncy) - t.row_lo;
  t.w = t.nrows + 1;
  for (int e = tile_lane(); e < 3 * t.w; e += kWave) {
    const int q = e / t.w, r = e - q * t.w;
    const int col = t.cx + q - 1;
    tab[e] = (col >= 0 && col < k.ncx) ? cell_start[col * k.ncy + t.row_lo + r] : 0;
  }
  wave_sync();
  t.own0 = tab[t.w + (t.cy0 - t.row_lo)];
  t.own1 = tab[t.w + (t.cy1 - t.row_lo)];
  int l = 0;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const int g0 = tab[q * t.w], g1 = tab[q * t.w + t.nrows];
    t.lq[q] = l;
    t.base[q] = l - g0;
    l += g1 - g0;
  }
  t.lq[3] = l;
  return t.own1 > t.own0;
}
__device__ __forceinline__ bool tile_begin(const Consts &k, const int *__restrict__ cell_start,
                                           int tile, int rows, int *tab, Tile &t) {
  const int nty = (k.ncy + rows - 1) / rows;
  const int cx = tile / nty, cy0 = (tile - cx * nty) * rows;
  return tile_begin(k, cell_start, cx, cy0, min(cy0 + rows, k.ncy), tab, t);
}

// Entries of a tile list.  The list of a static walk gives a tile of more than
// kWave particles two entries, one for the first kWave and one for the rest,
// so that another wavefront takes the second round: with about a tile per
// resident wavefront the tiles of two rounds set the pass's time (they are
// few on the lattice a run starts from, and up to a third later on).  The
// tile's frame and each particle's sums are the same either way.
constexpr int kTileFirst = 1 << 30, kTileRest = (int)(1u << 31), kTileMask = kTileFirst - 1;
__device__ __forceinline__ int entry_tile(int e) { return e & kTileMask; }
// the tile's own particles that entry e stands for
__device__ __forceinline__ void entry_part(int e, Tile &t) {
  if (e & kTileFirst) t.own1 = min(t.own1, t.own0 + kWave);
  if (e & kTileRest) t.own0 = min(t.own1, t.own0 + kWave);
}

// case of global tile t in a batched ensemble (tile_base: ncases+1 bounds)
__device__ __forceinline__ int case_of_tile(const int *__restrict__ tile_base, int ncases, int t) {
  int lo = 0, hi = ncases;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (tile_base[mid] <= t) lo = mid;
    else hi = mid;
  }
  return lo;
}

// own particles of global tile t (its `rows` cells of one column)
__device__ __forceinline__ int tile_own(const int *__restrict__ cell_start, const Consts &k0,
                                        const Consts *__restrict__ cases,
                                        const int *__restrict__ tile_base, int ncases, int rows,
                                        int t) {
  int lt = t, cell_base = k0.cell_base, ncy = k0.ncy;
  if (cases) {
    const int cse = case_of_tile(tile_base, ncases, t);
    lt = t - tile_base[cse];
    cell_base = cases[cse].cell_base;
    ncy = cases[cse].ncy;
  }
  const int *cs = cell_start + cell_base;
  const int nty = (ncy + rows - 1) / rows;
  const int cx = lt / nty, cy0 = (lt - cx * nty) * rows, cy1 = min(cy0 + rows, ncy);
  return cs[cx * ncy + cy1] - cs[cx * ncy + cy0];
}

// exclusive scan of a over the block (blockDim.x threads, a multiple of 64);
// total: the block's sum.  lds: one slot per wavefront.
template <typename T>
__device__ __forceinline__ T block_exscan(T a, T &total, T *lds) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  T x = a;
  for (int o = 1; o < 64; o <<= 1) {
    const T y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  __syncthreads();
  if (lane == 63) lds[wid] = x;
  __syncthreads();
  T before = 0;
  total = 0;
  for (int w = 0; w < nw; ++w) {
    const T v = lds[w];
    if (w < wid) before += v;
    total += v;
  }
  return before + x - a;
}

// Chunk starts of a pooled walk of `groups` workgroups over the listed tiles,
// cut by cost: listed tile t has the cost interval [W0, W0 + w) (W0: the costs
// of the tiles before it), and chunk g starts at the tile whose interval holds
// g W / groups (W: the total), so that every chunk holds about W / groups.
// The costs come by list position (list_cost, written with the list).  The
// list is cut in segments of kCutSeg entries, one workgroup of kCutBlock
// threads each (cut_segments: workgroups beyond the list exit at once), which
// share nothing: each reads the whole cost list, consecutive threads on
// consecutive entries and kCutBatch loads of each thread in flight together,
// to form the total and the costs of the segments before its own, and keeps
// its own segment in LDS; each thread then scans a contiguous run of it and
// finds the chunk starts there by comparing products (g W against (W0 + w)
// groups) rather than by divisions.
constexpr int kCutBlock = 1024, kCutBatch = 16, kCutSeg = kCutBlock * kCutBatch;

// workgroups that cut a list of at most `tiles` entries
inline int cut_segments(int tiles) { return tiles / kCutSeg + 1; }

// the cut of segment `seg` by one workgroup of kCutBlock threads; wl: kCutSeg
// ints, red: kCutBlock / 64 long longs of LDS
__device__ __forceinline__ void cut_chunks_block(const int *__restrict__ scal,
                                                 const int *__restrict__ list_cost, int groups,
                                                 int *__restrict__ bound, int seg, int *wl,
                                                 long long *red) {
  const int n = scal[S_NTILES];
  const int s0 = seg * kCutSeg;
  if (seg == 0) {
    if (threadIdx.x == 0) bound[groups] = n;
    if (n == 0)
      for (int g = threadIdx.x; g < groups; g += kCutBlock) bound[g] = 0;
  }
  if (s0 >= n) return;
  // the total and the costs before this segment; this segment's costs to LDS
  long long all = 0, before = 0;
  for (int b0 = 0; b0 < n; b0 += kCutSeg) {
    int w[kCutBatch];
#pragma unroll
    for (int u = 0; u < kCutBatch; ++u) {
      const int e = b0 + u * kCutBlock + (int)threadIdx.x;
      w[u] = e < n ? list_cost[e] : 0;
    }
    long long part = 0;
#pragma unroll
    for (int u = 0; u < kCutBatch; ++u) part += w[u];
    all += part;
    if (b0 < s0) before += part;
    if (b0 == s0) {
#pragma unroll
      for (int u = 0; u < kCutBatch; ++u) wl[u * kCutBlock + threadIdx.x] = w[u];
    }
  }
  long long total = 0, carry = 0;
  block_exscan(all, total, red);
  block_exscan(before, carry, red);
  const int m = min(kCutSeg, n - s0);
  const int per = (m + kCutBlock - 1) / kCutBlock;
  const int lo = min((int)threadIdx.x * per, m), hi = min(lo + per, m);
  long long r = 0;
  for (int e = lo; e < hi; ++e) r += wl[e];
  long long segsum = 0;
  long long p = carry + block_exscan(r, segsum, red);
  // first chunk whose start g W / groups >= p
  long long g = (p * groups + total - 1) / total;
  for (int e = lo; e < hi; ++e) {
    p += wl[e];
    const long long end = p * groups;  // chunk g starts in this tile while g W < end
    for (; g < groups && g * total < end; ++g) bound[g] = s0 + e;
  }
}

// The same cut right after the cell-list scan that listed the tiles, from its
// per-block sums: the listed tiles of scan block b sit at list positions
// [tile0[b], tile0[b + 1]) (the last block's end: the list length) and cost
// bsum[b] together.  Workgroup wg (blockDim.x threads, one wavefront per scan
// block, nb blocks) forms the costs before its blocks and the total from the
// nb block sums; each wavefront then reads its block's tile costs 64 at a
// time, scans them across the lanes, and writes the starts of the chunks that
// begin at its tiles.  red, pfx: blockDim.x / 64 long longs of LDS each.
__device__ __forceinline__ void cut_chunks_scan(const int *__restrict__ scal,
                                                const int *__restrict__ list_cost,
                                                const int *__restrict__ bsum,
                                                const int *__restrict__ tile0, int nb, int groups,
                                                int *__restrict__ bound, int wg, long long *red,
                                                long long *pfx) {
  const int n = scal[S_NTILES];
  const int nw = blockDim.x >> 6, wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (wg == 0) {
    if (threadIdx.x == 0) bound[groups] = n;
    if (n == 0)
      for (int g = threadIdx.x; g < groups; g += blockDim.x) bound[g] = 0;
  }
  if (n == 0 || wg * nw >= nb) return;
  long long carry = 0;
  for (int r0 = 0; r0 < nb; r0 += blockDim.x) {
    const int q = r0 + threadIdx.x;
    long long sum = 0;
    const long long ex = block_exscan<long long>(q < nb ? bsum[q] : 0, sum, red) + carry;
    const int qw = q - wg * nw;
    if (qw >= 0 && qw < nw) pfx[qw] = ex;
    carry += sum;
  }
  __syncthreads();
  const long long total = carry;
  const int b = wg * nw + wid;
  if (b >= nb || total <= 0) return;
  long long p = pfx[wid];
  const int t1 = b + 1 < nb ? tile0[b + 1] : n;
  for (int e0 = tile0[b]; e0 < t1; e0 += 64) {
    const int e = e0 + lane;
    const long long w = e < t1 ? list_cost[e] : 0;
    long long x = w;
    for (int o = 1; o < 64; o <<= 1) {
      const long long y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (e < t1) {
      const long long w0 = p + x - w;  // the costs before tile e
      long long g = (w0 * groups + total - 1) / total;
      const long long end = (w0 + w) * groups;
      for (; g < groups && g * total < end; ++g) bound[g] = e;
    }
    p += __shfl(x, 63, 64);
  }
}

__device__ __forceinline__ int slice_of(const Tile &t, int l) {
  return l >= t.lq[2] ? 2 : (l >= t.lq[1] ? 1 : 0);
}

// --------------------------------------------------------------------------
// Generic tile walk of the mixed passes (walk32).  A pass supplies a policy P:
//   P::Lds            pointers into the staged-slot area of LDS
//   P::lds(base, cap) carves that area (float2 arrays first)
//   P::kSlotBytes     bytes per staged slot
//   stage(L, l, j, ox, oy)  slot l <- particle j (tile-frame origin)
//   active(i)         whether particle i is active in the pass
//   Own own(i, ox, oy); Acc{} accumulators
//   pair_lds(acc, own, L, l, drx, dry, r2) / pair_glob(acc, own, j, ...)
//   finish(acc, own, i)
// It visits the three column slices in memory order with an FP32 test.
// --------------------------------------------------------------------------

// --------------------------------------------------------------------------
// Cell walk (FP64): one wavefront per cell, its pairs spread over all lanes
// --------------------------------------------------------------------------
// The tile walks give each lane a particle and its ~20 pairs one after the
// other, so a pass lasts at least that chain however few tiles there are, and
// its lanes wait for the longest list.  Here a wavefront takes one cell
// (about nine particles):
//   1. the particles of the 9 stencil cells are staged in LDS in the reference
//      order (cell order, ascending index), so slot order is candidate order
//      and the cell's own particles are the first slots;
//   2. for each own particle the lanes test all candidate slots at once (two
//      per lane, four in the wide form) and append the pairs, in order, to one
//      flat list (ballots and prefix counts; the bookkeeping is scalar);
//   3. the lanes evaluate 64 pairs of that list at a time, whichever particles
//      they belong to, and leave each pair's kSums terms in LDS;
//   4. lane (particle, term) adds its particle's terms in list order.
// Every sum is formed in the reference order from the same terms (a term
// leaves the pair function as 0 + x or 0 - x, exactly x or -x), so the results
// are the tile walks', bit for bit.
//
// A policy P supplies kSums, kSlotBytes, Lds and lds(base, cap), and
//   set(k)                        constants of the case (batched grids)
//   Rec load(j), store(L, l, rec) slot l <- particle j, in two halves
//   act_lds(L, l)                 slot l is active
//   kSkip, skip_lds(L, l)         pairs of two slots with skip_lds are no
//                                 candidates (DBC walls)
//   kWaves                        wavefronts of a workgroup
//   kSlots                        staged slots: cell_slots_of<H>(), H slots per
//                                 lane (2, or 4: the wide form)
//   kFlag                         sums() wants to know whether any of the
//                                 particle's pairs has bit 1 set (below)
//   terms(L, p, l, double (&t)[kSums])  the terms of pair (p, l), which is
//                                 inside the support (Consts::r2max); bit 0 of the
//                                 result: it counts as a pair interaction, bit 1: a flag
//   sums(L, p, i, const double (&s)[kSums], flag)  writes particle i, slot p
//   far(i, cs, g, c, counts...)   particle i of cell c from global memory
// staged slots of a cell's neighbourhood, and flat list entries (own particles
// listed together x candidates), for H slots per lane
template <int H>
constexpr int cell_slots_of() { return H == 2 ? 104 : 232; }
template <class P>
constexpr int cell_halves() { return (P::kSlots + kWave - 1) / kWave; }
template <class P>
constexpr int cell_flat() { return cell_halves<P>() == 2 ? 640 : 2048; }
constexpr double kFar64 = 1e150;  // coordinate of slots past the last (its square is finite)
constexpr int kCellBlock = 4 * kWave;  // most threads of a workgroup
constexpr int kCellRun = 6;      // log2 of the most consecutive listed cells of one XCD
template <class P>
constexpr int cell_terms() { return P::kSums <= 4 ? 184 : 128; }  // pairs whose terms are in LDS together
// a workgroup's non-empty cells (and their cases), and the next to take
struct CellQueue {
  int count, next, pad[2];
  int cell[kCellBlock];
  uint8_t cse[kCellBlock];
};
// LDS bytes of a wavefront of a cell walk
template <class P>
constexpr int cell_wave_bytes() {
  return (cell_terms<P>() * P::kSums * 8 + cell_flat<P>() * 2 + P::kSlots * P::kSlotBytes + 15) / 16 * 16;
}
template <class P>
constexpr int cell_lds_bytes() {
  return (int)sizeof(CellQueue) + P::kWaves * cell_wave_bytes<P>();
}

// what a cell walk knows of a case's grid
struct CellGrid {
  int ncx, ncy, cell_base;
  double c2;  // Consts::r2max
};
__host__ __device__ __forceinline__ CellGrid cell_grid(const Consts &k) {
  return {k.ncx, k.ncy, k.cell_base, k.r2max};
}

// case whose cell range holds global cell c
__device__ __forceinline__ int case_of_cell(const Consts *__restrict__ cases, int ncases, int c) {
  int lo = 0, hi = ncases;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (cases[mid].cell_base <= c) lo = mid;
    else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ int cell_take(CellQueue &cq) {
  int at = 0;
  if (tile_lane() == 0) at = atomicAdd(&cq.next, 1);
  return __builtin_amdgcn_readfirstlane(at);
}

// the 9 stencil cells of global cell gc, one per lane: first particle and
// count (cells the reference reaches by wrapping into the neighbouring column
// are not visited)
__device__ __forceinline__ void cell_ranges(const CellGrid &g, const int *__restrict__ cell_start,
                                            int gc, int &lo, int &cnt) {
  const int *cs = cell_start + g.cell_base;
  const int c = gc - g.cell_base;
  const int cx = c / g.ncy, cy = c - cx * g.ncy;
  lo = cnt = 0;
  if (tile_lane() < 9) {
    int dx, dy;
    stencil_dxy(tile_lane(), dx, dy);
    if (cx + dx >= 0 && cx + dx < g.ncx && cy + dy >= 0 && cy + dy < g.ncy) {
      const int cl = c + dy + dx * g.ncy;
      lo = cs[cl];
      cnt = cs[cl + 1] - lo;
    }
  }
}

// the slots of those cells (lo, cnt: cell_ranges), and the loads of the
// lane's slots, in flight together
struct CellSlots {
  int own0, nown, tot;
};
template <class P, int H>
__device__ __forceinline__ CellSlots cell_slots(int lo, int cnt, typename P::Rec (&rec)[H],
                                                const P &pol) {
  const int lane = tile_lane();
  // slot l of cell q holds particle l + dj[q], for l in [pre[q], pre[q + 1])
  int pre[9], dj[9], tot = 0;
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    pre[q] = tot;
    dj[q] = __builtin_amdgcn_readlane(lo, q) - tot;
    tot += __builtin_amdgcn_readlane(cnt, q);
  }
  int j[H];
#pragma unroll
  for (int h = 0; h < H; ++h) {
    const int l = h * kWave + lane;
    j[h] = l + dj[0];
#pragma unroll
    for (int q = 1; q < 9; ++q) j[h] = l >= pre[q] ? l + dj[q] : j[h];
    if (l >= tot) j[h] = dj[0];
  }
#pragma unroll
  for (int h = 0; h < H; ++h) rec[h] = pol.load(j[h]);
  return {dj[0], __builtin_amdgcn_readlane(cnt, 0), tot};
}

// the list of non-empty cells (global ids, ascending) that a cell walk goes through
struct CellSource {
  const int *list, *count;
  int room;  // entries of the list's buffer
  int run;   // log2 of the consecutive entries of one XCD
};

template <class P>
__device__ __forceinline__ void cells64(P &pol, CellGrid g, const int *__restrict__ cell_start,
                                        const Consts *__restrict__ cases, int ncases,
                                        const CellSource src,
                                        unsigned long long *__restrict__ counters) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int NS = P::kSums;
  constexpr int NT = cell_terms<P>();
  constexpr int H = cell_halves<P>();
  static_assert(H <= 4 && P::kSlots < 256, "a list entry holds the slot in 8 bits");
  constexpr int kBlock = P::kWaves * kWave;
  constexpr int kOwn = NS < 4 ? 16 : 64 / NS;  // particles whose sums are formed together
  CellQueue &cq = *reinterpret_cast<CellQueue *>(smem);
  unsigned char *wl = smem + sizeof(CellQueue) + (threadIdx.x >> 6) * cell_wave_bytes<P>();
  double *terms = reinterpret_cast<double *>(wl);
  uint16_t *flat = reinterpret_cast<uint16_t *>(terms + NT * NS);
  const typename P::Lds L = P::lds(reinterpret_cast<unsigned char *>(flat + cell_flat<P>()), P::kSlots);
  const int lane = tile_lane();
  if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&counters[C_PASSES], 1ull);
  unsigned npair = 0, ncand = 0, nact = 0, scand = 0, snact = 0;
  // Runs of 2^run listed cells are dealt to the 8 XCDs in turn, so that a run's
  // cells share staged particles through one L2 while every XCD gets a share
  // of each part of the domain.  The workgroups of an XCD stride through its
  // cells, a cell per thread, and their wavefronts take them from a counter in
  // LDS.  (Dealt by grid cell, empty ones included, every third column's water
  // fell to the same XCD where 512 cells were about three columns, and to few of
  // its workgroups where their stride was: 61k and 52k particles of the dam break
  // 152 and 88 us per step, 99 and 86 now.)
  const int band = blockIdx.x & 7, nwb = gridDim.x >> 3, wb = blockIdx.x >> 3;
  const auto entry = [&](int j0) {  // list position of the thread's cell from j0 on
    const int u = j0 + (int)threadIdx.x * nwb;
    return (((u >> src.run) * 8 + band) << src.run) + (u & ((1 << src.run) - 1));
  };
  // A wavefront's first cell is the one at its own position, turned by two for
  // every second round of the workgroups over the XCD's 32 CUs: where a
  // workgroup has but one or two cells, those of a CU's workgroups would meet on
  // the same SIMDs (a pass of 9k particles 12.9 us not turned, 13.8 with all cells
  // taken from the counter, 11.4 now; of 7k 11.4, 12.7 and 10.1).
  const int first =
      __builtin_amdgcn_readfirstlane(((threadIdx.x >> 6) + (wb >> 5) * 2) & (P::kWaves - 1));
  int at = entry(wb);
  int next = at < src.room ? src.list[at] : 0;  // (beside the list's length)
  const int all = *src.count;
  const int mine = ((all + (8 << src.run) - 1) >> (3 + src.run)) << src.run;  // entries per XCD
  for (int j0 = wb; j0 < mine; j0 += nwb * kBlock) {
    if (j0 != wb) {
      at = entry(j0);
      next = at < all ? src.list[at] : 0;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      cq.count = 0;
      cq.next = P::kWaves;
    }
    __syncthreads();
    if (at < all) {
      const int q = atomicAdd(&cq.count, 1);
      cq.cell[q] = next;
      if (cases) cq.cse[q] = (uint8_t)case_of_cell(cases, ncases, next);
    }
    __syncthreads();
    const int todo = cq.count;
    for (int q = first; q < todo; q = cell_take(cq)) {
      const int c = __builtin_amdgcn_readfirstlane(cq.cell[q]);
      if (cases) {
        const Consts &k = cases[__builtin_amdgcn_readfirstlane((int)cq.cse[q])];
        g = cell_grid(k);
        pol.set(k);
      }
      int lo, cnt;
      cell_ranges(g, cell_start, c, lo, cnt);
      typename P::Rec rec[H];
      const CellSlots sl = cell_slots(lo, cnt, rec, pol);
      const int own0 = sl.own0, nown = sl.nown, tot = sl.tot;
      if (tot > P::kSlots || nown > kWave) {
        // neighbourhood beyond the LDS budget: gather from global memory
        for (int p = lane; p < nown; p += kWave)
          pol.far(own0 + p, cell_start + g.cell_base, g, c - g.cell_base, npair, ncand, nact);
        continue;
      }
      wave_sync();  // the previous cell's LDS is no longer read
#pragma unroll
      for (int h = 0; h < H; ++h)
        if (h * kWave + lane < tot) pol.store(L, h * kWave + lane, rec[h]);
      wave_sync();
      // candidate slots lane, 64 + lane ... in registers (slots past the last:
      // far away); the active own particles, and the slots that skip each
      // other, as bit masks
      double2 cp[H];
      unsigned long long skp[H];
      int skips_tot = 0;
#pragma unroll
      for (int h = 0; h < H; ++h) {
        const int l = h * kWave + lane;
        const bool real = l < tot;
        const double2 r = pol.pos_lds(L, real ? l : 0);
        cp[h] = real ? r : make_double2(kFar64, kFar64);
        skp[h] = P::kSkip ? __ballot(real && pol.skip_lds(L, real ? l : 0)) : 0ull;
        skips_tot += __popcll(skp[h]);
      }
      const unsigned long long act =
          __ballot(lane < nown && pol.act_lds(L, lane < nown ? lane : 0));
      snact += __popcll(act);
      scand += __popcll(act & ~skp[0]) * (tot - 1);
      if (P::kSkip) scand += __popcll(act & skp[0]) * (tot - skips_tot);
      if (!act) continue;
      const int most = min(kOwn, cell_flat<P>() / tot);  // own particles listed together
      for (int p0 = 0; p0 < nown; p0 += most) {
        const int np = min(most, nown - p0);
        int e = 0, st = 0;  // st: lane p's first list position (lane np: the list's length)
        double2 pr = pol.pos_lds(L, p0);
        for (int p = 0; p < np; ++p) {
          const int q = p0 + p;
          const double2 own = pr;
          pr = pol.pos_lds(L, q + 1);  // the next one's (slot q + 1 exists or is unused LDS)
          st = lane == p ? e : st;
          if (!((act >> q) & 1ull)) continue;
          const bool skips = P::kSkip && ((skp[0] >> q) & 1ull);
          unsigned long long m[H];
#pragma unroll
          for (int h = 0; h < H; ++h) {
            const double drx = own.x - cp[h].x, dry = own.y - cp[h].y;
            m[h] = __ballot(drx * drx + dry * dry <= g.c2);
            if (skips) m[h] &= ~skp[h];
          }
          m[0] &= ~(1ull << q);
#pragma unroll
          for (int h = 0; h < H; ++h) {
            if (__builtin_amdgcn_inverse_ballot_w64(m[h]))
              flat[__builtin_amdgcn_mbcnt_hi((unsigned)(m[h] >> 32),
                                             __builtin_amdgcn_mbcnt_lo((unsigned)m[h], e))] =
                  (uint16_t)(p << 8 | h << 6 | lane);
            e += __popcll(m[h]);
          }
        }
        st = lane == np ? e : st;
        wave_sync();
        // lane (particle pc, term tc) sums particle pc's list range
        const int pc = lane / NS, tc = lane - pc * NS;
        const int x0 = __shfl(st, pc, kWave), x1 = pc < np ? __shfl(st, min(pc + 1, 63), kWave) : 0;
        double acc = 0.;
        bool flag = false;
        for (int w0 = 0; w0 < e; w0 += NT) {
          const int we = min(NT, e - w0);
          for (int w = 0; w < we; w += kWave) {
            int got = 0;
            if (w + lane < we) {
              const unsigned en = flat[w0 + w + lane];
              double t[NS];
              got = pol.terms(L, p0 + (int)(en >> 8), (int)(en & 255u), t);
#pragma unroll
              for (int q = 0; q < NS; ++q) terms[q * NT + w + lane] = t[q];
            }
            npair += got & 1;
            if (P::kFlag) {
              // this window's part of the particle's list range
              const unsigned long long m = __ballot(got & 2);
              const int a = max(x0 - w0 - w, 0), b = min(x1 - w0 - w, kWave);
              if (a < b) flag |= (m >> a & (~0ull >> (kWave - (b - a)))) != 0;
            }
          }
          wave_sync();
          // eight terms at a time, their loads in flight together
          const double *tp = terms + tc * NT;
          const int hi = min(x1 - w0, NT);
          int x = max(x0 - w0, 0);
          for (; x + 8 <= hi; x += 8) {
            double v[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = tp[x + q];
#pragma unroll
            for (int q = 0; q < 8; ++q) acc += v[q];
          }
          // the rest with one more batch of loads (reads past the range stay
          // in the wavefront's LDS; +0 leaves a sum that starts at +0 unchanged)
          if (x < hi) {
            double v[7];
#pragma unroll
            for (int q = 0; q < 7; ++q) v[q] = tp[x + q];
#pragma unroll
            for (int q = 0; q < 7; ++q) acc += x + q < hi ? v[q] : 0.;
          }
          wave_sync();
        }
        // lane p takes its particle's sums and writes the particle
        terms[lane] = acc;
        const bool mine_flag = P::kFlag && __shfl((int)flag, min(lane * NS, 63), kWave);
        wave_sync();
        if (lane < np && pol.act_lds(L, p0 + lane)) {
          double sum[NS];
#pragma unroll
          for (int q = 0; q < NS; ++q) sum[q] = terms[lane * NS + q];
          pol.sums(L, p0 + lane, own0 + p0 + lane, sum, mine_flag);
        }
        wave_sync();
      }
    }
  }
  if (lane == 0) {
    ncand += scand;
    nact += snact;
  }
  wave_count(npair, ncand, nact, counters);
}

template <class P>
__device__ __forceinline__ void walk32(const P &pol, const Consts &k, const int *__restrict__ cell_start,
                                       const int *__restrict__ cellof, int rows,
                                       int *__restrict__ scal, const int *__restrict__ tile_list,
                                       int cap, int lds_wave,
                                       unsigned long long *__restrict__ counters) {
#pragma clang fp contract(fast)
  extern __shared__ __align__(16) unsigned char smem[];
  unsigned char *wl = wave_lds<false>(smem, lds_wave);
  int *tab = reinterpret_cast<int *>(wl);
  uint16_t *s_list = reinterpret_cast<uint16_t *>(wl + kTabBytes);
  const typename P::Lds L = P::lds(wl + kTabBytes + sizeof(uint16_t) * kList * kWave, cap);
  const int lane = tile_lane();
  const float r2cut = 4.f * (float)k.h * (float)k.h;
  if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&counters[C_PASSES], 1ull);
  unsigned npair = 0, ncand = 0, nact = 0;
  TileQueue tq = tq_begin<false>(scal, nullptr, tile_list, smem);
  for (int it = tq_take<false>(tq, 0); it >= 0; it = tq_take<false>(tq, 0)) {
    wave_sync();
    const int entry = tile_list[it];
    Tile t;
    tile_begin(k, cell_start, entry_tile(entry), rows, tab, t);
    entry_part(entry, t);
    const int mid = t.row_lo + (t.nrows >> 1);
    const double ox = k.x0 - k.of + t.cx * k.kh, oy = k.y0 - k.of + mid * k.kh;
    // A tile whose slices do not fit is taken in runs of fewer rows (in the
    // tile's frame, so with the same bits), no more than the tile's mean per row
    // and the row on either side let fit.  Where a single row would not, the whole
    // tile is gathered from global memory, which takes about ten times as long,
    // with all lanes at work (727k ALE particles at h = 2.5 dp, 25 per cell: 4670
    // us per step, 5790 with runs of two rows that do not fit; at h = 3 dp 8800
    // and 10400).
    const int cy0 = t.cy0, cy1 = t.cy1, own0 = t.own0, own1 = t.own1;
    int sub = cy1 - cy0;
    if (t.lq[3] > cap) {
      const int fit = cap * t.nrows / t.lq[3] - 2;
      if (fit > 0) sub = max(1, min(fit, sub / ((t.lq[3] + cap - 1) / cap)));
    }
    for (int cy = cy0; cy < cy1; cy += sub) {
      if (sub < cy1 - cy0) {
        wave_sync();  // the previous run's LDS is no longer read
        tile_begin(k, cell_start, t.cx, cy, min(cy + sub, cy1), tab, t);
        t.own0 = max(t.own0, own0);
        t.own1 = min(t.own1, own1);
      }
      const bool staged = t.lq[3] <= cap;
      if (staged)
        for (int l = lane; l < t.lq[3]; l += kWave)
          pol.stage(L, l, l - sel3(t.base, slice_of(t, l)), ox, oy);
      wave_sync();
      uint16_t *my_list = s_list + lane;
      for (int i0 = t.own0; i0 < t.own1; i0 += kWave) {
        const int i = i0 + lane;
        int li = 0, ri = 0;
        bool act = false;
        if (i < t.own1) {
          li = i + t.base[1];
          act = pol.active(i);
          ri = cellof[i] - t.cx * k.ncy - t.row_lo;
        }
        nact += act;
        const typename P::Own o = pol.own(act ? i : -1, ox, oy);
        typename P::Acc acc{};
        if (!staged) {
          if (act) {
            const int cc = cellof[i];
            const int cy = cc - t.cx * k.ncy;
            for (int dx = -1; dx <= 1; ++dx) {
              if (t.cx + dx < 0 || t.cx + dx >= k.ncx) continue;
              for (int dy = -1; dy <= 1; ++dy) {
                if (cy + dy < 0 || cy + dy >= k.ncy) continue;
                const int cl = cc + dy + dx * k.ncy;
                for (int j = cell_start[cl]; j < cell_start[cl + 1]; ++j) {
                  if (j == i) continue;
                  ++ncand;
                  const float2 pj = pol.pos_glob(j, ox, oy);
                  const float drx = o.p.x - pj.x, dry = o.p.y - pj.y;
                  const float r2 = drx * drx + dry * dry;
                  if (!(r2 < r2cut)) continue;
                  ++npair;
                  pol.pair_glob(acc, o, j, drx, dry, r2);
                }
              }
            }
          }
        } else {
          const int rlo = max(ri - 1, 0), rhi = min(ri + 2, t.nrows);
          const int a0 = tab[rlo] + t.base[0], n0 = tab[rhi] + t.base[0] - a0;
          const int a1 = tab[t.w + rlo] + t.base[1], n1 = tab[t.w + rhi] + t.base[1] - a1;
          const int a2 = tab[2 * t.w + rlo] + t.base[2], n2 = tab[2 * t.w + rhi] + t.base[2] - a2;
          const int tot = act ? n0 + n1 + n2 : 0;
          // candidates kGroup at a time from one column slice, their LDS loads
          // in flight together, appended without branches; slots past the
          // slice's range are masked (they lie in the staged area or the next
          // array of the wave's slots, positions coming first)
          const int n01 = n0 + n1;
          int cur = 0;
          while (__any(cur < tot)) {
            int cnt = 0;
            while (cur < tot && cnt <= kList - kGroup) {
              const bool in0 = cur < n0, in01 = cur < n01;
              const int end = in0 ? n0 : (in01 ? n01 : tot);
              const int j0 = cur + (in0 ? a0 : (in01 ? a1 - n0 : a2 - n01));
              const int m = min(kGroup, end - cur);
              float2 pp[kGroup];
#pragma unroll
              for (int u = 0; u < kGroup; ++u) pp[u] = pol.pos_lds(L, j0 + u);
#pragma unroll
              for (int u = 0; u < kGroup; ++u) {
                const int j = j0 + u;
                const bool cand = u < m && j != li;
                ncand += cand;
                const float drx = o.p.x - pp[u].x, dry = o.p.y - pp[u].y;
                my_list[cnt * kWave] = (uint16_t)j;
                cnt += cand && drx * drx + dry * dry < r2cut;
              }
              cur += m;
            }
            npair += cnt;
            for (int e = 0; e < cnt; ++e) {
              const int j = my_list[e * kWave];
              const float2 pj = pol.pos_lds(L, j);
              const float drx = o.p.x - pj.x, dry = o.p.y - pj.y;
              pol.pair_lds(acc, o, L, j, drx, dry, drx * drx + dry * dry);
            }
          }
        }
        if (act) pol.finish(acc, o, i);
      }
    }
  }
  wave_count(npair, ncand, nact, counters);
}

// Whether a context's cell walks take the wide form: where the lattice puts more
// into a neighbourhood than the narrow one's slots hold at most places, and no more
// than the wide one's hold.  What is not staged is gathered from global memory,
// which takes 3 to 5 times as long; the wide form's LDS leaves fewer wavefronts.
// us per step, narrow and wide, at h = 1.5, 1.6, 1.7, 2, 2.2 and 2.5 dp (89, 102,
// 115, 159, 192 and 248 in a neighbourhood): dam break of 61k particles 102 and
// 127, 236 and 137, 390 and 141, 376 and 158, 377 and 192, 481 and 509; ALE of 183k
// 397 and 600, 1132 and 700, 2379 and 686, 2390 and 805, 2536 and 969, 2607 and 3827.
// (By tiles before, which staged 99 per neighbourhood: dam break at 1.7 dp 377, ALE
// 1900.)
constexpr double kWideFrom = 97., kWideTo = 215.;
inline bool cells_wide(const tsph_ctx *c) {
  return 9. * c->cell_lattice > kWideFrom && 9. * c->cell_lattice <= kWideTo;
}

// workgroups of a cell-walk launch: those that are resident at once (the walk
// strides, so a workgroup that waits for a slot would run its whole share
// after the others'), fewer for a system that has not a cell for each
// wavefront of those.  fit: the context's record of the kernel's occupancy
// (0: not asked yet).
template <typename K>
int cell_groups(const tsph_ctx *c, K kernel, int waves, int lds, int &fit) {
  if (fit < 1 && (hipOccupancyMaxActiveBlocksPerMultiprocessor(&fit, kernel, waves * kWave, lds) !=
                      hipSuccess || fit < 1))
    fit = 1;
  const int most = c->num_cu * std::min(fit, 32 / waves), want = std::max(c->num_cu, c->n_ub / (3 * waves));
  return 8 * ((std::min(most, want) + 7) / 8);
}

// Runs of up to 64 cells, shorter ones where an XCD would get fewer than about 8
// runs: some XCDs then have one run more than others (runs of 64 against the
// shorter ones: a pass of 6k particles 12.3 and 11.2 us, of 7k 11.1 and 10.1; from
// 18k particles on no difference).
inline CellSource cell_source(const tsph_ctx *c) {
  int run = kCellRun;
  while (run > 2 && c->n_ub / 8 < 64 << run) --run;
  return {c->tile_list, c->scal + S_NTILES, (int)std::min<size_t>(tile_list_room(c), INT_MAX), run};
}

// a pair-loop launch, bracketed by HIP events while pair timing is enabled
template <typename K>
int launch_timed(tsph_ctx *c, K kernel_launch) {
  const bool timed = c->time_pairs && c->tev_used + 2 <= (int)c->tev.size();
  if (timed) TSPH_HIP(hipEventRecord(c->tev[c->tev_used], c->stream));
  kernel_launch();
  TSPH_HIP(hipGetLastError());
  if (timed) {
    TSPH_HIP(hipEventRecord(c->tev[c->tev_used + 1], c->stream));
    c->tev_used += 2;
  }
  return 0;
}

}  // namespace tiles
}  // namespace tsph
