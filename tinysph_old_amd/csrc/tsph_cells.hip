// Cell-list build: the device form of Clear_cells + Particle_To_Cell
// (src/SPH_find_pairs.h:45-92).
//
//   1. k_hash     cell id of every particle (reference truncation) and its
//                 arrival rank in the cell; lanes of a wavefront that fall in
//                 the same cell share one atomic increment (the input is in
//                 cell order from the previous build, so a wavefront spans only
//                 a handful of cells); the particle's seq goes to that place
//                 in the cell's row; removed particles go to the extra bucket
//                 `ncells`
//   2. scan       exclusive scan of the per-cell counts -> cell_start (CSR);
//                 also lists the non-empty pair-loop tiles
//   3. k_reorder  each particle ranks its seq among those in its cell's row
//                 (reference particle order), which makes the result identical
//                 to the reference's serial push_back in ascending particle
//                 index and independent of the atomic arrival order, and moves
//                 the SoA fields to the ranked slot; also lists the wall
//                 particles for the wall-density gathers and clears the counts
//
// This is a one-digit counting sort on the cell key (the key range is the cell
// count, so a single digit covers it and its scan is the cell-start table the
// pair loops need anyway); the rank in step 3 supplies the stability.  With the
// rows a build is three launches, one fewer where the build before took its
// hash, and one fewer on grids of up to 65k cells, whose scan runs beside the
// reorder (the bins: kBinMax);
// a placement pass between scan and reorder (each slot's source, then the
// reorder as a gather) measured 4.7 us more per build on 6k to 50k particles
// and 8 of 271 us per step on 740k (the FP32-pair dam break: 271 -> 259 us).
// All passes read the particle count from device memory, so the sequence can
// be captured in a HIP graph.  The per-cell counters are cleared by the reorder
// that follows their scan, so no separate clearing pass is needed.
#include "tsph_internal.h"
#include "tsph_physics.h"
#include "tsph_tiles.h"
#include "tsph_walls.h"

namespace tsph {

namespace {

constexpr int kScanBlock = 256;
// cells per thread of the scan: 4 for grids of up to kScanWide cells, 16 above
// (so that grids of up to 4M cells keep at most 1024 blocks: one look-back round)
constexpr int kScanWide = 1 << 20;
inline int scan_items(const tsph_ctx *c) { return c->ncells_tot + 1 <= kScanWide ? 4 : 16; }

// blocks of the cell-list scan (ncells + 1 counts)
inline int scan_blocks(const tsph_ctx *c) {
  const int tile = kScanBlock * scan_items(c);
  return (c->ncells_tot + 1 + tile - 1) / tile;
}

__device__ __forceinline__ unsigned long long lanemask_lt() {
  return (1ull << (threadIdx.x & 63)) - 1ull;
}

// PRED: the cell of the position the symplectic predictor gives (the
// predictor itself is applied by the reorder that follows).  DECIDE: the
// removal decision of RemoveParticlesOutOfDomain (k_rm_decide's) is taken here,
// from the removal states of the corrector that precedes the build.  The
// reference positions of removed particles are marked absent by the reorder
// (or k_scatter), so no decision in this pass reads a state that this pass changes.
// The wall-density pass that precedes a build in the symplectic step (WALLS:
// TSPH_WALL_MDBC or TSPH_WALL_BT; 0: none) runs in the first wb.walls +
// wb.sweep wavefronts of the hash launch, or of the scan launch where the
// build needs no hash, beside that pass rather than before it: it reads the
// previous cell list and writes wall densities, the hash reads positions and
// writes the new cell counts, the scan the new cell offsets.
using walls::WallPass;
using walls::wall_wave;

// global cell of a particle at r (counted and clamped beyond its case's grid)
__device__ __forceinline__ int hash_cell(const Consts &k, double2 r,
                                         unsigned long long *__restrict__ counters) {
  const int cx = cell_coord(r.x, k.x0, k.of, k.kh);
  const int cy = cell_coord(r.y, k.y0, k.of, k.kh);
  int c = cy + cx * k.ncy;  // POS(x,y) = y + x*Y, src/SPH_defs.h:36
  if (c < 0 || c >= k.ncells) {
    // undefined behaviour in the reference; counted and clamped here
    atomicAdd(&counters[C_OUTGRID], 1ull);
    c = c < 0 ? 0 : k.ncells - 1;
  }
  return c + k.cell_base;  // the case's segment of the global cell range
}

// counts the lanes' particles (live lanes) into their cells c: the lanes of a
// wavefront that share a cell are grouped, and the lowest lane of each group
// does the atomic.  rank() gives each particle's arrival rank once the atomic
// has returned.
struct CellCount {
  int leader, base;
  unsigned before;  // lanes of the group before this one
  __device__ __forceinline__ CellCount(bool live, int c, int *__restrict__ cell_count,
                                       int *__restrict__ bin) {
    const int lane = threadIdx.x & 63;
    unsigned long long rem = __ballot(live);
    leader = 0;
    unsigned long long grp = 0;
    while (rem) {
      const int l = __builtin_ctzll(rem);
      const int key = __shfl(c, l, 64);
      const unsigned long long m = __ballot(c == key) & rem;
      if ((m >> lane) & 1ull) {
        leader = l;
        grp = m;
      }
      rem &= ~m;
    }
    before = __popcll(grp & lanemask_lt());
    base = 0;
    if (live && lane == leader) base = atomicAdd(&cell_count[c], __popcll(grp));
    if (bin) {  // one add per bin and wavefront: few addresses, many wavefronts
      const int b = c / kBinCells;
      for (rem = __ballot(live); rem;) {
        const int l = __builtin_ctzll(rem);
        const unsigned long long m = __ballot(b == __shfl(b, l, 64)) & rem;
        if (lane == l) atomicAdd(&bin[b], __popcll(m));
        rem &= ~m;
      }
    }
  }
  __device__ __forceinline__ int rank() const { return __shfl(base, leader, 64) + before; }
};

// What a build clears for the one after it, which shares its buffers with the
// one before: in its hash, or in its reorder if the build before took its hash
// (that reorder takes no hash itself).
struct Clear {
  int *word[3];  // cell counts, bins, row heads
  int n4[3];     // int4 words of each
};
__device__ __forceinline__ void clear_next(const Clear &cl, int i, int stride) {
#pragma unroll
  for (int a = 0; a < 3; ++a)
    for (int k = i; k < cl.n4[a]; k += stride)
      reinterpret_cast<int4 *>(cl.word[a])[k] = make_int4(0, 0, 0, 0);
}

// The rows in which a hash leaves the seqs of every cell's particles, in arrival
// order, for the reorder to rank: `width` entries per cell, the rest of a
// fuller cell chained by input slot (link, one more than the slot; 0 ends) from
// one of kRowHeads heads.  width == 0: no rows (the hash stores arrival ranks).
struct CellRows {
  uint32_t *seq;
  int *head, *link;
  int width;
};

// slot i (seq q) as the rank-th arrival of cell c
__device__ __forceinline__ void put_row(const CellRows &rw, int c, int rank, int i, uint32_t q) {
  if (rank < rw.width) rw.seq[(size_t)c * rw.width + rank] = q;
  else rw.link[i] = atomicExch(&rw.head[c & (kRowHeads - 1)], i + 1);
}

template <bool PRED, bool DECIDE, int WALLS>
__global__ void k_hash(const double2 *__restrict__ r, const double2 *__restrict__ v,
                       uint8_t *__restrict__ type,
                       const uint32_t *__restrict__ seq, const int *__restrict__ scal, Consts k0,
                       const Consts *__restrict__ cases, const uint8_t *__restrict__ cid, double dt0,
                       int ncells_tot, int *__restrict__ cell_count, int *__restrict__ hcell,
                       int *__restrict__ hrank, CellRows rows, int *__restrict__ bin, Clear cl,
                       uint8_t *__restrict__ seqstate,
                       unsigned long long *__restrict__ counters, WallPass wp) {
  int hb = blockIdx.x;  // hash workgroup
  if (WALLS) {
    __shared__ __align__(16) double s_terms[walls::kTerms];
    const int b = blockIdx.x;  // (64 threads)
    if (b < wp.walls + wp.sweep) {
      wall_wave<WALLS>(b, wp, k0, cases, scal, s_terms);
      return;
    }
    hb = b - wp.walls - wp.sweep;
  }
  const int n = scal[S_NP];
  const int i = hb * blockDim.x + threadIdx.x;
  const bool live = i < n;
  int c = -1;
  uint32_t mine = 0;
  if (live) {
    mine = seq[i];
    bool removed = type[i] == kRemoved;
    if (DECIDE && !removed && removal_decided(seqstate, mine)) {
      removed = true;
      type[i] = kRemoved;
      atomicAdd(&counters[C_REMOVED], 1ull);
    }
    if (removed) {
      c = ncells_tot;
    } else {
      const Consts k = case_consts(k0, cases, cid, i);
      double2 ri = r[i];
      if (PRED) ri = predicted_r(ri, v[i], cases ? k.dt : dt0);
      c = hash_cell(k, ri, counters);
    }
  }
  const int rank = CellCount(live, c, cell_count, bin).rank();
  if (live) {
    hcell[i] = c;
    if (!rows.width) hrank[i] = rank;
    else if (c != ncells_tot) put_row(rows, c, rank, i, mine);
  }
  clear_next(cl, i, (gridDim.x - (WALLS ? wp.walls + wp.sweep : 0)) * blockDim.x);
}

template <int NT>
__device__ __forceinline__ int block_exclusive_scan(int v, int *lds, int &total) {
  constexpr int NW = NT / 64;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) lds[wid] = x;
  __syncthreads();
  int wo = 0, t = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const int s = lds[w];
    if (w < wid) wo += s;
    t += s;
  }
  total = t;
  __syncthreads();
  return wo + x - v;
}

// The pair loops' tiles (runs of `rows` cells of a grid column, per case) are
// listed by the scan too: a tile belongs to the scan block that holds its
// first cell.  A block stages its counts in LDS with the counts of the next
// kMaxTileRows cells after it, marks the tiles whose first cell is in the
// block (non-empty: one of their cells holds a particle), and lists them in
// tile order.  The counts are cleared later, by the reorder, so the scan reads
// them intact (the fallback of a stalled block included).
struct TileScan {
  int ncy, ncells, cell_base;  // the single case (cases == nullptr)
  const Consts *cases;
  const int *tile_base;
  int ncases;
  int rows;
  int *list;
  // with cost_in (one cost table: tile t at cost_in[kCostTables t]): each
  // listed tile's cost (or own-particle estimate) at its list position in
  // cost_list, for the chunk cut of a pooled pass
  const int *cost_in;
  int *cost_list;
  CostEstimate cm;  // the estimate for a tile without a recorded cost
  bool split;  // list the entries of a static walk (tiles::entry_part)
  // with cost_list: per scan block, the listed tiles' summed cost and the
  // list position of the first (tiles::cut_chunks_scan)
  int *blk_cost, *blk_tile0;
};

// the case whose cell range holds cell c (batched grids)
__device__ __forceinline__ int case_of(const TileScan &ts, int c) {
  int lo = 0, hi = ts.ncases;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (ts.cases[mid].cell_base <= c) lo = mid;
    else hi = mid;
  }
  return lo;
}

// the grid geometry of one case, in registers: cells [cell_base, next) belong
// to it (next: the following case's first cell)
struct CaseGrid {
  int cse, cell_base, ncy, ncells, tile_base, next;
};

__device__ __forceinline__ CaseGrid case_grid(const TileScan &ts, int cse) {
  if (!ts.cases) return {0, ts.cell_base, ts.ncy, ts.ncells, 0, INT_MAX};
  const Consts &k = ts.cases[cse];
  return {cse, k.cell_base, k.ncy, k.ncells, ts.tile_base[cse],
          cse + 1 < ts.ncases ? ts.cases[cse + 1].cell_base : INT_MAX};
}

// the grid of cell c, starting from g (cells ascending); a reload only at a
// case boundary
__device__ __forceinline__ void advance_grid(const TileScan &ts, int c, CaseGrid &g) {
  if (c < g.next) return;
  int cse = g.cse;
  while (cse + 1 < ts.ncases && ts.cases[cse + 1].cell_base <= c) ++cse;
  g = case_grid(ts, cse);
}

// {tile, cells of the tile} if cell c (in grid g) is a tile's first cell,
// else {-1, 0}
__device__ __forceinline__ int2 tile_at(const TileScan &ts, int c, const CaseGrid &g) {
  const int lc = c - g.cell_base;
  if (lc < 0 || lc >= g.ncells) return make_int2(-1, 0);
  const int cx = lc / g.ncy, cy = lc - cx * g.ncy;
  if (cy % ts.rows) return make_int2(-1, 0);
  const int t = g.tile_base + cx * ((g.ncy + ts.rows - 1) / ts.rows) + cy / ts.rows;
  return make_int2(t, min(ts.rows, g.ncy - cy));
}

// entries of a tile with `own` particles
__device__ __forceinline__ int tile_entries(const TileScan &ts, int own) {
  return own == 0 ? 0 : ts.split && own > tiles::kWave ? 2 : 1;
}

// the thread's counts (v) and, for the first kMaxTileRows threads, one count
// of the next block (halo)
template <int IT>
__device__ __forceinline__ void load_counts(const int *__restrict__ in, int len, int block,
                                            int (&v)[IT], int &halo) {
  constexpr int kTile = kScanBlock * IT;
  const int b0 = block * kTile, base = b0 + threadIdx.x * IT;
#pragma unroll
  for (int j = 0; j < IT; ++j) v[j] = (base + j < len) ? in[base + j] : 0;
  const int c = b0 + kTile + threadIdx.x;
  halo = threadIdx.x < kMaxTileRows && c < len ? in[c] : 0;
}

// the block's counts + halo staged in s_cnt; tl[j] >= 0: cell base + j
// starts a non-empty tile; returns the number of such tiles.  On a batched
// grid one thread finds the case of the block's first cell (s_case) and every
// thread steps from there to its own cells.
template <int IT>
__device__ __forceinline__ int stage_counts(int len, int block, const TileScan ts,
                                            const int (&v)[IT], int halo, int (&tl)[IT],
                                            int (&own)[IT], int *s_cnt, int *s_case) {
  constexpr int kTile = kScanBlock * IT;
  const int b0 = block * kTile, base = b0 + threadIdx.x * IT;
#pragma unroll
  for (int j = 0; j < IT; ++j) s_cnt[threadIdx.x * IT + j] = v[j];
  if (threadIdx.x < kMaxTileRows) s_cnt[kTile + threadIdx.x] = halo;
  if (ts.cases && threadIdx.x == 0) *s_case = case_of(ts, b0);
  __syncthreads();
  int nt = 0;
  CaseGrid g = case_grid(ts, ts.cases ? *s_case : 0);
  advance_grid(ts, base, g);
#pragma unroll
  for (int j = 0; j < IT; ++j) {
    advance_grid(ts, base + j, g);
    const int2 tn = base + j < len ? tile_at(ts, base + j, g) : make_int2(-1, 0);
    int o = 0;
    for (int r = 0; r < tn.y; ++r) o += s_cnt[threadIdx.x * IT + j + r];
    tl[j] = o ? tn.x : -1;
    own[j] = o;
    nt += tile_entries(ts, o);
  }
  return nt;
}

// Single-pass scan with decoupled look-back.  Every block publishes its sums
// (cells, tiles) in one 64-bit word (bits 0-30 cells, 31-61 tiles, 62 set
// once the word holds the inclusive prefix instead of the block's own sums,
// 63 set once written).  A block then walks back over the words of the blocks
// before it, 1024 at a time (four per thread), until it meets an inclusive
// prefix, adds up what it passed, and publishes its own inclusive prefix
// (a grid of at most 1024 blocks reads all its words in one round and
// publishes no inclusive prefixes).  Blocks cover 256 IT cells: IT = 16 above
// 1M cells keeps grids of up to 4M cells in one round.
// Every scan clears the words of the next (two sets take turns).  Blocks are
// dispatched in index order, so a block waits only for blocks that have started, and those
// publish their own sums before they wait themselves.  A block whose wait
// exceeds spin_limit polls (the context's scan_wait; -1: it does not poll)
// forms its sums from the counts of the cells before it instead (and counts
// the stall): a late publisher costs time, never correctness, and every wait
// ends.
constexpr int kLookBack = 4;  // words per thread and look-back round
constexpr unsigned long long kScanField = 0x7fffffffull;
constexpr unsigned long long kScanSet = 1ull << 63, kScanIncl = 1ull << 62;

__device__ __forceinline__ unsigned long long scan_word(int cells, int tiles, bool incl) {
  return kScanSet | (incl ? kScanIncl : 0ull) | ((unsigned long long)tiles << 31) |
         (unsigned long long)cells;
}

// block-wide sums of a and b, and the minimum of m
__device__ __forceinline__ void block_reduce3(int &a, int &b, int &m, int *lds) {
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b += __shfl_xor(b, o, 64);
    m = min(m, __shfl_xor(m, o, 64));
  }
  const int wid = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    lds[3 * wid] = a;
    lds[3 * wid + 1] = b;
    lds[3 * wid + 2] = m;
  }
  __syncthreads();
  a = b = 0;
  m = INT_MAX;
  for (int w = 0; w < kScanBlock / 64; ++w) {
    a += lds[3 * w];
    b += lds[3 * w + 1];
    m = min(m, lds[3 * w + 2]);
  }
  __syncthreads();
}

struct ScanArgs {
  const int *in;  // the cells' counts, len of them
  int len;
  unsigned long long *state, *state_next;
  int *out;
  TileScan ts;
  int spin_limit;
};

// block blk of nb
template <int IT>
__device__ __forceinline__ void scan_block(const ScanArgs &sa, int blk, int nb,
                                           int *__restrict__ scal,
                                           unsigned long long *__restrict__ counters) {
  __shared__ int lds[3 * kScanBlock / 64];
  constexpr int kTile = kScanBlock * IT;
  __shared__ int s_cnt[kTile + kMaxTileRows];
  __shared__ int s_case;
  const int *__restrict__ in = sa.in;
  const int len = sa.len, spin_limit = sa.spin_limit;
  unsigned long long *__restrict__ state = sa.state;
  int *__restrict__ out = sa.out;
  const TileScan &ts = sa.ts;
  int v[IT], tl[IT], own[IT], halo;
  load_counts<IT>(in, len, blk, v, halo);
  const int nt = stage_counts<IT>(len, blk, ts, v, halo, tl, own, s_cnt, &s_case);
  // the listed tiles' recorded costs, in flight during the look-back
  int w[IT];
#pragma unroll
  for (int j = 0; j < IT; ++j) w[j] = ts.cost_in && tl[j] >= 0 ? ts.cost_in[kCostTables * tl[j]] : 0;
  int s = 0;
#pragma unroll
  for (int j = 0; j < IT; ++j) s += v[j];
  int total, tiles;
  int ex = block_exclusive_scan<kScanBlock>(s, lds, total);
  int et = block_exclusive_scan<kScanBlock>(nt, lds, tiles);
  // a grid that one look-back round covers needs no inclusive prefixes
  const bool chain = nb > kLookBack * kScanBlock;
  if (threadIdx.x == 0)
    __hip_atomic_store(&state[blk], scan_word(total, tiles, chain && blk == 0), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  // pc, pt = sums of the blocks before this one.  Look-back: a round reads
  // the words of the kLookBack * kScanBlock nearest blocks not yet covered
  // (entry j = thread + kScanBlock q: block hi - j), all loads in flight
  // together.
  int pc = 0, pt = 0;
  bool stalled = false;
  if (!chain) {
    // one round over all the blocks before this one, farthest first (they
    // published first)
    for (int b = threadIdx.x; b < blk && !stalled; b += kScanBlock) {
      unsigned long long word = 0;
      for (int spin = 0;; ++spin) {
        if (spin > spin_limit) {
          stalled = true;
          break;
        }
        word = __hip_atomic_load(&state[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (word & kScanSet) break;
        __builtin_amdgcn_s_sleep(1);
      }
      pc += (int)(word & kScanField);
      pt += (int)((word >> 31) & kScanField);
    }
    if (!__syncthreads_or(stalled)) {
      int unused = 0;
      block_reduce3(pc, pt, unused, lds);
    }
  }
  for (int hi = chain ? blk - 1 : -1; hi >= 0;) {
    unsigned long long word[kLookBack];
#pragma unroll
    for (int q = 0; q < kLookBack; ++q) {
      const int b = hi - (int)threadIdx.x - kScanBlock * q;
      // before block 0: an empty inclusive prefix
      word[q] = b < 0 ? kScanSet | kScanIncl
                : spin_limit >= 0 ? __hip_atomic_load(&state[b], __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT)
                                  : 0ull;
    }
#pragma unroll
    for (int q = 0; q < kLookBack; ++q) {
      const int b = hi - (int)threadIdx.x - kScanBlock * q;
      for (int spin = 1; !(word[q] & kScanSet) && !stalled; ++spin) {
        if (spin > spin_limit) {
          stalled = true;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
        word[q] = __hip_atomic_load(&state[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    if (__syncthreads_or(stalled)) break;
    // the nearest inclusive prefix ends the walk; the words up to it count
    int f = INT_MAX, c = 0, t = 0;
    if (chain) {
#pragma unroll
      for (int q = 0; q < kLookBack; ++q)
        if (word[q] & kScanIncl) f = min(f, (int)threadIdx.x + kScanBlock * q);
      block_reduce3(c, t, f, lds);
    }
#pragma unroll
    for (int q = 0; q < kLookBack; ++q)
      if ((int)threadIdx.x + kScanBlock * q <= f) {
        c += (int)(word[q] & kScanField);
        t += (int)((word[q] >> 31) & kScanField);
      }
    int unused = 0;
    block_reduce3(c, t, unused, lds);
    pc += c;
    pt += t;
    if (f != INT_MAX) break;
    hi -= kLookBack * kScanBlock;
  }
  if (__syncthreads_or(stalled)) {
    // the same sums from the counts of the cells before the block
    pc = pt = 0;
    for (int c = threadIdx.x; c < blk * kTile; c += kScanBlock) {
      pc += in[c];
      const int2 tn = tile_at(ts, c, case_grid(ts, ts.cases ? case_of(ts, c) : 0));
      int own = 0;
      for (int r = 0; r < tn.y; ++r) own += in[c + r];
      pt += tile_entries(ts, own);
    }
    int unused = 0;
    block_reduce3(pc, pt, unused, lds);
    if (threadIdx.x == 0) atomicAdd(&counters[C_SCANSTALL], 1ull);
  }
  if (chain && threadIdx.x == 0 && blk > 0)
    __hip_atomic_store(&state[blk], scan_word(pc + total, pt + tiles, true), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  ex += pc;
  et += pt;
  const int base = blk * kTile + threadIdx.x * IT;
  int csum = 0;
#pragma unroll
  for (int j = 0; j < IT; ++j) {
    if (base + j < len) out[base + j] = ex;
    ex += v[j];
    if (tl[j] >= 0) {
      if (ts.cost_list) {
        const int wc = w[j] > 0 ? w[j] : ts.cm.own * own[j] + ts.cm.tile;
        ts.cost_list[et] = wc;
        csum += wc;
      }
      if (ts.split && own[j] > tiles::kWave) {
        ts.list[et++] = tl[j] | tiles::kTileFirst;
        ts.list[et++] = tl[j] | tiles::kTileRest;
      } else {
        ts.list[et++] = tl[j];
      }
    }
  }
  if (ts.cost_list) {
    int unused0 = 0, unused1 = 0;
    block_reduce3(csum, unused0, unused1, lds);
    if (threadIdx.x == 0) {
      ts.blk_cost[blk] = csum;
      ts.blk_tile0[blk] = pt;
    }
  }
  if (threadIdx.x == 0) sa.state_next[blk] = 0;
  if (threadIdx.x == 0 && blk == nb - 1) {
    out[len] = pc + total;
    scal[S_NTILES] = pt + tiles;
  }
}

// the scan, with the wall pass (WALLS) in the last wall_groups workgroups, a
// wavefront's share per wavefront
template <int IT, int WALLS>
__global__ __launch_bounds__(kScanBlock, WALLS ? 4 : 1) void k_scan(ScanArgs sa, int *__restrict__ scal,
                                                     unsigned long long *__restrict__ counters,
                                                     int wall_groups, WallPass wp, Consts k0,
                                                     const Consts *__restrict__ cases) {
  const int nb = gridDim.x - (WALLS ? wall_groups : 0), blk = blockIdx.x;
  if (WALLS && blk >= nb) {
    constexpr int kWaves = kScanBlock / 64;
    __shared__ __align__(16) double s_terms[kWaves * walls::kTerms];
    const int wid = threadIdx.x >> 6, b = (blk - nb) * kWaves + wid;
    if (b < wp.walls + wp.sweep)
      wall_wave<WALLS ? WALLS : TSPH_WALL_MDBC>(b, wp, k0, cases, scal,
                                                s_terms + wid * walls::kTerms);
    return;
  }
  scan_block<IT>(sa, blk, nb, scal, counters);
}

// Placement without rows: arrival position of every particle (cell_start[cell]
// + its arrival rank from the hash), whose cells k_order / k_order_tiles order
// in place.  Also marks the reference positions of removed particles (the
// trailing bucket) absent in the removal states.  The first `cuts` workgroups (one wavefront per scan block)
// cut the new tile list into the chunks of the pooled pair pass that follows
// from the scan's per-block sums (cut_chunks_scan), beside the placement.
constexpr int kScatterBlock = 256;
// ordering workgroups (of 256 threads) per compute unit, single case
constexpr int kOrderWaves = 4;
// the chunk cut's share of a launch of kScatterBlock-thread workgroups
struct ChunkCut {
  int cuts;  // cutting workgroups (0: no cut)
  int scan_blocks, groups;
  const int *list_cost, *blk_cost, *blk_tile0;
  int *bound;
};
__device__ __forceinline__ void cut_wave(const ChunkCut &cc, const int *__restrict__ scal) {
  __shared__ long long red[kScatterBlock / 64], pfx[kScatterBlock / 64];
  tiles::cut_chunks_scan(scal, cc.list_cost, cc.blk_cost, cc.blk_tile0, cc.scan_blocks, cc.groups,
                         cc.bound, blockIdx.x, red, pfx);
}
__global__ __launch_bounds__(kScatterBlock) void k_scatter(
    const int *__restrict__ scal, const int *__restrict__ hcell, const int *__restrict__ hrank,
    const int *__restrict__ cell_start, int *__restrict__ arrival, int *__restrict__ cellof,
    int ncells_tot, const uint32_t *__restrict__ seq, uint8_t *__restrict__ seqstate,
    ChunkCut cc) {
  if ((int)blockIdx.x < cc.cuts) {
    cut_wave(cc, scal);
    return;
  }
  const int n = scal[S_NP], blk = blockIdx.x - cc.cuts;
  const int i = blk * kScatterBlock + threadIdx.x;
  if (i >= n) return;
  const int c = hcell[i];
  if (c == ncells_tot) seqstate[seq[i]] = 0;
  const int pos = cell_start[c] + hrank[i];
  arrival[pos] = i;
  cellof[pos] = c;
}

// Orders each cell's slots by reference order (seq).  Cells of up to 16
// particles are sorted in registers (all loads in flight together, then an
// odd-even transposition network); larger cells use an insertion sort.
// Also clears the per-cell counts (ncells + 1 of them) for the next build.
// orders cell c's slots by seq
__device__ __forceinline__ void order_cell(const int *__restrict__ cell_start, int c,
                                           const uint32_t *__restrict__ seq,
                                           int *__restrict__ perm) {
  constexpr int R = 16;
  const int s = cell_start[c], e = cell_start[c + 1];
  const int cnt = e - s;
  if (cnt <= 1) return;
  if (cnt <= R) {
    int pv[R];
    uint32_t kv[R];
#pragma unroll
    for (int a = 0; a < R; ++a) {
      pv[a] = a < cnt ? perm[s + a] : 0;
      kv[a] = 0xffffffffu;
    }
#pragma unroll
    for (int a = 0; a < R; ++a)
      if (a < cnt) kv[a] = seq[pv[a]];
    bool sorted = true;
#pragma unroll
    for (int a = 1; a < R; ++a) sorted &= kv[a - 1] <= kv[a];
    if (sorted) return;
#pragma unroll
    for (int pass = 0; pass < R; ++pass) {
#pragma unroll
      for (int a = pass & 1; a + 1 < R; a += 2) {
        if (kv[a] > kv[a + 1]) {
          const uint32_t tk = kv[a]; kv[a] = kv[a + 1]; kv[a + 1] = tk;
          const int tp = pv[a]; pv[a] = pv[a + 1]; pv[a + 1] = tp;
        }
      }
    }
#pragma unroll
    for (int a = 0; a < R; ++a)
      if (a < cnt) perm[s + a] = pv[a];
    return;
  }
  for (int a = s + 1; a < e; ++a) {
    const int pa = perm[a];
    const uint32_t ka = seq[pa];
    int b = a - 1;
    while (b >= s) {
      const int pb = perm[b];
      if (seq[pb] <= ka) break;
      perm[b + 1] = pb;
      --b;
    }
    perm[b + 1] = pa;
  }
}

// per cell of a batched grid: its slots ordered by seq, its count cleared
__global__ void k_order(const int *__restrict__ cell_start, int ncells,
                        const uint32_t *__restrict__ seq, int *__restrict__ perm,
                        int *__restrict__ cell_count) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c <= ncells) cell_count[c] = 0;
  if (c < ncells) order_cell(cell_start, c, seq, perm);
}

// The same over the cells of the listed (non-empty) tiles only, for a single
// case: every occupied cell lies in a listed tile, so the other cells need
// neither ordering nor clearing (their counts are 0).  A bounded grid strides
// over the (tile, row) items.
__global__ void k_order_tiles(const int *__restrict__ cell_start, const int *__restrict__ scal,
                              const int *__restrict__ tile_list, int rows, int ncy, int ncells,
                              const uint32_t *__restrict__ seq, int *__restrict__ perm,
                              int *__restrict__ cell_count) {
  const int ntiles = scal[S_NTILES];
  if (blockIdx.x == 0 && threadIdx.x == 0) cell_count[ncells] = 0;  // the removed bucket
  const int items = ntiles * rows;
  const int nty = (ncy + rows - 1) / rows;
  for (int item = blockIdx.x * blockDim.x + threadIdx.x; item < items;
       item += gridDim.x * blockDim.x) {
    const int it = item / rows, r = item - it * rows;
    const int tile = tile_list[it];
    const int cx = tile / nty, cy = (tile - cx * nty) * rows + r;
    if (cy >= ncy) continue;
    const int c = cx * ncy + cy;
    cell_count[c] = 0;
    order_cell(cell_start, c, seq, perm);
  }
}

// rank of the particle with seq `mine` in cell c (of cnt particles): the number
// of the cell's particles that precede it in seq.  The row is read 16 entries
// at a time, all of them in flight together (one round for all but the fullest
// cells); the chained ones one by one.
__device__ __forceinline__ int rank_in_cell(const CellRows &rw, const int *__restrict__ hcell,
                                            const uint32_t *__restrict__ seq, int n, int c, int cnt,
                                            uint32_t mine) {
  const uint4 *row = reinterpret_cast<const uint4 *>(rw.seq + (size_t)c * rw.width);
  const int in_row = min(cnt, rw.width);
  int rank = 0;
  for (int a = 0; a < in_row; a += 16) {
    uint4 q[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      q[u] = a + 4 * u < in_row ? row[a / 4 + u] : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int o = a + 4 * u;
      rank += (o < in_row && q[u].x < mine) + (o + 1 < in_row && q[u].y < mine) +
              (o + 2 < in_row && q[u].z < mine) + (o + 3 < in_row && q[u].w < mine);
    }
  }
  if (cnt > rw.width) {
    int y = rw.head[c & (kRowHeads - 1)];
    for (int left = n; y > 0 && left > 0; --left) {
      rank += hcell[y - 1] == c && seq[y - 1] < mine;
      y = rw.link[y - 1];
    }
  }
  return rank;
}

// exclusive prefix of the bins (a multiple of kBinChunk of them) into pre, by
// one workgroup; returns their sum
__device__ __forceinline__ int scan_bins(const int *__restrict__ bin, int bins, int *pre) {
  constexpr int kU = 4, kWaves = kScanBlock / 64;
  __shared__ int tot[kU * kWaves];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, chunks = bins / kBinChunk;
  int carry = 0;
  for (int c0 = 0; c0 < chunks; c0 += kU) {
    int4 q[kU];
    int inc[kU], off[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u)
      q[u] = c0 + u < chunks
                 ? reinterpret_cast<const int4 *>(bin)[(c0 + u) * kScanBlock + threadIdx.x]
                 : make_int4(0, 0, 0, 0);
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      if (c0 + u >= chunks) break;
      q[u].y += q[u].x;
      q[u].z += q[u].y;
      q[u].w += q[u].z;
      int x = q[u].w;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
      }
      inc[u] = x;
      if (lane == 63) tot[u * kWaves + wid] = x;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      if (c0 + u >= chunks) break;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        if (w == wid) off[u] = carry;
        carry += tot[u * kWaves + w];
      }
      const int ex = off[u] + inc[u] - q[u].w;
      reinterpret_cast<int4 *>(pre)[(c0 + u) * kScanBlock + threadIdx.x] =
          make_int4(ex, ex + q[u].x, ex + q[u].y, ex + q[u].z);
    }
    __syncthreads();
  }
  return carry;
}

// particles in the cells of c's bin before c; cnt: those in c
__device__ __forceinline__ int bin_offset(const int *__restrict__ cell_count, int c, int &cnt) {
  const int4 *q = reinterpret_cast<const int4 *>(cell_count) + c / kBinCells * (kBinCells / 4);
  const int m = c % kBinCells;
  int4 v[kBinCells / 4];
#pragma unroll
  for (int u = 0; u < kBinCells / 4; ++u) v[u] = q[u];
  int s = 0;
  cnt = 0;
#pragma unroll
  for (int u = 0; u < kBinCells; ++u) {
    const int4 &w = v[u / 4];
    const int x = u % 4 == 0 ? w.x : u % 4 == 1 ? w.y : u % 4 == 2 ? w.z : w.w;
    s += u < m ? x : 0;
    cnt = u == m ? x : cnt;
  }
  return s;
}

// what a build moves beside the fields that every build does: the old state
// (PRED: writes it), pressures (other than the inlet and outlet particles',
// which no EOS rewrites), the permutation
enum : unsigned { kMoveOlds = 1, kMoveP = 2, kMovePerm = 4 };

// Moves every field to its slot of the new order (the state after the build is
// the reference's state, permuted; perm records the permutation), lists the
// wall particles and sets the new particle count (removed particles are
// dropped).  RANK: thread x moves input slot x to the slot that the hash's rows
// give it (reads in a row, writes nearly so: few particles change cells in a
// step), and does the placement's other work: the cell of each slot, the cell
// counts cleared for the next build, removed particles marked absent, the
// pooled pass's chunk cut (cc) in the first workgroups.
// Otherwise thread x fills slot x from where the placement says.
// SCAN (with RANK): the scan runs in the first workgroups of the launch; the
// others find their cells' offsets from the bins, which every workgroup scans
// in LDS.
// With EOS the pressure is recomputed as Density_to_pressure does
// (src/SPH_pressure.h:65-89) and the FP32 records of the mixed path are
// written, for the step sequences in which that stage follows the cell build.
// With PRED the symplectic predictor (src/SPH_integration.h:266-287) is
// applied to the moved particles, for the step sequences in which it
// immediately precedes the cell build.  With NEXT the hash of the next step's
// first build is taken on the way (next_count, next_hcell, next_rows or
// next_hrank): that build sorts by the positions the predictor will give,
// which need no forces, so a step inside a run of steps starts with its scan.
// ad_skip (a type mask): a and drho of those types are not moved, for the step
// sequences in which a pair pass that overwrites them for exactly those types
// follows the build.
template <bool EOS, bool PRED, bool RANK, bool NEXT, bool SCAN>
__global__ __launch_bounds__(kScatterBlock, SCAN ? 1 : 6) void k_reorder(
    const int *__restrict__ cell_start, int ncells, int n_ub, const int *__restrict__ hcell,
    CellRows rows, const int *__restrict__ bin, int nbins, Clear cl, ScanArgs sa,
    int *__restrict__ perm,
    int *__restrict__ cell_count, uint8_t *__restrict__ seqstate, ChunkCut cc, Soa src, Soa dst,
    int *__restrict__ scal, int2 *__restrict__ wall_list, int *__restrict__ cellof, Consts k0,
    const Consts *__restrict__ cases, Mixed mx, double dt0, unsigned ad_skip,
    unsigned long long *__restrict__ counters, int nwall_idx, int nwall_next, unsigned moves,
    int *__restrict__ next_count, int *__restrict__ next_bin, int *__restrict__ next_hcell,
    int *__restrict__ next_hrank, CellRows next_rows) {
  extern __shared__ __align__(16) int s_pre[];  // SCAN: the bins' offsets
  int blk = blockIdx.x;
  if (RANK) {
    if (blk < cc.cuts) {
      cut_wave(cc, scal);
      return;
    }
    blk -= cc.cuts;
  }
  if (SCAN) {
    if (blk < cc.scan_blocks) {
      scan_block<4>(sa, blk, cc.scan_blocks, scal, counters);
      return;
    }
    blk -= cc.scan_blocks;
  }
  // Every load before the first store (loads and stores complete in order, so
  // a load behind a store would wait for the store's acknowledgement too), and
  // those of the particle's fields beside those that find its slot.
  const int x = blk * kScatterBlock + threadIdx.x;
  int cell = 0, j = x;
  uint32_t mine = 0;
  uint8_t t = kRemoved;
  bool move_ad = false;
  double2 r = {}, v = {}, a = {}, r_o = {}, v_o = {}, nv = {};
  double rho = 0., drho = 0., rho_o = 0., p = 0.;
  int cid = 0;
  if (x < n_ub) {
    if (RANK) {
      cell = hcell[x];
    } else {
      j = min((unsigned)perm[x], (unsigned)(n_ub - 1));  // (slots past the last hold any value)
      if (EOS && mx.rv) cell = cellof[x];
    }
    mine = src.seq[j];
    t = src.type[j];
    r = src.r[j];
    v = src.v[j];
    rho = src.rho[j];
    if (src.cid) cid = src.cid[j];
    if (PRED) {
      a = src.a[j];
      drho = src.drho[j];
    } else if (moves & kMoveOlds) {
      r_o = src.r_o[j];
      v_o = src.v_o[j];
      rho_o = src.rho_o[j];
    }
    if (src.n) nv = src.n[j];
  }
  int n_new, n;  // RANK: n with the removed ones
  if (SCAN) {
    n = scan_bins(bin, nbins, s_pre);
    n_new = n - cell_count[ncells];
  } else {
    n_new = cell_start[ncells];
    n = RANK ? cell_start[ncells + 1] : n_new;
  }
  bool live = x < n, gone = false;
  if (RANK) {
    gone = live && cell == ncells;
    live = live && !gone;
  }
  int k = x, next_c = -1;
  unsigned bad = 0;
  Consts kc = k0;
  if (live) {
    if (RANK) {
      int cnt;
      if (SCAN) {
        k = s_pre[cell / kBinCells] + bin_offset(cell_count, cell, cnt);
      } else {
        k = cell_start[cell];
        cnt = cell_start[cell + 1] - k;
      }
      k += rank_in_cell(rows, hcell, src.seq, n, cell, cnt, mine);
    }
    if (cases && (EOS || PRED)) kc = cases[cid];
    move_ad = !((ad_skip >> t) & 1u);
    if (!PRED && move_ad) {
      a = src.a[j];
      drho = src.drho[j];
    }
    // with the EOS the old pressure is read only where it is kept
    if (!EOS || t == TSPH_OUTLET || t == TSPH_INLET) p = src.p[j];
    if (src.omega) {
      const double w0 = src.omega[j], w1 = src.omegarho[j], w2 = src.omega_o[j],
                   w3 = src.omegarho_o[j], w4 = src.domega[j], w5 = src.domegarho[j];
      const double2 u0 = src.omegav[j], u1 = src.omegav_o[j], u2 = src.domegav[j];
      dst.omega[k] = w0;
      dst.omegarho[k] = w1;
      dst.omega_o[k] = w2;
      dst.omegarho_o[k] = w3;
      dst.domega[k] = w4;
      dst.domegarho[k] = w5;
      dst.omegav[k] = u0;
      dst.omegav_o[k] = u1;
      dst.domegav[k] = u2;
      if (src.gradrho) {
        const double2 g0 = src.gradrho[j], g1 = src.gradvx[j], g2 = src.gradvy[j];
        dst.gradrho[k] = g0;
        dst.gradvx[k] = g1;
        dst.gradvy[k] = g2;
      }
    }
    if (src.v_oo) {
      const double2 u0 = src.v_oo[j];
      const double w0 = src.rho_oo[j], w1 = src.rho_tmp[j];
      dst.v_oo[k] = u0;
      dst.rho_oo[k] = w0;
      dst.rho_tmp[k] = w1;
    }
    if (src.rc) {
      const double2 u0 = src.rc[j];
      const double w0 = src.rhoc[j];
      dst.rc[k] = u0;
      dst.rhoc[k] = w0;
    }
    if (PRED) {
      r_o = r;
      v_o = v;
      rho_o = rho;
      predict(r, v, rho, a, drho, cases ? kc.dt : dt0);
    }
    if (NEXT) next_c = hash_cell(kc, predicted_r(r, v, cases ? kc.dt : dt0), counters);
    if (EOS && t != TSPH_OUTLET && t != TSPH_INLET) {
      bad = rho > 1500. || rho < 0.;
      p = tait64(rho, kc.rho0, kc.cs);
    }
  }
  const bool wall = live && t == TSPH_WALL;
  auto store = [&] {
    if (moves & kMoveOlds) {
      dst.r_o[k] = r_o;
      dst.v_o[k] = v_o;
      dst.rho_o[k] = rho_o;
    }
    dst.r[k] = r;
    dst.v[k] = v;
    if (move_ad) {
      dst.a[k] = a;
      dst.drho[k] = drho;
    }
    dst.rho[k] = rho;
    if ((moves & kMoveP) || t == TSPH_OUTLET || t == TSPH_INLET) dst.p[k] = p;
    dst.type[k] = t;
    dst.seq[k] = mine;
    if (src.cid) dst.cid[k] = cid;
    if (src.n) dst.n[k] = nv;
    if (EOS && mx.rv)
      write_mixed_record(mx, kc, cell - kc.cell_base, k, r, v, rho, p, src.n != nullptr, nv);
    if (RANK) {
      if (moves & kMovePerm) perm[k] = j;
      cellof[k] = cell;
      if (!SCAN && !bin) cell_count[cell] = 0;
    }
  };
  if (NEXT) {
    const CellCount cn(live, next_c, next_count, next_bin);
    if (live) store();
    const int rank = cn.rank();
    if (live) {
      next_hcell[k] = next_c;
      if (RANK) put_row(next_rows, next_c, rank, k, mine);
      else next_hrank[k] = rank;
    }
  } else if (live) {
    store();
  }
  if (gone) seqstate[mine] = 0;
  if (blk == 0 && threadIdx.x == 0) {
    scal[S_NP] = n_new;
    scal[nwall_next] = 0;
    if (RANK && !bin) cell_count[ncells] = 0;  // the removed bucket
  }
  clear_next(cl, x, (gridDim.x - (blockIdx.x - blk)) * kScatterBlock);
  const unsigned long long m = __ballot(wall);
  if (m) {
    const int lane = threadIdx.x & 63;
    int base = 0;
    if (lane == __builtin_ctzll(m)) base = atomicAdd(&scal[nwall_idx], __popcll(m));
    base = __shfl(base, __builtin_ctzll(m), 64);
    if (wall) wall_list[base + __popcll(m & lanemask_lt())] = make_int2(k, (int)mine);
  }
  if (EOS) {
    const unsigned long long w = __ballot(bad);
    if (w && (threadIdx.x & 63) == 0) atomicAdd(&counters[C_BADRHO], (unsigned long long)__popcll(w));
  }
}

// r_o, v_o, rho_o of slot k taken from the generation before the last build
// (cur <- alt through perm), for a build that left them behind
__global__ void k_gather_olds(const int *__restrict__ scal, const int *__restrict__ perm, Soa src,
                              Soa dst) {
  const int n = scal[S_NP];
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int j = perm[k];
  dst.r_o[k] = src.r_o[j];
  dst.v_o[k] = src.v_o[j];
  dst.rho_o[k] = src.rho_o[j];
}

// The builds' cells are ordered from rows by the reorder: wherever the context
// has rows.  Ranked against placement and ordering passes, us per step of the
// dam break: FP32 pairs 258 / 276 at 740k particles, 670 / 692 at 2.0M, 1232 /
// 1253 at 3.9M, 2279 / 2306 at 7.6M; FP64 511 / 533, 1336 / 1346, 2561 / 2574,
// 4788 / 4776 (within the runs' spread).
bool cells_ranked(const tsph_ctx *c) { return c->row_width > 0 && c->cell_order != 2; }

// the arguments of the scan of the cell counts into cs, with the tile list of
// the current tile_rows (and, for cost_table >= 0, the listed tiles' costs)
// or the list of non-empty cells
ScanArgs scan_args(tsph_ctx *c, int *cs, int cost_table, bool split, bool cells) {
  const TileScan ts{cells ? c->ncells_tot : c->k.ncy, cells ? c->ncells_tot : c->k.ncells,
                    cells ? 0 : c->k.cell_base, cells ? nullptr : c->cases, c->tile_base, c->ncases,
                    cells ? 1 : c->tile_rows, c->tile_list,
                    cost_table >= 0 ? c->scal + S_NSCAL + cost_table : nullptr,
                    cost_table >= 0 ? c->list_cost : nullptr,
                    cost_estimate(c->prm.precision == TSPH_PREC_MIXED), split, c->scan_cost,
                    c->scan_tile0};
  c->list_split = split;
  c->list_rows = cells ? kListCells : c->tile_rows;
  c->list_groups = 0;  // a pooled pass cuts the new list
  c->list_cost_table = cost_table;
  return {c->cell_count, c->ncells_tot + 1, c->scan_state, c->scan_state_next, cs, ts, c->scan_wait};
}

// the scan in a launch of its own, with walls (TSPH_WALL_*; 0: none) the wall
// pass wp beside it
int launch_scan(tsph_ctx *c, const ScanArgs &sa, int walls, const WallPass &wp) {
  const int wg = walls ? grid_for(wp.walls + wp.sweep, kScanBlock / 64) : 0;
#define TSPH_SCAN(IT, W)                                                                        \
  hipLaunchKernelGGL((k_scan<IT, W>), dim3(scan_blocks(c) + wg), dim3(kScanBlock), 0, c->stream, \
                     sa, c->scal, c->counters, wg, wp, c->k, c->cases)
#define TSPH_SCAN_W(IT)                                                                         \
  if (walls == TSPH_WALL_MDBC) TSPH_SCAN(IT, TSPH_WALL_MDBC);                                  \
  else if (walls == TSPH_WALL_BT) TSPH_SCAN(IT, TSPH_WALL_BT);                                 \
  else TSPH_SCAN(IT, 0)
  if (scan_items(c) == 4) {
    TSPH_SCAN_W(4);
  } else {
    TSPH_SCAN_W(16);
  }
#undef TSPH_SCAN_W
#undef TSPH_SCAN
  TSPH_HIP(hipGetLastError());
  return 0;
}

}  // namespace

void flip_build(tsph_ctx *c) {
  std::swap(c->cur, c->alt);
  std::swap(c->cell_start, c->cell_start_next);
  std::swap(c->cell_count, c->cell_count_next);
  std::swap(c->bin_count, c->bin_count_next);
  std::swap(c->scan_state, c->scan_state_next);
  std::swap(c->hcell, c->hcell_next);
  std::swap(c->hrank, c->hrank_next);
  std::swap(c->row_seq, c->row_seq_next);
  std::swap(c->row_head, c->row_head_next);
  c->nwall_idx = c->nwall_idx == S_NWALL ? S_NWALL_B : S_NWALL;
  c->parity ^= 1;
}

int ensure_olds(tsph_ctx *c) {
  if (!c->olds_stale) return 0;
  hipLaunchKernelGGL(k_gather_olds, dim3(grid_for(c->n_ub, 256)), dim3(256), 0, c->stream, c->scal,
                     c->perm, c->alt, c->cur);
  TSPH_HIP(hipGetLastError());
  c->olds_stale = false;
  return 0;
}

int launch_cell_list(tsph_ctx *c, bool eos, bool predict, double dt, unsigned ad_skip,
                     bool decide, bool skip_olds, int walls, bool count_density, bool hashed,
                     bool hash_next, bool skip_p) {
  // a build that moves r_o, v_o, rho_o needs them current (the predictor's
  // build rewrites them instead)
  if (!predict && !skip_olds)
    if (int e = ensure_olds(c)) return e;
  const Consts &k = c->k;
  const int nb = 256;
  const int g = grid_for(c->n_ub, nb);
  hipStream_t s = c->stream;
  const int nct = c->ncells_tot;
  // this build's cell offsets and wall count go to the buffers the current
  // cell list does not use (swapped in at the end)
  int *cs = c->cell_start_next;
  const int wslot = c->nwall_idx == S_NWALL ? S_NWALL_B : S_NWALL;
  WallPass wp{};
  int hg = g, hbs = nb;
  if (walls) {
    wp = walls::wall_pass(c, count_density);
    hbs = 64;
    hg = wp.walls + wp.sweep + grid_for(c->n_ub, hbs);
    c->records_valid = false;
  }
  // the per-cell order: ranked by the reorder from rows that the hash leaves (two
  // launches and a hash), or by passes of its own
  const bool rank = cells_ranked(c);
  const CellRows rw{c->row_seq, c->row_head, rank ? c->hrank : nullptr, rank ? c->row_width : 0};
  // (without bins a build's reorder clears the counts it has used)
  const bool binned = c->bin_count != nullptr;
  const Clear clear{{c->cell_count_next, c->bin_count_next, c->row_head_next},
                    {binned ? count_words(c) / 4 : 0, binned ? bin_words(c) / 4 : 0,
                     c->row_width ? kRowHeads / 4 : 0}};
  if (hashed && hash_next) {
    set_error("cell list: a build whose hash was taken takes no next hash");
    return TSPH_ESTATE;
  }
  const CellRows rw_next{c->row_seq_next, c->row_head_next, rank ? c->hrank_next : nullptr,
                         rank ? c->row_width : 0};
#define TSPH_HASH(P, D, W)                                                                     \
  hipLaunchKernelGGL((k_hash<P, D, W>), dim3(hg), dim3(hbs), 0, s, c->cur.r, c->cur.v,         \
                     c->cur.type, c->cur.seq, c->scal, k, c->cases, c->cur.cid, dt, nct,       \
                     c->cell_count, c->hcell, c->hrank, rw, c->bin_count, clear, c->seqstate,  \
                     c->counters, wp)
#define TSPH_HASH_W(P, D)                                                                      \
  if (walls == TSPH_WALL_MDBC) TSPH_HASH(P, D, TSPH_WALL_MDBC);                                \
  else if (walls == TSPH_WALL_BT) TSPH_HASH(P, D, TSPH_WALL_BT);                               \
  else TSPH_HASH(P, D, 0)
  if (hashed) {
    // the build before took it
  } else if (predict && decide) {
    TSPH_HASH_W(true, true);
  } else if (predict) {
    TSPH_HASH_W(true, false);
  } else if (decide) {
    TSPH_HASH_W(false, true);
  } else {
    TSPH_HASH_W(false, false);
  }
#undef TSPH_HASH_W
#undef TSPH_HASH
  // the pooled pair pass that follows (if any) has its chunks cut in the first
  // workgroups of the reorder (or the scatter), from the costs the scan lists
  // beside the tiles and its per-block sums of them
  const int cut = c->cut_groups;
  c->cut_groups = 0;
  if (cut > c->bound_cap) {
    set_error("tile list: more pooled workgroups than allocated");
    return TSPH_ESTATE;
  }
  // two entries for the fuller tiles (the FP64 lists also serve the cell walks,
  // and k_order_tiles takes each tile once)
  const bool split = rank && cut == 0 && c->prm.precision == TSPH_PREC_MIXED && split_pays(c);
  // the cells for the FP64 passes that go by cells
  const bool cells = cut == 0 && c->prm.precision == TSPH_PREC_FP64 && (c->has_ale || cells_walk(c));
  const ScanArgs sa = scan_args(c, cs, cut > 0 ? c->cut_table : -1, split, cells);
  const bool own_scan = !(rank && binned) || cut > 0 || (hashed && walls);
  if (own_scan)
    if (int e = launch_scan(c, sa, hashed ? walls : 0, wp)) return e;
  const int sg = grid_for(c->n_ub, kScatterBlock);
  // one cutting wavefront per scan block, in the first workgroups
  const int cuts = cut > 0 ? grid_for(scan_blocks(c), kScatterBlock / 64) : 0;
  const ChunkCut cc{cuts, scan_blocks(c), cut, c->list_cost, c->scan_cost, c->scan_tile0,
                    c->tile_bound};
  if (cut > 0) {
    c->list_groups = cut;
    c->list_table = c->cut_table;
  }
  if (!rank) {
    hipLaunchKernelGGL(k_scatter, dim3(cuts + sg), dim3(kScatterBlock), 0, s, c->scal, c->hcell,
                       c->hrank, cs, c->perm, c->cellof, nct, c->cur.seq, c->seqstate, cc);
    if (c->cases)
      hipLaunchKernelGGL(k_order, dim3(grid_for(nct + 1, nb)), dim3(nb), 0, s, cs, nct, c->cur.seq,
                         c->perm, c->cell_count);
    else
      hipLaunchKernelGGL(k_order_tiles, dim3(kOrderWaves * std::max(1, c->num_cu)), dim3(nb), 0, s,
                         cs, c->scal, c->tile_list, cells ? 1 : c->tile_rows, k.ncy, nct, c->cur.seq, c->perm,
                         c->cell_count);
  }
  const Mixed mx = c->prm.precision == TSPH_PREC_MIXED ? c->mx : Mixed{};
  const Clear cl = hashed ? clear : Clear{};
  const unsigned moves = (skip_olds ? 0 : kMoveOlds) | (skip_p ? 0 : kMoveP) |
                         (skip_olds ? kMovePerm : 0);
#define TSPH_REORDER(E, P, R, N, S)                                                           \
  hipLaunchKernelGGL((k_reorder<E, P, R, N, S>),                                              \
                     dim3((R ? cuts : 0) + (S ? cc.scan_blocks : 0) + sg), dim3(kScatterBlock),    \
                     S ? sizeof(int) * bin_words(c) : 0, s, cs, nct, c->n_ub, c->hcell, rw,         \
                     c->bin_count, bin_words(c), cl, sa, c->perm, c->cell_count, c->seqstate, cc, c->cur, c->alt,     \
                     c->scal, c->wall_list, c->cellof, k, c->cases, mx, dt, ad_skip, c->counters,   \
                     wslot, c->nwall_idx, moves, c->cell_count_next, c->bin_count_next,        \
                     c->hcell_next, c->hrank_next, rw_next)
#define TSPH_REORDER_R(E, P, N)                                                               \
  if (!rank) TSPH_REORDER(E, P, false, N, false);                                             \
  else if (own_scan) TSPH_REORDER(E, P, true, N, false);                                      \
  else TSPH_REORDER(E, P, true, N, true)
  if (hash_next) {
    TSPH_REORDER_R(true, false, true);
  } else if (eos && predict) {
    TSPH_REORDER_R(true, true, false);
  } else if (eos) {
    TSPH_REORDER_R(true, false, false);
  } else if (predict) {
    TSPH_REORDER_R(false, true, false);
  } else {
    TSPH_REORDER_R(false, false, false);
  }
#undef TSPH_REORDER_R
#undef TSPH_REORDER
  TSPH_HIP(hipGetLastError());
  flip_build(c);
  c->olds_stale = skip_olds && !predict;
  c->olds_in_alt = skip_olds && predict;
  c->cells_valid = true;
  c->tiles_valid = true;  // listed by the scan
  c->records_valid = eos && c->prm.precision == TSPH_PREC_MIXED;
  if (predict || decide) c->marks_valid = false;
  return 0;
}

}  // namespace tsph
