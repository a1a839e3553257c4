// Internal declarations shared by the translation units of libtinysph_hip.so.
// Device data layout (HBM), one SoA generation per field:
//   r, v, a, r_o, v_o, n      : double2   (16 B per particle each)
//   rho, drho, p, rho_o       : double    ( 8 B)
//   type                      : uint8     (reference part_type; 255 = removed)
//   seq                       : uint32    (position in reference order; gaps allowed)
//   gnr, index                : double2, int32 (ghost node, reference data.index), by
//                               reference position: one generation, never moved
// After every Particle_To_Cell the arrays are permuted into (cell, seq) order,
// so a cell's particles are contiguous and ordered exactly as the reference
// iterates them; `cellof[k]` holds the cell of slot k and `cell_start` the CSR
// offsets.  The particle count lives on the device (`scal[S_NP]`) so that a
// whole step can be captured in a HIP graph; the host keeps an upper bound.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../../include/tinysph.h"

namespace tsph {

constexpr uint8_t kRemoved = 255;

constexpr int kMaxTileRows = 24;  // upper bound of tile_rows
// Pooled walk's cost model.  Every pooled pass records the time each tile took
// its wavefront (tq_mark, tsph_tiles.h; 10 ns ticks of the device's constant
// clock, averaged with the tile's previous record) in one of kCostTables
// tables, at scal[S_NSCAL + kCostTables t + table] for global tile t; the
// next pooled pass of the same table cuts its chunks by these costs
// (cut_chunks_scan in a cell-list build, cut_chunks_block for a list reused
// without one).  A recorded time carries what a model of the tile's
// work would not: what else ran on its compute unit, so that the chunks of a
// compute unit that ran slow shrink in the next pass.  Table 1 holds the mixed
// pair passes that apply the symplectic corrector as well, table 0 every
// other pooled pass.  A tile without a record (the first pass after a change of
// tile layout, or a tile newly occupied) is estimated from its own particles:
// own particles x own + tile, the least-squares fit of the measured times of
// the 740k-particle dam break's 13,147 tiles (near-empty tiles 4.4 us mixed,
// 3.3 us FP64; full 14.2 us and 32 us).
struct CostEstimate {
  int own, tile;
};
constexpr CostEstimate kCostMixed{19, 425}, kCostFp64{54, 300};
constexpr int kCostTables = 2;
inline CostEstimate cost_estimate(bool mixed) { return mixed ? kCostMixed : kCostFp64; }

// device scalar slots
// (the wall count alternates between S_NWALL and S_NWALL_B with the cell-offset
// buffers: a build fills the other one, see cell_start_next); the per-tile
// costs follow them (kCostTables (ncells_tot + 8) slots)
enum { S_NP = 0, S_MAXSEQ = 1, S_NTILES = 2, S_NWALL = 3, S_BZCNT = 4, S_NWALL_B = 5,
       S_DLNP = 6, S_NEWSEQ = 7, S_NSCAL = 32 };
// device counter slots (uint64)
enum {
  C_PAIRS = 0, C_CAND = 1, C_ACTIVE = 2, C_PASSES = 3, C_BADRHO = 4, C_OUTGRID = 5,
  C_REMOVED = 6, C_APPENDED = 7, C_BZREJECT = 8, C_BZCHAIN = 9, C_REINIT = 10, C_SCANSTALL = 11,
  C_NCOUNT = 12
};
// The pair loops' counts (pairs, candidates, active) go to per-wavefront
// slots after the counters above, 4 words per wavefront, and are summed when
// read: one device-wide atomic per wavefront on three shared words, all at the
// end of a launch, serialises there and delays the launch's last tiles.
constexpr int kWaveCtr0 = 16;


// buffer zone (BufferZone, src/SPH_inlet_outlet_data.h:18-46)
struct Zone {
  double x0, xm, y0, ym, bl, bh, vx, vy;
  int ox, oy, btype;
};
constexpr int kBzMax = 4096;  // zone particles an inlet pass may convert

struct Soa {
  uint8_t *cid = nullptr;  // case of each particle (batched ensembles only)
  double2 *r = nullptr, *v = nullptr, *a = nullptr, *r_o = nullptr, *v_o = nullptr;
  // by reference position (seq), as is index: nothing changes them, so the
  // builds need not move them; cur's and alt's are the same arrays
  double2 *gnr = nullptr;
  double2 *n = nullptr;
  double *rho = nullptr, *drho = nullptr, *p = nullptr, *rho_o = nullptr;
  uint8_t *type = nullptr;
  uint32_t *seq = nullptr;
  int32_t *index = nullptr;
  // ALE-SPH volume variables (allocated for ALE runs only)
  double *omega = nullptr, *omegarho = nullptr, *omega_o = nullptr, *omegarho_o = nullptr;
  double *domega = nullptr, *domegarho = nullptr;
  double2 *omegav = nullptr, *omegav_o = nullptr, *domegav = nullptr;
  // ALE-SPH MUSCL gradients of rho, vx, vy (allocated with the volume variables)
  double2 *gradrho = nullptr, *gradvx = nullptr, *gradvy = nullptr;
  // Verlet second time layer and the density-reinitialisation buffer (rhoTemp)
  // (allocated by tsph_history_enable)
  double2 *v_oo = nullptr;
  double *rho_oo = nullptr, *rho_tmp = nullptr;
  // Kahan compensation terms of the symplectic corrector's position and
  // density updates (allocated by tsph_set_compensated)
  double2 *rc = nullptr;
  double *rhoc = nullptr;
  // where particle i's r_o, v_o, rho_o are (nullptr: at i), for the corrector
  const int *old_at = nullptr;
};

// FP32 pair records of the mixed path, rebuilt after every reorder.
struct Mixed {
  float4 *rv = nullptr;   // {x - cell origin x, y - cell origin y, vx, vy}
  float2 *rp = nullptr;   // {rho - rho0, p}
  float2 *nrm = nullptr;  // BT wall normal
};

// constants of the physics, precomputed on the host exactly as the reference does
struct Consts {
  double h, kap, cs, rho0, avisc, delta, dp, m, gx, gy;
  double x0, xm, y0, ym;
  double kh, of;
  double awen, bwen;  // float-rounded Wendland constants, src/SPH_kernel.h:56-57
  double ih, cb, icb; // 1/h, cs^2 rho0 / 7, 1/cb
  // the largest r^2 whose rounded sqrt(r^2) / h is at most 2: r^2 <= r2max is the
  // reference's qq <= 2 without its root and division (both are monotonic)
  double r2max;
  int ncx, ncy, ncells;
  // batched ensembles: the case's first global cell id and its time step
  // (single cases: 0 and unused)
  int cell_base;
  double dt;
};

// constants of particle i: its case's entry of the batch table, or k0
__device__ __forceinline__ Consts case_consts(const Consts &k0, const Consts *__restrict__ cases,
                                              const uint8_t *__restrict__ cid, int i) {
  return cases ? cases[cid[i]] : k0;
}

// host-side flags that describe what the device buffers hold
struct HostState {
  bool cells_valid, tiles_valid, records_valid, marks_valid, olds_stale, list_split;
  int list_groups, list_table, list_cost_table, list_rows;
};

// one captured step.  A step may rebuild the cell list an odd number of times
// (the Riemann-ALE step does it once), which swaps the cur/alt particle buffers:
// graphs are therefore kept per buffer parity, and a replay applies the swap
// and the host flags that the captured step left behind.
struct Graph {
  hipGraphExec_t exec = nullptr;
  int wall = -1;
  double dt = 0;
  int n_ub = -1;
  bool flips = false;  // the step swaps cur and alt an odd number of times
  HostState post{};    // host flags after the step
  int steps = 1;       // steps captured in the graph
};
// steps captured in one graph of a run of whole symplectic steps: each graph
// launch costs about 8 us of idle time between the steps it separates
constexpr int kGraphSteps = 8;

}  // namespace tsph

struct tsph_ctx {
  tsph_params prm;
  tsph::Consts k;
  int capacity = 0;
  int n_ub = 0;  // host upper bound of the device particle count
  int ncells_tot = 0;            // cells of all cases (the single case: k.ncells)
  double cell_lattice = 0.;      // particles that a lattice of spacing dp puts in a cell (the most of the cases)
  // batched ensembles: per-case constants on the device (nullptr for one case)
  int ncases = 1;
  tsph::Consts *cases = nullptr;
  std::vector<tsph::Consts> host_cases;
  int *tile_base = nullptr;      // ncases+1 first global tile id per case (current tile_rows)
  std::vector<int> host_tile_base;  // host copy of tile_base
  std::vector<int> seq_base;     // first reference position per case (ncases+1)
  std::vector<int> case_cap;     // particle slots reserved per case
  bool has_gnr = false, has_n = false;
  bool cells_valid = false;
  int tile_rows = 16;  // cells per pair-loop tile (one grid-column run)
  bool rows_set = false;  // by tsph_set_tile_rows
  int waves_per_cu = 8;  // persistent pair-loop waves per compute unit
  int num_cu = 256;      // compute units of the device
  int max_lds_block = 65536;  // LDS bytes a workgroup may allocate
  int lds_cu = 163840;        // LDS bytes of one compute unit
  // workgroups per compute unit of the cell walks, by kernel (0: not asked yet)
  int cells_fit[3] = {}, ale_fit[8] = {};
  // pair-loop tile walk per precision (FP64, mixed): pooled (work-balanced
  // chunks per workgroup, tiles taken from an LDS counter by the workgroup's
  // waves) or the plain static walk; defaults set at creation
  bool balanced[2] = {false, false};
  int cell_order = 0;  // tsph_set_cell_order: 0 and 1 ranked, 2 separate passes
  // the entries of the pair walks: non-empty tiles of the current cell list, in
  // tile order (tiles::part of each), or non-empty cells (list_rows kListCells)
  int *tile_list = nullptr;
  bool list_split = false;  // tiles of more than a wavefront of particles have two entries
  int list_rows = 0;        // cells per listed tile (kListCells: the list is one of cells)
  bool tiles_valid = false;  // tile_list is of the current cell list, list_rows deep
  int *list_part = nullptr;  // per list-build block: tiles, work
  int list_part_cap = 0;     // list-build blocks list_part holds
  int *tile_bound = nullptr; // pooled walk: first list entry of each workgroup's chunk
  int wave_ctr_cap = 0;      // wavefronts with count slots in `counters`
  int bound_cap = 0;         // chunks tile_bound holds
  int list_groups = 0;       // chunks the current tile_bound was cut for (0: none or stale)
  int list_table = 0;        // the cost table they were cut by
  int *list_cost = nullptr;  // costs of the listed tiles by list position (pooled cuts)
  int list_cost_table = -1;  // the cost table list_cost was gathered from (-1: none)
  // a pooled pair pass of `cut_groups` workgroups and cost table `cut_table`
  // follows the next cell build (0: none): the build cuts its chunks
  int cut_groups = 0, cut_table = 0;
  int last_variant = TSPH_FORCES_WCSPH;  // of the last pair pass
  // {slot, reference position} of the wall particles of the current cell list
  int2 *wall_list = nullptr;
  int n_wall = 0;            // wall particles (walls are never created or removed)
  bool records_valid = false;  // mixed-path FP32 records match the FP64 state
  bool marks_valid = false;    // removal marks match the current positions
  // r_o, v_o, rho_o were not moved by the last cell build (the build that
  // follows a symplectic corrector: the next predictor rewrites them); until
  // rebuilt they are alt's values through perm (ensure_olds)
  bool olds_stale = false;
  // device address of the allocation-free interpolation grid's static scratch
  // array on this context's device (looked up at creation)
  double *grid_scratch = nullptr;
  bool has_ale = false;        // ALE volume variables allocated
  uint8_t *ale_flag = nullptr; // per particle: its own ALE gamma sum is non-zero
  hipStream_t stream = nullptr;
  tsph::Soa cur, alt;
  // gnr and index in upload or download order, on their way
  double2 *pos_gnr = nullptr;
  int32_t *pos_index = nullptr;
  tsph::Mixed mx;
  unsigned char *arena = nullptr;      // holds scal and the cell-list buffers below
  int *scal = nullptr;                 // S_* slots, then the per-tile costs
  unsigned long long *counters = nullptr;
  int *cell_count = nullptr;           // ncells+1 (last = removed bucket)
  int *cell_count_next = nullptr;      // the next build's
  // sums of kBinCells counts (nullptr: too many cells)
  int *bin_count = nullptr, *bin_count_next = nullptr;
  int *cell_start = nullptr;           // ncells+2
  // Every build writes its cell offsets and wall count into the buffers the
  // previous build did not (cell_start_next, the other wall-count slot) and
  // then swaps, so that the wall-density pass that reads the previous cell
  // list can run while the next build sorts (record_step).
  int *cell_start_next = nullptr;      // ncells+2
  int nwall_idx = 3;                   // S_NWALL or S_NWALL_B: the current wall count
  int *cellof = nullptr;               // cell of each slot (sorted order)
  int *hrank = nullptr;                // rank inside the cell from the hash pass, or row links
  int *hcell = nullptr;                // cell from the hash pass (pre-sort order)
  int *perm = nullptr;                 // sorted position -> old slot
  // the seqs of each cell's particles as the hash leaves them for the reorder
  // to rank (row_width per cell, fuller cells chained from row_head; 0: the
  // builds order the cells in passes of their own)
  int row_width = 0;
  uint32_t *row_seq = nullptr;
  int *row_head = nullptr;
  // the next build's (flip_build swaps them in), so that a build's reorder can
  // take the hash of the build after it
  int *hcell_next = nullptr, *hrank_next = nullptr;
  uint32_t *row_seq_next = nullptr;
  int *row_head_next = nullptr;
  // cell-list scan: one published word per block (zero: not yet published),
  // and the polls a block makes for an earlier block's word (-1: none)
  unsigned long long *scan_state = nullptr, *scan_state_next = nullptr;
  // per scan block: the listed tiles' summed cost and first list position
  int *scan_cost = nullptr, *scan_tile0 = nullptr;
  int scan_wait = 1 << 20;
  uint8_t *seqstate = nullptr;         // removal: per-seq state
  double *probe_out = nullptr;         // tsph::kProbeOut doubles for probe results
  // pair-kernel timing: one event pair per pair launch while enabled
  bool time_pairs = false;
  std::vector<hipEvent_t> tev;         // 2 per recorded launch
  int tev_used = 0;
  float last_pair_ms = 0.f;
  bool olds_in_alt = false;   // the old state is alt's r, v, rho, through perm
  int parity = 0;             // flips whenever cur and alt are swapped
  // the steps' graphs, by parity at the step's start: one step ([0], [1]) or a
  // run of kGraphSteps ([2], [3]; each graph launch leaves some us idle before
  // the next: Riemann-ALE steps of 47k particles 68.6 us one by one, 64.8 in
  // runs, ALE ones of 183k 240 and 236, of 12k 109 and 105; 1M particles with
  // buffer zones 447 and 446, so those stay single)
  tsph::Graph graph[4];       // symplectic
  tsph::Graph rale_graph[4];  // Riemann-ALE
  tsph::Graph ale_graph[4];   // ALE-SPH MUSCL
  tsph::Graph lf_graph[4];    // leap-frog driver (after the first step)
  tsph::Graph inflow_graph[2];  // symplectic with buffer zones
  tsph::Graph verlet_graph[2];  // Verlet driver (Verlet integrator)
  tsph::Graph euler_graph[2];   // Verlet driver on its Euler steps
  // the step being recorded of the run that one graph holds
  int rec_step = 0, rec_steps = 1;
  bool has_history = false;     // v_oo, rho_oo, rhoTemp allocated
  // asynchronous output (tsph_write_vtk): writer threads and their first error
  std::vector<std::thread> writers;
  std::mutex io_mu;
  std::string io_error;
  tsph::Zone zones[TSPH_MAX_ZONES];
  int n_zones = 0;
  int *bz_list = nullptr;     // 2 * kBzMax ints: {seq, slot} of the crossing zone particles
  int seq_cap = 0;            // size of seqstate (reference positions ever handed out)
  int seq_ub = 0;             // host upper bound of scal[S_MAXSEQ]
};

namespace tsph {

void set_error(const std::string &msg);
int hip_fail(hipError_t e, const char *what, const char *file, int line);

#define TSPH_HIP(call)                                                  \
  do {                                                                  \
    hipError_t e_ = (call);                                             \
    if (e_ != hipSuccess) return tsph::hip_fail(e_, #call, __FILE__, __LINE__); \
  } while (0)

inline int grid_for(int n, int block) { return n <= 0 ? 1 : (n + block - 1) / block; }

// words of the counters buffer: the counters, then the per-wavefront slots
inline size_t counter_words(const tsph_ctx *c) { return kWaveCtr0 + 4 * (size_t)c->wave_ctr_cap; }

// pair-loop tiles of the cell grid(s) at the current tile_rows
inline int total_tiles(const tsph_ctx *c) {
  if (!c->cases) return c->k.ncx * ((c->k.ncy + c->tile_rows - 1) / c->tile_rows);
  return c->host_tile_base[c->ncases];
}

// whether a pair launch of `waves` persistent waves takes the pooled walk:
// the precision's setting, for systems that give each wave enough particles to
// balance.  Dam breaks, us per step pooled and static, on the first 400 steps
// and after 1500: mixed (3072 waves) 210k particles 130 and 124, 143 and 126,
// 260k 137 and 130, 151 and 131, 333k 149 and 168, 161 and 174; FP64 (2048
// waves; static with 6 rows) 233k 227 and 222, 266 and 225, 333k 294 and 291,
// 298 and 312, 517k 390 and 427, 392 and 428; 16 tanks of 879k particles in
// all, mixed, 354 and 432.
constexpr int kPoolMixed = 95, kPoolFp64 = 150;  // particles per wave
// Rows of a tile unless tsph_set_tile_rows chose them: 7, about a wavefront of
// particles, or 6 in FP64 systems too small for the pooled walk.  There, with
// about a tile per resident wavefront, the tiles of more than 64 particles set
// the pass's time by their second round (after 1500 steps: 92k particles 187
// us per step with 7 rows and 135 with 6, 233k 292 and 225; at the start both
// alike), and FP64 results do not depend on the rows.  The mixed path, whose
// bits do (it rounds in the tile's frame), gives such tiles two list entries
// instead.  Pooled FP64 passes hold fewer waves with 6 rows (740k: 520 and 862).
constexpr int kTileRows = 7, kTileRowsFp64 = 6;
inline bool walk_balanced(const tsph_ctx *c, bool fp32, int waves) {
  return c->balanced[fp32 ? 1 : 0] && c->n_ub >= (long long)(fp32 ? kPoolMixed : kPoolFp64) * waves;
}
// Whether a mixed system's tile list gives the fuller tiles two entries
// (tiles::entry_part): where a wave has about a tile, that is up to the pooled
// walk's limit.  Above it for the ALE passes alone, which always stride, and only
// where a tile of the lattice is no fuller than a wavefront: if all tiles had two
// entries, the waves, which stride by an even number, would meet only first or
// only second ones.  us per step, one entry and two: ALE of 324k particles after
// 1500 steps 431 and 377, of 727k 808 and 800; of 727k with 74 particles per tile
// 1619 and 2160, Riemann-ALE 560 and 620.  (A pooled pass would list anew: 293k
// particles stage by stage 85 and 91.)
inline bool split_pays(const tsph_ctx *c) {
  if (c->n_ub < (long long)kPoolMixed * c->num_cu * c->waves_per_cu) return true;
  return c->has_ale && c->tile_rows * c->cell_lattice <= 64.;
}

// launch geometry of a tile kernel: `groups` workgroups (a multiple of 8) of
// block.x / 64 wavefronts, each wavefront with lds_wave bytes of LDS
struct TileGrid {
  dim3 grid, block;
  size_t lds = 0;    // dynamic LDS per workgroup
  int lds_wave = 0;
  int groups = 0;
  bool pooled = false;
};

// doubles of probe results (tsph_stages.hip: {level, index} of 32 chunks, a height)
constexpr int kProbeOut = 65;
// tsph_cells.hip
// heads of the chains that hold what the cells' rows do not (a power of two)
constexpr int kRowHeads = 4096;
// cells per bin, bins per round of a workgroup's scan of them, and the most
// bins: with the scan in the reorder's launch a step of the dam break takes
// 75.5 us instead of 80.2 on 44k cells (50k particles, FP32 pairs), 124.4
// instead of 125.0 on 84k (92k particles, FP64) and 244 instead of 241 on 177k
// (183k ALE particles); still water on 0.7k cells 50.0 instead of 59.6
constexpr int kBinCells = 16, kBinChunk = 1024, kBinMax = 4096;
// allocated words: whole bins of counts, whole rounds of bins
inline int count_words(const tsph_ctx *c) {
  return (c->ncells_tot + 1 + kBinCells - 1) / kBinCells * kBinCells;
}
inline int bin_words(const tsph_ctx *c) {
  return (count_words(c) / kBinCells + kBinChunk - 1) / kBinChunk * kBinChunk;
}
// the buffers that change places with every cell build: cur and alt, and this
// build's cell-list buffers and the next one's
void flip_build(tsph_ctx *c);
// hash, scan, reorder; eos: the reorder also runs
// Density_to_pressure (and writes the mixed records) for the moved particles
// predict: the symplectic predictor (step dt; per case in a batch) is applied
// on the way, in place of a launch_predictor immediately before.  ad_skip: a
// mask of particle types (bit t: type t) whose a, drho are left behind, for a
// build that a pair pass overwriting exactly those follows (forces_active_types)
// decide: RemoveParticlesOutOfDomain's decision is taken by the build, in
// place of a launch_remove immediately before (the removal states must be
// current: a corrector precedes)
// skip_olds: r_o, v_o, rho_o are not moved (olds_stale afterwards), for a build
// after which they are dead until the next predictor rewrites them; with
// predict they are not written: a corrector that follows takes them from the
// previous generation (old_state), and they are dead after it
// skip_p: pressures are not written where an EOS will rewrite them before
// anything reads them (the mixed path's pair passes read its records)
// walls (TSPH_WALL_MDBC or TSPH_WALL_BT; 0: none): the wall densities of that
// treatment are computed first, from the previous cell list, in the same
// launch as the build's hash, or as its scan where it has none (as launch_mdbc
// / launch_bt_density with count_density)
// hash_next (with eos, without predict): the build's reorder also takes the
// hash of the predict build that follows it with nothing but a pair pass
// between them (the next step's first, with time step dt); hashed: that build
int launch_cell_list(tsph_ctx *c, bool eos = false, bool predict = false, double dt = 0.,
                     unsigned ad_skip = 0, bool decide = false, bool skip_olds = false,
                     int walls = 0, bool count_density = false, bool hashed = false,
                     bool hash_next = false, bool skip_p = false);
// r_o, v_o, rho_o of the current generation, gathered from the previous one
// through the last build's permutation if that build left them behind; every
// launch that reads or moves them calls this first
int ensure_olds(tsph_ctx *c);
// cur, with the old state where the last build left it
inline Soa old_state(const tsph_ctx *c) {
  Soa d = c->cur;
  if (c->olds_in_alt) {
    d.r_o = c->alt.r;
    d.v_o = c->alt.v;
    d.rho_o = c->alt.rho;
    d.old_at = c->perm;
  }
  return d;
}
// types whose a, drho a pair pass of `variant` writes (its active particles)
inline unsigned forces_active_types(int variant) {
  return variant == TSPH_FORCES_DBC ? (1u << TSPH_FLUID) | (1u << TSPH_WALL) : 1u << TSPH_FLUID;
}
// tsph_pairs.hip
// list of the non-empty pair-loop tiles; groups > 0: also its chunk bounds
// for a pooled walk of that many workgroups, cut by the tile costs recorded
// in cost table `table`
int ensure_tile_list(tsph_ctx *c, int groups, int table = 0);
// list of the non-empty cells, for a cell walk
int ensure_cell_entries(tsph_ctx *c);
// geometry of a tile-kernel launch at the context's waves per CU (pooled when
// may_pool and walk_balanced hold for the precision)
TileGrid tile_grid(tsph_ctx *c, bool fp32, size_t lds_wave, bool may_pool = true);
// clears the per-tile costs (the tile layout changed)
int clear_tile_costs(tsph_ctx *c);
// cuts the current tile list into `groups` chunks by cost table `table` on
// stream s (gathering the listed tiles' costs first unless the list build did)
int launch_cut(tsph_ctx *c, hipStream_t s, int groups, int table);
// whether the pair pass goes by cells instead of tiles
bool cells_walk(const tsph_ctx *c);
// entries of the tile list's buffer
inline size_t tile_list_room(const tsph_ctx *c) { return 2 * ((size_t)c->ncells_tot + 8); }
// list_rows of a list of non-empty cells (global ids): what the cell walks go
// through, listed like tiles of one cell of a grid with a single column
constexpr int kListCells = 0;
// workgroups of a pair pass of `variant` if it takes the pooled walk, else 0
int pass_groups(tsph_ctx *c, int variant);
// corr (mixed path only): the pass also applies the symplectic corrector to
// every particle, with time step corr_dt (batched contexts: each case's own)
// walls (mixed path, static walk, not with corr): the wall densities that the
// next step begins with are computed beside the pass
int launch_forces(tsph_ctx *c, int variant, bool corr = false, double corr_dt = 0.,
                  bool walls = false);
int launch_mixed_records(tsph_ctx *c);
// tsph_stages.hip
int launch_eos(tsph_ctx *c);
int launch_predictor(tsph_ctx *c, double dt);
int launch_corrector(tsph_ctx *c, double dt);
// count_density: also take the out-of-range density count of an EOS pass
// right after (in place of that pass, where nothing reads its pressures)
int launch_mdbc(tsph_ctx *c, bool count_density = false);
int launch_bt_density(tsph_ctx *c, bool count_density = false);
int launch_remove(tsph_ctx *c);
int run_water_elevation(tsph_ctx *c, double x, double y0, int inverse, double *out);
// soa: out holds rho[n], p[n], then v[2n] (n = ncx ncy); else 4 values per point
int launch_interp_grid(tsph_ctx *c, double x0, double y0, double dh, int ncx, int ncy, double *out,
                       bool soa = false);
// The live particles of one case (icase; -1: all) gathered from cur into the
// same fields of alt, in reference order, for a download; alt holds nothing
// between builds once the olds are in place (ensure_olds first).  fields: a
// mask of DL_*.  Leaves the particle count in scal[S_DLNP].
enum {
  DL_R = 1, DL_V = 2, DL_A = 4, DL_R_O = 8, DL_V_O = 16, DL_GNR = 32, DL_N = 64, DL_P = 128,
  DL_RHO = 256, DL_DRHO = 512, DL_RHO_O = 1024, DL_TYPE = 2048, DL_INDEX = 4096
};
int launch_download_gather(tsph_ctx *c, int icase, unsigned fields);
// The live particles' reference positions relabelled 0..m-1 in order, the removed
// slots' m..; the removal states, gnr, index and the wall list's positions move
// along, S_MAXSEQ follows (alt's seq and type, pos_gnr and pos_index are scratch).
int launch_renumber(tsph_ctx *c);
// p[i] = i for i < n
int launch_iota(tsph_ctx *c, int *p, int n);
// gnr (if gnr) and index of n uploaded particles from pos_gnr, pos_index to their
// reference positions (cur.seq)
int launch_place(tsph_ctx *c, int n, bool gnr);
// live particles of every case of a batch into counts[ncases] (device memory)
int launch_case_counts(tsph_ctx *c, int *counts);
// words of the bitmap over reference positions that launch_download_gather
// keeps in hcell (and its prefix in hrank)
inline size_t dl_words(int seq_cap) { return ((size_t)seq_cap + 31) / 32; }
// device address of the allocation-free interpolation grid's scratch on the
// current device (looked up once per device)
int grid_scratch_ptr(double **out);
// tsph_ale.hip
int launch_ale_init(tsph_ctx *c);
int launch_rale_forces(tsph_ctx *c);
int launch_rale_leapfrog_one(tsph_ctx *c, double dt);
int launch_rale_leapfrog_two(tsph_ctx *c, double dt, int step);
int run_interpolate_point(tsph_ctx *c, double x, double y, double *out4);
// tsph_alemuscl.hip (muscl: 0 first order, 1 alpha = 1, 2 minmod-limited)
int launch_ale_density(tsph_ctx *c, int muscl);
int launch_ale_acceleration(tsph_ctx *c, int muscl);
int launch_ale_gradient(tsph_ctx *c);
int launch_ale_density_pressure(tsph_ctx *c, double dt);
int launch_ale_leapfrog_one(tsph_ctx *c, double dt);
// tsph_integrators.hip
int launch_history_init(tsph_ctx *c);
int launch_verlet(tsph_ctx *c, double dt, bool euler);
int launch_leapfrog_one(tsph_ctx *c, double dt);
int launch_leapfrog_two(tsph_ctx *c, double dt, int step);
int launch_reinit_sum(tsph_ctx *c);
int launch_reinit_overwrite(tsph_ctx *c);
int launch_ale_leapfrog_two(tsph_ctx *c, double dt, int step);
// tsph_zones.hip
int launch_bz_inlet(tsph_ctx *c, int zone, double dt);
int launch_bz_outlet(tsph_ctx *c, int zone, double dt);

}  // namespace tsph
