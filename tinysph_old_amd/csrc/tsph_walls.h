// Wall densities (mDBC, BT) by wavefronts, shared by their own launches
// (tsph_stages.hip), the first cell build of a symplectic step, whose hash or
// scan launch runs them in wavefronts of its own (tsph_cells.hip), and static
// mixed pair passes (tsph_pairs.hip):
//   mDBC_compute_density_mdbcGeo   src/SPH_mDBC.h:9-50 with
//                                  Kernel_density_approximation_MATRIX_mDBC,
//                                  src/SPH_kernel_approx.h:1141-1342
//   BT_compute_density_BTGeo       src/SPH_BT.h:9-50 with
//                                  Kernel_density_approximation_BT_update,
//                                  src/SPH_kernel_approx.h:1838-1953
#pragma once

#include "tsph_internal.h"
#include "tsph_physics.h"

namespace tsph {
namespace walls {

// cell of a sampling point, computed like Particle_To_Cell
__device__ __forceinline__ int point_cell(const Consts &k, double x, double y) {
  return cell_coord(y, k.y0, k.of, k.kh) + cell_coord(x, k.x0, k.of, k.kh) * k.ncy;
}

// Wall densities: kWG lanes per wall particle.  The 9 stencil cells (cells
// outside the grid skipped) form one candidate sequence in the reference order
// (stencil order, ascending index within a cell); lane u of the group takes
// candidates u, u + kWG, u + 2 kWG, ...  The records of kWPre such rounds are
// loaded together (all in flight at once).  The fluid neighbours among them (a
// sixth to a third) are held in LDS in candidate order, and whenever there are
// kWG of them the group's lanes evaluate their terms at once, put them in
// LDS, and lane u adds sums q = u, u + kWG, ... over them in order, so every
// sum is formed in the reference order.  A candidate that is not a fluid
// neighbour within the support adds nothing, as in the reference.
// The pass is bound by its loads (scattered over nine cells for each group) and
// by FP64 issue: the cells' bounds by one load and broadcasts, rounds over the
// neighbours instead of all candidates (two instead of five) and shared
// reciprocals took it beside the scan, us, from 42 to 34 for the 57k walls of a
// 16-tank ensemble, 22 to 19.5 for 20k and 10.7 to 9 for 5k.
constexpr int kWG = 16;
constexpr int kWPre = 3;
constexpr int kWHeld = 2 * kWG;  // neighbours a group can hold
constexpr int kWallsPerWave = 64 / kWG;
constexpr int kTerms = 64 * 12;  // doubles of LDS of a wavefront of the pass

template <int NS, typename Term>
__device__ __forceinline__ void wall_sums(const Soa &d, const int *__restrict__ cell_start,
                                          const Consts &k, double2 ar, bool live,
                                          double (&acc)[NS], double *__restrict__ terms,
                                          Term term) {
  constexpr int QPL = (NS + kWG - 1) / kWG;  // sums per lane
  const int u = threadIdx.x & (kWG - 1);
  const int g0 = threadIdx.x & 63 & ~(kWG - 1);  // the group's first lane
  // the group's LDS: held neighbours' {dx, dy, rho}, or a round's kWG x NS terms
  constexpr int kArea = kWG * NS > kWHeld * 3 ? kWG * NS : kWHeld * 3;
  static_assert(kArea * kWallsPerWave <= kTerms, "");
  double *grp = terms + g0 / kWG * kArea;
  const double r2cut = 4.0 * k.h * k.h * (1.0 + 1e-12);
  // candidate f lies in the last cell s with pre[s] <= f, at index f + dj[s]
  int pre[9], dj[9], tot = 0;
#pragma unroll
  for (int s = 0; s < 9; ++s) {
    pre[s] = 0;
    dj[s] = 0;
  }
  // The 12 offsets that bound the cells, one load by the group's first 12 lanes
  // (4 for each of the 3 columns; outside the grid the nearest end, so that the
  // cell is empty) and broadcast: 18 loads by every lane took a fourth of the
  // pass.
  static_assert(kWG == 16, "a group is a DPP row");
  int edge = 0;
  if (live && u < 12) {
    const int c = point_cell(k, ar.x, ar.y) + (u / 4 - 1) * k.ncy + u % 4 - 1;
    edge = cell_start[min(max(c, 0), k.ncells)];
  }
  int at[12];  // (lanes of groups that are not live: all 0)
#define TSPH_EDGE(E) at[E] = __builtin_amdgcn_mov_dpp(edge, 0x150 + E, 0xf, 0xf, false);  // row_newbcast
  TSPH_EDGE(0) TSPH_EDGE(1) TSPH_EDGE(2) TSPH_EDGE(3) TSPH_EDGE(4) TSPH_EDGE(5)
  TSPH_EDGE(6) TSPH_EDGE(7) TSPH_EDGE(8) TSPH_EDGE(9) TSPH_EDGE(10) TSPH_EDGE(11)
#undef TSPH_EDGE
#pragma unroll
  for (int s = 0; s < 9; ++s) {
    int dx, dy;
    stencil_dxy(s, dx, dy);
    const int e = (dx + 1) * 4 + dy + 1;
    pre[s] = tot;
    dj[s] = at[e] - tot;
    tot += at[e + 1] - at[e];
  }
  double mine[QPL];  // sums u + kWG x
#pragma unroll
  for (int x = 0; x < QPL; ++x) mine[x] = 0.;
  int held = 0;
  // the terms of the first n (up to kWG) held neighbours into the sums
  auto round = [&](int n) {
    bool ok = false;
    double drx = 0., dry = 0., nrho = 1., lx = 0., ly = 0., lr = 0.;
    if (u < n) {
      drx = grp[3 * u];
      dry = grp[3 * u + 1];
      nrho = grp[3 * u + 2];
    }
    const bool left = kWG + u < held;  // kept for the next round
    if (left) {
      lx = grp[3 * (kWG + u)];
      ly = grp[3 * (kWG + u) + 1];
      lr = grp[3 * (kWG + u) + 2];
    }
    const Root64 rt = sqrt64(drx * drx + dry * dry);
    const double qq = quot64(rt.s, k.h, k.ih);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // the candidate's terms, straight into the group's LDS slots (the
    // reference adds each to a running sum that starts at +0, which
    // never turns -0, so the term x itself stands for 0 + x)
    ok = u < n && qq <= 2.0;
    if (ok) term(nrho, drx, dry, wendland64(rt, qq, k.awen, k.bwen), grp + u * NS);
    const unsigned gm = (unsigned)(__ballot(ok) >> g0) & ((1u << kWG) - 1u);
    // LDS accesses of one wavefront complete in issue order; the fences keep
    // the compiler from moving them across the hand-over
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // the round's terms of sum q = u + kWG x, read for all kWG candidates at
    // once (the LDS reads in flight together), then added in candidate
    // order; a candidate that is not a neighbour adds +0, which leaves the
    // sum unchanged (a sum that starts at +0 and adds terms is never -0).
    // Lanes past the last sum read sum NS - 1 and discard it.
#pragma unroll
    for (int x = 0; x < QPL; ++x) {
      const int q = min(u + kWG * x, NS - 1);
#pragma unroll
      for (int h = 0; h < kWG; h += kWG / 2) {
        double tv[kWG / 2];
#pragma unroll
        for (int w = 0; w < kWG / 2; ++w) tv[w] = grp[(h + w) * NS + q];
#pragma unroll
        for (int w = 0; w < kWG / 2; ++w) mine[x] += ((gm >> (h + w)) & 1u) ? tv[w] : 0.;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (left) {
      grp[3 * u] = lx;
      grp[3 * u + 1] = ly;
      grp[3 * u + 2] = lr;
    }
    held -= n;
  };
  for (int base = 0; base < tot; base += kWG * kWPre) {  // uniform within the group
    int tt[kWPre];
    double2 rr[kWPre];
    double hh[kWPre];
#pragma unroll
    for (int v = 0; v < kWPre; ++v) {
      const int f = base + v * kWG + u;
      int j = f + dj[0];
#pragma unroll
      for (int s = 1; s < 9; ++s) j = f >= pre[s] ? f + dj[s] : j;
      tt[v] = -1;
      rr[v] = make_double2(0., 0.);
      hh[v] = 1.;
      if (f < tot) {
        tt[v] = d.type[j];
        rr[v] = d.r[j];
        hh[v] = d.rho[j];
      }
    }
#pragma unroll
    for (int v = 0; v < kWPre; ++v) {
      if (base + v * kWG >= tot) break;
      const double drx = ar.x - rr[v].x, dry = ar.y - rr[v].y;
      const bool near = tt[v] == TSPH_FLUID && drx * drx + dry * dry <= r2cut;
      const unsigned gm = (unsigned)(__ballot(near) >> g0) & ((1u << kWG) - 1u);
      if (near) {
        double *e = grp + 3 * (held + __popc(gm & ((1u << u) - 1u)));
        e[0] = drx;
        e[1] = dry;
        e[2] = hh[v];
      }
      held += __popc(gm);
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (held >= kWG) round(kWG);
    }
  }
  if (held > 0) round(held);  // (fewer than kWG)
  // every lane of the group gets all NS sums
#pragma unroll
  for (int x = 0; x < QPL; ++x)
    if (u + kWG * x < NS) grp[u + kWG * x] = mine[x];
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int q = 0; q < NS; ++q) acc[q] = grp[q];
}

// The out-of-range density count of the EOS pass that follows the wall
// densities in the symplectic step (k_eos's count; the pass itself is not
// needed there): the wall densities just computed are counted by the lanes
// that computed them (count_walls), every other particle by a sweep that
// runs in workgroups of its own at the end of the same launch, beside the
// wall workgroups rather than after them.  A sweep thread loads kSweep
// particles at a time, type and density together.
constexpr int kSweep = 4;

__device__ __forceinline__ void count_walls(bool wall_bad, unsigned long long *__restrict__ counters) {
  const unsigned long long w = __ballot(wall_bad);
  if (w && (threadIdx.x & 63) == 0) atomicAdd(&counters[C_BADRHO], (unsigned long long)__popcll(w));
}

// sweep wavefront sb of nsb
__device__ __forceinline__ void sweep_density(const Soa &d, const int *__restrict__ scal, int sb,
                                              int nsb, unsigned long long *__restrict__ counters) {
  const int n = scal[S_NP];
  const int stride = nsb * 64;
  unsigned bad = 0;
  for (int p0 = sb * 64 + (int)(threadIdx.x & 63); p0 < n; p0 += kSweep * stride) {
    int t[kSweep];
    double rho[kSweep];
#pragma unroll
    for (int q = 0; q < kSweep; ++q) {
      const int p = p0 + q * stride;
      t[q] = p < n ? d.type[p] : TSPH_WALL;
      rho[q] = p < n ? d.rho[p] : 0.;
    }
#pragma unroll
    for (int q = 0; q < kSweep; ++q)
      if (t[q] != TSPH_WALL && t[q] != TSPH_INLET && t[q] != TSPH_OUTLET)
        bad += rho[q] > 1500. || rho[q] < 0.;
  }
  for (int o = 32; o > 0; o >>= 1) bad += __shfl_xor(bad, o, 64);
  if (bad && (threadIdx.x & 63) == 0) atomicAdd(&counters[C_BADRHO], (unsigned long long)bad);
}

// sweep workgroups that follow wall_blocks wall workgroups for n particles
inline int sweep_blocks(int n) { return grid_for(n, 64 * kSweep); }

// the constants of particle i's case, by scalar loads where the wavefront's
// particles are of one case (nearly all are)
__device__ __forceinline__ Consts wave_consts(const Consts &k0, const Consts *__restrict__ cases,
                                              const uint8_t *__restrict__ cid, int i, bool live) {
  if (!cases) return k0;
  const int c = live ? cid[i] : 0, first = __builtin_amdgcn_readfirstlane(c);
  if (__all(!live || c == first)) return cases[first];
  return cases[c];
}

// The wall-density passes by wavefronts: wavefront b < wall_blocks takes walls
// kWallsPerWave b ..., wavefront wall_blocks + s (s < nsweep) the
// density sweep's share s (counters set).  nwall: the wall count of the cell
// list in use (one of the two alternating slots).
__device__ __forceinline__ void mdbc_wave(int b, int wall_blocks, int nsweep, const Soa &d,
                                           const int *__restrict__ cell_start,
                                           const int *__restrict__ nwall,
                                           const int2 *__restrict__ wall_list, const Consts &k0,
                                           const Consts *__restrict__ cases,
                                           unsigned long long *__restrict__ counters,
                                           const int *__restrict__ scal, double *s_terms) {
  if (b >= wall_blocks) {
    sweep_density(d, scal, b - wall_blocks, nsweep, counters);
    return;
  }
  const int w = b * kWallsPerWave + (int)(threadIdx.x & 63) / kWG;
  const bool live = w < *nwall;
  const int2 wl = live ? wall_list[w] : make_int2(0, 0);
  const int i = wl.x;
  const Consts k = wave_consts(k0, cases, d.cid, i, live);
  const double2 gn = live ? d.gnr[wl.y] : make_double2(0., 0.);
  const double2 r = live ? d.r[i] : make_double2(0., 0.);  // loaded with the ghost node
  const double m = k.m;
  // sums of src/SPH_kernel_approx.h:1141-1342 in its order:
  // rhowsum, drhodx, drhody, a11, a12, a13, a21, a22, a23, a31, a32, a33
  double acc[12];
  wall_sums<12>(d, cell_start + k.cell_base, k, gn, live, acc, s_terms,
                [&](double nrho, double drx, double dry, const KW64 &kw, double *a) {
                  const double mr = quot64_any(m, nrho, recip64(nrho));
                  a[0] = m * kw.w;
                  a[1] = drx * kw.f * m;
                  a[2] = dry * kw.f * m;
                  a[3] = kw.w * mr;
                  a[4] = drx * kw.w * mr;
                  a[5] = dry * kw.w * mr;
                  a[6] = drx * kw.f * mr;
                  a[7] = drx * drx * kw.f * mr;
                  a[8] = drx * dry * kw.f * mr;
                  a[9] = dry * kw.f * mr;
                  a[10] = dry * drx * kw.f * mr;
                  a[11] = dry * dry * kw.f * mr;
                });
  bool wall_bad = false;
  if (live && (threadIdx.x & (kWG - 1)) == 0) {
  const double rhowsum = acc[0], drhodx = acc[1], drhody = acc[2];
  const double a11 = acc[3], a12 = acc[4], a13 = acc[5], a21 = acc[6], a22 = acc[7], a23 = acc[8];
  const double a31 = acc[9], a32 = acc[10], a33 = acc[11];
  const double2 gnd = make_double2(r.x - gn.x, r.y - gn.y);
  double rho = 1000.;
  // determinant, src/SPH_kernel_approx.h:663-675
  const double det = (a11 * a22 * a33 + a12 * a23 * a31 + a13 * a21 * a32 - a31 * a22 * a13 -
                      a32 * a23 * a11 - a33 * a21 * a12);
  if (det > 0.001) {
    const double i11 = (a22 * a33 - a23 * a32) / det;
    const double i12 = -(a12 * a33 - a13 * a32) / det;
    const double i13 = (a12 * a23 - a13 * a22) / det;
    const double i21 = -(a21 * a33 - a23 * a31) / det;
    const double i22 = (a11 * a33 - a13 * a31) / det;
    const double i23 = -(a11 * a23 - a13 * a21) / det;
    const double i31 = (a21 * a32 - a22 * a31) / det;
    const double i32 = -(a11 * a32 - a12 * a31) / det;
    const double i33 = (a11 * a22 - a12 * a21) / det;
    const double dtemp = rhowsum * i11 + drhodx * i12 + drhody * i13;
    const double grx = -(rhowsum * i21 + drhodx * i22 + drhody * i23);
    const double gry = -(rhowsum * i31 + drhodx * i32 + drhody * i33);
    rho = dtemp + grx * gnd.x + gry * gnd.y;
  } else if (a11 > 0) {
    rho = rhowsum / a11;
  }
  if (rho < 1000.) rho = 1000.;  // src/SPH_mDBC.h:44
  d.rho[i] = rho;
  wall_bad = rho > 1500. || rho < 0.;
  }
  if (counters) count_walls(wall_bad, counters);
}

__device__ __forceinline__ void bt_wave(int b, int wall_blocks, int nsweep, const Soa &d,
                                         const int *__restrict__ cell_start,
                                         const int *__restrict__ nwall,
                                         const int2 *__restrict__ wall_list, const Consts &k0,
                                         const Consts *__restrict__ cases,
                                         unsigned long long *__restrict__ counters,
                                         const int *__restrict__ scal, double *s_terms) {
  if (b >= wall_blocks) {
    sweep_density(d, scal, b - wall_blocks, nsweep, counters);
    return;
  }
  const int w = b * kWallsPerWave + (int)(threadIdx.x & 63) / kWG;
  const bool live = w < *nwall;
  const int i = live ? wall_list[w].x : 0;
  const Consts k = wave_consts(k0, cases, d.cid, i, live);
  const double m = k.m;
  double acc[2];  // wsum, rhowsum (src/SPH_kernel_approx.h:1838-1953)
  wall_sums<2>(d, cell_start + k.cell_base, k, live ? d.r[i] : make_double2(0., 0.), live, acc,
               s_terms, [&](double nrho, double, double, const KW64 &kw, double *a) {
                 a[0] = quot64_any(kw.w * m, nrho, recip64(nrho));
                 a[1] = m * kw.w;
               });
  bool wall_bad = false;
  if (live && (threadIdx.x & (kWG - 1)) == 0) {
    double rho = acc[0] > 0. ? acc[1] / acc[0] : 1000.;
    if (rho < 1000.) rho = 1000.;
    d.rho[i] = rho;
    wall_bad = rho > 1500. || rho < 0.;
  }
  if (counters) count_walls(wall_bad, counters);
}

// workgroups of a wall pass: wall workgroups, then sweep workgroups
inline int wall_blocks(const tsph_ctx *c) { return grid_for(c->n_wall, kWallsPerWave); }

// the pass beside another launch: its wavefronts' share
struct WallPass {
  Soa d;
  const int *cell_start, *nwall;
  const int2 *wall_list;
  int walls, sweep;  // wall and sweep wavefronts
  unsigned long long *counters;  // the density count (or nullptr)
};
inline WallPass wall_pass(const tsph_ctx *c, bool count_density) {
  return {c->cur, c->cell_start, c->scal + c->nwall_idx, c->wall_list, wall_blocks(c),
          count_density ? sweep_blocks(c->n_ub) : 0, count_density ? c->counters : nullptr};
}

// wavefront b of the wall pass; terms: walls::kTerms doubles of LDS
template <int WALLS>
__device__ __forceinline__ void wall_wave(int b, const WallPass &wp, const Consts &k0,
                                          const Consts *__restrict__ cases,
                                          const int *__restrict__ scal, double *terms) {
  if (WALLS == TSPH_WALL_MDBC)
    mdbc_wave(b, wp.walls, wp.sweep, wp.d, wp.cell_start, wp.nwall, wp.wall_list, k0, cases,
              wp.counters, scal, terms);
  else
    bt_wave(b, wp.walls, wp.sweep, wp.d, wp.cell_start, wp.nwall, wp.wall_list, k0, cases,
            wp.counters, scal, terms);
}

}  // namespace walls
}  // namespace tsph
