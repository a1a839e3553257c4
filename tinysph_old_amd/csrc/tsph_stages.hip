// Per-particle streaming stages and the wall / probe gathers:
//   Density_to_pressure            src/SPH_pressure.h:65-89
//   Integrate_SymplecticPredictor  src/SPH_integration.h:266-287
//   Integrate_SymplecticCorrector  src/SPH_integration.h:289-309
//   mDBC_compute_density_mdbcGeo, BT_compute_density_BTGeo (tsph_walls.h)
//   RemoveParticlesOutOfDomain     src/SPH_btdebug.h:4-31
//   Water_Elevation(_inverse)      src/SPH_water_level.h:6-150
//   Kernel_velocity_approximation_TEST  src/testing.h:6-148
// The streaming stages are HBM-bound (a few flops per 16-100 bytes).
#include <climits>
#include <cmath>
#include <vector>

#include <algorithm>

#include "tsph_internal.h"
#include "tsph_physics.h"
#include "tsph_walls.h"

namespace tsph {

namespace {

// EOS; on the mixed path it also writes the FP32 pair records of every
// particle (mx.rv != nullptr), which the pair loop that follows reads
__global__ void k_eos(Soa d, Mixed mx, const int *__restrict__ cellof, const int *__restrict__ scal,
                      Consts k0, const Consts *__restrict__ cases,
                      unsigned long long *__restrict__ counters) {
  const int n = scal[S_NP];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned bad = 0;
  if (i < n) {
    const Consts k = case_consts(k0, cases, d.cid, i);
    const int t = d.type[i];
    const double rho = d.rho[i];
    double p;
    if (t != TSPH_OUTLET && t != TSPH_INLET) {
      if (rho > 1500. || rho < 0.) bad = 1;
      p = tait64(rho, k.rho0, k.cs);
      d.p[i] = p;
    } else {
      p = d.p[i];
    }
    if (mx.rv) write_mixed_record(d, mx, cellof, k, i, rho, p);
  }
  const unsigned long long w = __ballot(bad);
  if (w && (threadIdx.x & 63) == 0) atomicAdd(&counters[C_BADRHO], (unsigned long long)__popcll(w));
}

__global__ void k_predictor(Soa d, const int *__restrict__ scal, double dt0,
                            const Consts *__restrict__ cases) {
  const int n = scal[S_NP];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double dt = cases ? cases[d.cid[i]].dt : dt0;
  double rho = d.rho[i];
  double2 r = d.r[i], v = d.v[i];
  d.rho_o[i] = rho;
  d.r_o[i] = r;
  d.v_o[i] = v;
  predict(r, v, rho, d.a[i], d.drho[i], dt);
  d.rho[i] = rho;
  d.r[i] = r;
  d.v[i] = v;
}

// corrector; also records the removal state for the RemoveParticlesOutOfDomain
// that follows it in every driver
__global__ void k_corrector(Soa d, const int *__restrict__ scal, Consts k0,
                            const Consts *__restrict__ cases, double dt0,
                            uint8_t *__restrict__ state) {
  const int n = scal[S_NP];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const Consts k = case_consts(k0, cases, d.cid, i);
  correct_particle(d, k, cases ? k.dt : dt0, i, d.a[i], d.drho[i], state);
}

using namespace walls;

// nwall: the wall count of the cell list in use (one of the two alternating
// slots); workgroups past wall_blocks sweep the other particles' densities
// (counters set)
__global__ __launch_bounds__(64) void k_mdbc(Soa d, const int *__restrict__ cell_start,
                                             const int *__restrict__ nwall,
                                             const int2 *__restrict__ wall_list, Consts k0,
                                             const Consts *__restrict__ cases,
                                             unsigned long long *__restrict__ counters,
                                             const int *__restrict__ scal, int wall_blocks) {
  __shared__ __align__(16) double s_terms[walls::kTerms];
  mdbc_wave(blockIdx.x, wall_blocks, gridDim.x - wall_blocks, d, cell_start, nwall, wall_list, k0,
            cases, counters, scal, s_terms);
}

__global__ __launch_bounds__(64) void k_bt_density(Soa d, const int *__restrict__ cell_start,
                                                   const int *__restrict__ nwall,
                                                   const int2 *__restrict__ wall_list, Consts k0,
                                                   const Consts *__restrict__ cases,
                                                   unsigned long long *__restrict__ counters,
                                                   const int *__restrict__ scal, int wall_blocks) {
  __shared__ __align__(16) double s_terms[walls::kTerms];
  bt_wave(blockIdx.x, wall_blocks, gridDim.x - wall_blocks, d, cell_start, nwall, wall_list, k0,
          cases, counters, scal, s_terms);
}

// Removal.  The reference erases inside an ascending loop without stepping
// back, so the particle that follows an erased one in reference order is never
// examined: in a run of consecutive candidates every other one (the 1st, 3rd,
// ...) is removed.  State per reference position (seq): 0 absent, 1 kept,
// 2 candidate.
// marks for a removal that does not directly follow a corrector
__global__ void k_rm_mark(Soa d, const int *__restrict__ scal, Consts k0,
                          const Consts *__restrict__ cases, uint8_t *__restrict__ state) {
  const int n = scal[S_NP];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  state[d.seq[i]] = removal_state(case_consts(k0, cases, d.cid, i), d.type[i], d.r[i]);
}

__global__ void k_rm_decide(Soa d, const int *__restrict__ scal, const uint8_t *__restrict__ state,
                            unsigned long long *__restrict__ counters) {
  const int n = scal[S_NP];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (removal_decided(state, d.seq[i])) {
    d.type[i] = kRemoved;
    atomicAdd(&counters[C_REMOVED], 1ull);
  }
}

// bounds of the 9 stencil cells about a sampling point in the reference's
// order (cells outside the grid empty)
__device__ __forceinline__ void probe_cells(const int *__restrict__ cell_start, const Consts &k,
                                            double x, double y, int (&lo)[9], int (&hi)[9]) {
  const unsigned npx = (unsigned)(int)((x - k.x0 + k.of) / k.kh);
  const unsigned npy = (unsigned)(int)((y - k.y0 + k.of) / k.kh);
  const int c = (int)(npy + npx * (unsigned)k.ncy);
#pragma unroll
  for (int s = 0; s < 9; ++s) {
    const int cl = c + stencil_off(s, k.ncy);
    const bool in = cl >= 0 && cl < k.ncells;
    lo[s] = in ? cell_start[cl] : 0;
    hi[s] = in ? cell_start[cl + 1] : 0;
  }
}

// Shepard volume sum, src/SPH_water_level.h:6-82 (all particle types), the
// records of kProbePre candidates in flight together
constexpr int kProbePre = 8;
__device__ double sum_kernel_at(const Soa &d, const int *__restrict__ cell_start, const Consts &k,
                                double x, double y) {
  int lo[9], hi[9];
  probe_cells(cell_start, k, x, y, lo, hi);
  const double h = k.h, m = k.m, r2cut = 4.0 * h * h * (1.0 + 1e-12);
  double msum = 0;
#pragma unroll
  for (int s = 0; s < 9; ++s) {
    for (int j = lo[s]; j < hi[s]; j += kProbePre) {
      double2 r[kProbePre];
      double rho[kProbePre];
#pragma unroll
      for (int u = 0; u < kProbePre; ++u) {
        r[u] = d.r[min(j + u, hi[s] - 1)];
        rho[u] = d.rho[min(j + u, hi[s] - 1)];
      }
#pragma unroll
      for (int u = 0; u < kProbePre; ++u) {
        const double drx = x - r[u].x, dry = y - r[u].y;
        const double r2 = drx * drx + dry * dry;
        if (j + u >= hi[s] || !(r2 <= r2cut)) continue;
        const Root64 rt = sqrt64(r2);
        const double qq = quot64(rt.s, h, k.ih);
        if (qq > 2.0) continue;
        const double w = wendland64(rt, qq, k.awen, k.bwen).w;
        msum += quot64_any(m * w, rho[u], recip64(rho[u]));
      }
    }
  }
  return msum;
}

// Water_Elevation's march over the sampling heights (y += i dp_wl, formed in
// the reference's sequential order), kWlBlock heights per workgroup: workgroup
// g takes chunk g, so it adds up the increments before its chunk as well (one
// lane, 9 cycles each, the increments formed by all lanes), and leaves
// {level, index of its first height that meets the threshold} or index -1 (the
// last one also its last height, from which a next launch goes on).
// The chain bounds the launch (4 us per 1000 heights); one workgroup that
// marched chunk after chunk took 83 us per gauge of an 8k-particle dam break
// (1100 to 2200 heights), this 29.
constexpr int kWlBlock = 256, kWlChunks = (kProbeOut - 1) / 2;
// y plus the kWlBlock increments one by one, the next 16 read from LDS while 16
// are added; KEEP: every partial sum to ys
template <bool KEEP>
__device__ __forceinline__ double add_up(double y, const double *inc, double *ys) {
  double q[16], next[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) q[e] = inc[e];
  for (int e0 = 0; e0 < kWlBlock; e0 += 16) {
    const int n0 = e0 + 16 < kWlBlock ? e0 + 16 : 0;
#pragma unroll
    for (int e = 0; e < 16; ++e) next[e] = inc[n0 + e];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      y += q[e];
      if (KEEP) ys[e0 + e] = y;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) q[e] = next[e];
  }
  return y;
}
__global__ __launch_bounds__(kWlBlock) void k_water_level(Soa d, const int *__restrict__ cell_start,
                                                          Consts k, double x, double y0, int inverse,
                                                          int nmax, int chunk0, double *__restrict__ out) {
  __shared__ __align__(16) double inc[2][kWlBlock];
  __shared__ double ys[kWlBlock];
  __shared__ int found;
  const double dp_wl = k.dp * 0.00005;
  const int t = threadIdx.x, chunk = chunk0 + blockIdx.x;  // (y0: before chunk0's first height)
  double y = y0;
  if (t == 0) found = INT_MAX;
  const double sign = inverse ? -1. : 1.;
  inc[chunk0 & 1][t] = sign * ((chunk0 * kWlBlock + t) * dp_wl);
  __syncthreads();
  for (int c = chunk0; c < chunk; ++c) {
    if (t == 0) y = add_up<false>(y, inc[c & 1], ys);
    inc[(c + 1) & 1][t] = sign * (((c + 1) * kWlBlock + t) * dp_wl);
    __syncthreads();
  }
  if (t == 0) y = add_up<true>(y, inc[chunk & 1], ys);
  __syncthreads();
  const int i = chunk * kWlBlock + t;
  if (i < nmax) {
    const double msum = sum_kernel_at(d, cell_start, k, x, ys[t]);
    if (inverse ? (msum >= 0.5) : (msum <= 0.5)) atomicMin(&found, i);
  }
  __syncthreads();
  if (t == 0) {
    double *o = out + 2 * blockIdx.x;
    const int f = found;
    const double yf = ys[f == INT_MAX ? 0 : f - chunk * kWlBlock];
    o[0] = inverse ? yf + f * dp_wl : yf - f * dp_wl;
    o[1] = f == INT_MAX ? -1. : (double)f;
    if (blockIdx.x == gridDim.x - 1) o[2] = y;
  }
}

// Kernel_velocity_approximation_TEST, src/testing.h:6-148, at one point:
// out4 = {rho, p, vx, vy}
__device__ void interpolate_at(const Soa &d, const int *__restrict__ cell_start, const Consts &k,
                               double x, double y, double *out4) {
  const double kh = k.kh, of = k.of;
  const unsigned npx = (unsigned)(int)((x - k.x0 + of) / kh);
  const unsigned npy = (unsigned)(int)((y - k.y0 + of) / kh);
  const int c = (int)(npy + npx * (unsigned)k.ncy);
  double vwx = 0, vwy = 0, wsum = 0, rhow = 0, pw = 0, mw = 0;
  for (int s = 0; s < 9; ++s) {
    const int cl = c + stencil_off(s, k.ncy);
    if (cl < 0 || cl >= k.ncells) continue;
    const int j1 = cell_start[cl + 1];
    for (int j = cell_start[cl]; j < j1; ++j) {
      const double2 nr = d.r[j];
      const double drx = x - nr.x, dry = y - nr.y;
      const double drs = sqrt(drx * drx + dry * dry);
      if (drs / k.h > 2.0) continue;
      const KW64 kw = wendland64(drs, k.h, k.awen, k.bwen);
      const double2 nv = d.v[j];
      wsum += kw.w;
      vwx = vwx + nv.x * kw.w;
      vwy = vwy + nv.y * kw.w;
      rhow = rhow + d.rho[j] * kw.w;
      pw = pw + d.p[j] * kw.w;
      mw += k.m * kw.w / d.rho[j];
    }
  }
  double rho = 0, p = 0, vx = 0, vy = 0;
  if (mw > 0.5) {
    vx = 0. + vwx / wsum;
    vy = 0. + vwy / wsum;
    rho = 0 + rhow / wsum;
    p = 0 + pw / wsum;
  }
  if (wsum == 0) { vx = 0.; vy = 0.; }
  out4[0] = rho; out4[1] = p; out4[2] = vx; out4[3] = vy;
}

// the same by one wavefront: each lane a candidate's terms, then a lane per sum
// adds them in the reference order (one lane walking all candidates: 17 us)
__global__ __launch_bounds__(64) void k_interp_point(Soa d, const int *__restrict__ cell_start,
                                                     Consts k, double x, double y,
                                                     double *__restrict__ out) {
  __shared__ double terms[6][64];
  int lo[9], hi[9];
  probe_cells(cell_start, k, x, y, lo, hi);
  int tot = 0;
#pragma unroll
  for (int s = 0; s < 9; ++s) tot += hi[s] - lo[s];
  const int lane = threadIdx.x;
  const double r2cut = 4.0 * k.h * k.h * (1.0 + 1e-12);
  double sum = 0.;  // lanes 0-5: wsum, vwx, vwy, rhow, pw, mw
  for (int base = 0; base < tot; base += 64) {
    const int f = base + lane;
    int j = 0, pre = 0;
#pragma unroll
    for (int s = 0; s < 9; ++s) {
      j = f >= pre ? lo[s] + f - pre : j;
      pre += hi[s] - lo[s];
    }
    bool ok = f < tot;
    if (ok) {
      const double2 nr = d.r[j], nv = d.v[j];
      const double rho = d.rho[j], p = d.p[j];
      const double drx = x - nr.x, dry = y - nr.y;
      const double r2 = drx * drx + dry * dry;
      const Root64 rt = sqrt64(r2);
      const double qq = quot64(rt.s, k.h, k.ih);
      ok = r2 <= r2cut && qq <= 2.0;
      if (ok) {
        const double w = wendland64(rt, qq, k.awen, k.bwen).w;
        terms[0][lane] = w;
        terms[1][lane] = nv.x * w;
        terms[2][lane] = nv.y * w;
        terms[3][lane] = rho * w;
        terms[4][lane] = p * w;
        terms[5][lane] = quot64_any(k.m * w, rho, recip64(rho));
      }
    }
    const unsigned long long near = __ballot(ok);
    __syncthreads();
    if (lane < 6)
      for (unsigned long long m = near; m; m &= m - 1) sum += terms[lane][__builtin_ctzll(m)];
    __syncthreads();
  }
  const double wsum = __shfl(sum, 0, 64), mw = __shfl(sum, 5, 64);
  // out4 = {rho, p, vx, vy}: sums 3, 4, 1, 2
  const double part = __shfl(sum, lane == 0 ? 3 : lane == 1 ? 4 : lane - 1, 64);
  if (lane < 4) out[lane] = mw > 0.5 && wsum != 0 ? 0. + part / wsum : 0.;
}

// GenerateInterpol's grid, src/SPH_dataInterpolation.h:13-91: point (gx, gy) at
// (x0 + gx dh, y0 + gy dh), stored at POS(gx, gy) = gy + gx ncy
// (src/SPH_defs.h:36), one lane per point
__global__ void k_interp_grid(Soa d, const int *__restrict__ cell_start, Consts k, double x0,
                              double y0, double dh, int ncx, int ncy, double *__restrict__ out,
                              bool soa) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = ncx * ncy;
  if (t >= n) return;
  const int gx = t / ncy, gy = t - gx * ncy;
  double v[4];
  interpolate_at(d, cell_start, k, x0 + gx * dh, y0 + gy * dh, v);
  if (soa) {  // rho[n], p[n], v[2n]
    out[t] = v[0];
    out[n + t] = v[1];
    out[2 * n + 2 * t] = v[2];
    out[2 * n + 2 * t + 1] = v[3];
  } else {
    out[4 * t] = v[0];
    out[4 * t + 1] = v[1];
    out[4 * t + 2] = v[2];
    out[4 * t + 3] = v[3];
  }
}

// --------------------------------------------------------------------------
// Download: the live particles in reference order.  A particle's place is the
// number of live particles with a smaller reference position, so the order
// needs no sort: a bitmap over the positions, its prefix popcounts, and a
// gather into the other particle generation, whose fields then go to the host
// as they are.  Bound by the copies over PCIe that follow (740k particles, r v
// rho p: 36 MB, 0.7 ms at the link's rate; the four launches take 70 us); the
// host sort and permuting copies this replaces took 40 ms.
// --------------------------------------------------------------------------
constexpr int kDlScan = 1024;  // threads of the one workgroup that scans the bitmap
constexpr int kDlItems = 4;    // words per thread and round

__global__ void k_dl_clear(const int *__restrict__ scal, uint32_t *__restrict__ bits) {
  const int w = (scal[S_MAXSEQ] + 31) / 32;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < w; i += gridDim.x * blockDim.x) bits[i] = 0;
}

__device__ __forceinline__ bool dl_live(const Soa &d, int i, int icase) {
  return d.type[i] != kRemoved && (icase < 0 || d.cid[i] == icase);
}

__global__ void k_dl_mark(Soa d, const int *__restrict__ scal, int icase,
                          uint32_t *__restrict__ bits) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= scal[S_NP] || !dl_live(d, i, icase)) return;
  const uint32_t s = d.seq[i];
  atomicOr(&bits[s >> 5], 1u << (s & 31));
}

// live positions before each word, and their total (scal[S_DLNP])
__global__ __launch_bounds__(kDlScan) void k_dl_scan(int *__restrict__ scal,
                                                     const uint32_t *__restrict__ bits,
                                                     int *__restrict__ before) {
  __shared__ int part[kDlScan / 64];
  const int words = (scal[S_MAXSEQ] + 31) / 32;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int carry = 0;
  for (int w0 = 0; w0 < words; w0 += kDlScan * kDlItems) {
    const int w = w0 + threadIdx.x * kDlItems;
    int n[kDlItems], sum = 0;
#pragma unroll
    for (int q = 0; q < kDlItems; ++q) {
      n[q] = w + q < words ? __popc(bits[w + q]) : 0;
      sum += n[q];
    }
    int x = sum;
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) part[wid] = x;
    __syncthreads();
    int at = carry + x - sum;
    for (int u = 0; u < kDlScan / 64; ++u) {
      const int v = part[u];
      if (u < wid) at += v;
      carry += v;
    }
#pragma unroll
    for (int q = 0; q < kDlItems; ++q) {
      if (w + q < words) before[w + q] = at;
      at += n[q];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) scal[S_DLNP] = scal[S_NEWSEQ] = carry;
}

__global__ void k_dl_gather(Soa d, Soa o, const int *__restrict__ scal, int icase, unsigned fields,
                            const uint32_t *__restrict__ bits, const int *__restrict__ before) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= scal[S_NP] || !dl_live(d, i, icase)) return;
  const uint32_t s = d.seq[i];
  const int k = before[s >> 5] + __popc(bits[s >> 5] & ((1u << (s & 31)) - 1u));
  if (fields & DL_R) o.r[k] = d.r[i];
  if (fields & DL_V) o.v[k] = d.v[i];
  if (fields & DL_A) o.a[k] = d.a[i];
  if (fields & DL_R_O) o.r_o[k] = d.r_o[i];
  if (fields & DL_V_O) o.v_o[k] = d.v_o[i];
  if (fields & DL_GNR) o.gnr[k] = d.gnr[s];
  if (fields & DL_N) o.n[k] = d.n[i];
  if (fields & DL_P) o.p[k] = d.p[i];
  if (fields & DL_RHO) o.rho[k] = d.rho[i];
  if (fields & DL_DRHO) o.drho[k] = d.drho[i];
  if (fields & DL_RHO_O) o.rho_o[k] = d.rho_o[i];
  if (fields & DL_TYPE) o.type[k] = d.type[i];
  if (fields & DL_INDEX) o.index[k] = d.index[s];
}

// A relabel of the reference positions in two passes (the new positions are those
// of a download): first every slot's new position and what moves with it into the
// other generation and the download's buffers, then all of it to its place.  The
// removed slots take the positions after the live ones, in any order.  Five
// launches: 333k particles 71 us, on the host 12 ms (a sort, and the fields by
// position down and up).
__global__ void k_renumber_gather(Soa d, Soa o, int *__restrict__ scal,
                                  const uint8_t *__restrict__ state, const uint32_t *__restrict__ bits,
                                  const int *__restrict__ before) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= scal[S_NP]) return;
  if (d.type[i] == kRemoved) {
    o.seq[i] = (uint32_t)atomicAdd(&scal[S_NEWSEQ], 1);
    return;
  }
  const uint32_t s = d.seq[i];
  const int k = before[s >> 5] + __popc(bits[s >> 5] & ((1u << (s & 31)) - 1u));
  o.seq[i] = (uint32_t)k;
  o.type[k] = state[s];
  o.index[k] = d.index[s];
  if (d.gnr) o.gnr[k] = d.gnr[s];
}

__global__ void k_renumber_place(Soa d, Soa o, int *__restrict__ scal, uint8_t *__restrict__ state,
                                 int seq_cap, const int *__restrict__ nwall,
                                 int2 *__restrict__ wall_list) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = scal[S_NP], m = scal[S_DLNP];
  if (i < seq_cap) state[i] = i < m ? o.type[i] : 0;
  if (i < m) {
    d.index[i] = o.index[i];
    if (d.gnr) d.gnr[i] = o.gnr[i];
  }
  if (i < n) d.seq[i] = o.seq[i];
  if (i < *nwall) wall_list[i].y = (int)o.seq[wall_list[i].x];
  if (i == 0) scal[S_MAXSEQ] = scal[S_NEWSEQ];
}

// live particles per case: a histogram in LDS per workgroup, then one atomic
// per case that the workgroup saw
__global__ __launch_bounds__(256) void k_case_counts(Soa d, const int *__restrict__ scal, int ncases,
                                                     int *__restrict__ counts) {
  __shared__ int h[256];
  h[threadIdx.x] = 0;
  __syncthreads();
  const int n = scal[S_NP];
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    if (d.type[i] != kRemoved) atomicAdd(&h[d.cid[i]], 1);
  __syncthreads();
  if ((int)threadIdx.x < ncases && h[threadIdx.x]) atomicAdd(&counts[threadIdx.x], h[threadIdx.x]);
}

__global__ void k_iota(int *__restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = i;
}

__global__ void k_zero_ints(int *__restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

}  // namespace

int launch_download_gather(tsph_ctx *c, int icase, unsigned fields) {
  uint32_t *bits = reinterpret_cast<uint32_t *>(c->hcell);
  const int g = grid_for(c->n_ub, 256);
  Soa to = c->alt;
  to.gnr = c->pos_gnr;
  to.index = c->pos_index;
  const int wg = grid_for((int)std::min<size_t>(dl_words(c->seq_cap), 1 << 18), 256);
  hipLaunchKernelGGL(k_dl_clear, dim3(wg), dim3(256), 0, c->stream, c->scal, bits);
  hipLaunchKernelGGL(k_dl_mark, dim3(g), dim3(256), 0, c->stream, c->cur, c->scal, icase, bits);
  hipLaunchKernelGGL(k_dl_scan, dim3(1), dim3(kDlScan), 0, c->stream, c->scal, bits, c->hrank);
  hipLaunchKernelGGL(k_dl_gather, dim3(g), dim3(256), 0, c->stream, c->cur, to, c->scal, icase, fields,
                     bits, c->hrank);
  TSPH_HIP(hipGetLastError());
  return 0;
}

int launch_renumber(tsph_ctx *c) {
  uint32_t *bits = reinterpret_cast<uint32_t *>(c->hcell);
  const int g = grid_for(c->n_ub, 256);
  Soa to = c->alt;
  to.gnr = c->pos_gnr;
  to.index = c->pos_index;
  const int wg = grid_for((int)std::min<size_t>(dl_words(c->seq_cap), 1 << 18), 256);
  hipLaunchKernelGGL(k_dl_clear, dim3(wg), dim3(256), 0, c->stream, c->scal, bits);
  hipLaunchKernelGGL(k_dl_mark, dim3(g), dim3(256), 0, c->stream, c->cur, c->scal, -1, bits);
  hipLaunchKernelGGL(k_dl_scan, dim3(1), dim3(kDlScan), 0, c->stream, c->scal, bits, c->hrank);
  hipLaunchKernelGGL(k_renumber_gather, dim3(g), dim3(256), 0, c->stream, c->cur, to, c->scal,
                     c->seqstate, bits, c->hrank);
  hipLaunchKernelGGL(k_renumber_place, dim3(grid_for(c->seq_cap, 256)), dim3(256), 0, c->stream, c->cur,
                     to, c->scal, c->seqstate, c->seq_cap, c->scal + c->nwall_idx, c->wall_list);
  TSPH_HIP(hipGetLastError());
  return 0;
}

int launch_iota(tsph_ctx *c, int *p, int n) {
  hipLaunchKernelGGL(k_iota, dim3(grid_for(n, 256)), dim3(256), 0, c->stream, p, n);
  TSPH_HIP(hipGetLastError());
  return 0;
}

// k_place: to[at[i]] = from[i]
namespace {
template <typename V>
__global__ void k_place(V *__restrict__ to, const V *__restrict__ from,
                        const uint32_t *__restrict__ at, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) to[at[i]] = from[i];
}
}  // namespace

int launch_place(tsph_ctx *c, int n, bool gnr) {
  const dim3 g(grid_for(n, 256)), b(256);
  hipLaunchKernelGGL(k_place<int32_t>, g, b, 0, c->stream, c->cur.index, c->pos_index, c->cur.seq, n);
  if (gnr)
    hipLaunchKernelGGL(k_place<double2>, g, b, 0, c->stream, c->cur.gnr, c->pos_gnr, c->cur.seq, n);
  TSPH_HIP(hipGetLastError());
  return 0;
}

int launch_case_counts(tsph_ctx *c, int *counts) {
  hipLaunchKernelGGL(k_zero_ints, dim3(1), dim3(256), 0, c->stream, counts, c->ncases);
  hipLaunchKernelGGL(k_case_counts, dim3(std::min(grid_for(c->n_ub, 1024), 4 * c->num_cu)), dim3(256), 0,
                     c->stream, c->cur, c->scal, c->ncases, counts);
  TSPH_HIP(hipGetLastError());
  return 0;
}

int launch_eos(tsph_ctx *c) {
  Mixed mx = c->prm.precision == TSPH_PREC_MIXED ? c->mx : Mixed{};
  hipLaunchKernelGGL(k_eos, dim3(grid_for(c->n_ub, 256)), dim3(256), 0, c->stream, c->cur, mx,
                     c->cellof, c->scal, c->k, c->cases, c->counters);
  TSPH_HIP(hipGetLastError());
  // the records are only meaningful for the cell list they were built on
  c->records_valid = c->prm.precision == TSPH_PREC_MIXED && c->cells_valid;
  return 0;
}

int launch_predictor(tsph_ctx *c, double dt) {
  c->olds_stale = false;  // it rewrites r_o, v_o, rho_o of every particle
  hipLaunchKernelGGL(k_predictor, dim3(grid_for(c->n_ub, 256)), dim3(256), 0, c->stream, c->cur,
                     c->scal, dt, c->cases);
  TSPH_HIP(hipGetLastError());
  c->records_valid = false;
  c->marks_valid = false;
  return 0;
}

int launch_corrector(tsph_ctx *c, double dt) {
  if (int e = ensure_olds(c)) return e;
  hipLaunchKernelGGL(k_corrector, dim3(grid_for(c->n_ub, 256)), dim3(256), 0, c->stream, old_state(c),
                     c->scal, c->k, c->cases, dt, c->seqstate);
  TSPH_HIP(hipGetLastError());
  c->records_valid = false;
  c->marks_valid = true;
  return 0;
}

int launch_mdbc(tsph_ctx *c, bool count_density) {
  const int wb = grid_for(c->n_wall, kWallsPerWave), sb = count_density ? sweep_blocks(c->n_ub) : 0;
  hipLaunchKernelGGL(k_mdbc, dim3(wb + sb), dim3(64), 0, c->stream, c->cur, c->cell_start,
                     c->scal + c->nwall_idx, c->wall_list, c->k, c->cases,
                     count_density ? c->counters : nullptr, c->scal, wb);
  TSPH_HIP(hipGetLastError());
  c->records_valid = false;
  return 0;
}

int launch_bt_density(tsph_ctx *c, bool count_density) {
  const int wb = grid_for(c->n_wall, kWallsPerWave), sb = count_density ? sweep_blocks(c->n_ub) : 0;
  hipLaunchKernelGGL(k_bt_density, dim3(wb + sb), dim3(64), 0, c->stream, c->cur,
                     c->cell_start, c->scal + c->nwall_idx, c->wall_list, c->k, c->cases,
                     count_density ? c->counters : nullptr, c->scal, wb);
  TSPH_HIP(hipGetLastError());
  c->records_valid = false;
  return 0;
}

int launch_remove(tsph_ctx *c) {
  if (!c->marks_valid) {
    hipLaunchKernelGGL(k_rm_mark, dim3(grid_for(c->n_ub, 256)), dim3(256), 0, c->stream, c->cur,
                       c->scal, c->k, c->cases, c->seqstate);
  }
  hipLaunchKernelGGL(k_rm_decide, dim3(grid_for(c->n_ub, 256)), dim3(256), 0, c->stream, c->cur,
                     c->scal, c->seqstate, c->counters);
  TSPH_HIP(hipGetLastError());
  c->marks_valid = false;  // removed particles are re-marked as absent next time
  return 0;
}

int run_water_elevation(tsph_ctx *c, double x, double y0, int inverse, double *out) {
  const Consts &k = c->k;
  const double dp_wl = k.dp * 0.00005;
  // heights up to the top, as many as an int counts (a conversion beyond that is
  // undefined on the host; on the device it saturates)
  const int nmax = (int)std::clamp(k.ym / dp_wl, (double)INT_MIN, (double)INT_MAX);
  *out = NAN;
  // the march is out of the domain after sqrt(2 distance / dp_wl) heights; one
  // launch covers that, and the few calls that march on take more of them
  const double far = std::max(0., inverse ? y0 - k.y0 : k.ym - y0);
  int n = 1 + (int)std::min<double>(kWlChunks - 1, std::sqrt(2. * far / dp_wl) / kWlBlock);
  for (int chunk = 0; (long long)chunk * kWlBlock < nmax; chunk += n, n = kWlChunks) {
    double res[2 * kWlChunks + 1];
    hipLaunchKernelGGL(k_water_level, dim3(n), dim3(kWlBlock), 0, c->stream, c->cur, c->cell_start, k,
                       x, y0, inverse, nmax, chunk, c->probe_out);
    TSPH_HIP(hipGetLastError());
    TSPH_HIP(hipMemcpyAsync(res, c->probe_out, (2 * n + 1) * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    TSPH_HIP(hipStreamSynchronize(c->stream));
    for (int g = 0; g < n; ++g)
      if (res[2 * g + 1] >= 0.) {
        *out = res[2 * g];
        return 0;
      }
    y0 = res[2 * n];
  }
  return 0;
}

// out: 4 doubles per grid point, device memory
int launch_interp_grid(tsph_ctx *c, double x0, double y0, double dh, int ncx, int ncy, double *out,
                       bool soa) {
  hipLaunchKernelGGL(k_interp_grid, dim3(grid_for(ncx * ncy, 64)), dim3(64), 0, c->stream, c->cur,
                     c->cell_start, c->k, x0, y0, dh, ncx, ncy, out, soa);
  TSPH_HIP(hipGetLastError());
  return 0;
}

int run_interpolate_point(tsph_ctx *c, double x, double y, double *out4) {
  double *dout = c->probe_out;
  hipLaunchKernelGGL(k_interp_point, dim3(1), dim3(64), 0, c->stream, c->cur, c->cell_start, c->k,
                     x, y, dout);
  TSPH_HIP(hipGetLastError());
  TSPH_HIP(hipMemcpyAsync(out4, dout, 4 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  TSPH_HIP(hipStreamSynchronize(c->stream));
  return 0;
}

}  // namespace tsph
