// Riemann-ALE-SPH, first order: the pipeline the ALE dam-break driver runs
// (cases/ALESPH_dambreakLong/run.sh -> SPH_simulationINT.h:84-132):
//   Integrate_LeapFrog_partOne  src/RALESPH_integration.h:10-36
//   Compute_Forces              src/RALESPH_interaction.h:12-287
//   Integrate_LeapFrog_partTwo  src/RALESPH_integration.h:38-107
// with the particle volume variables of ALESPH_Add_particle
// (src/SPH_particle_system.h:51-108).
//
// The pair loop is the cell walk of tsph_tiles.h in FP64 and reuses the tile
// machinery of the WCSPH loops in the mixed form (persistent waves over
// XCD-banded tiles, neighbour slices staged in LDS, lane-private neighbour
// lists).  Per pair it solves the linearised Riemann problem along
// the pair normal (src/ALESPH_riemann_solver.h:20-34, 86-96), with a
// one-sided wall state for BT wall neighbours (src/RALESPH_interaction.h:217-253).
//
// Reference quirk kept: gamma_sum is declared per cell and never reset between
// the cell's particles (src/RALESPH_interaction.h:48, 257, 277-280), so a fluid
// particle with no neighbour in its support takes the "gamma == 0" (all-zero)
// branch only if no earlier fluid particle of its cell had one.  The pair loop
// records whether each particle's own sum is non-zero; k_rale_isolated then
// settles the particles whose own sum is zero by looking at the earlier
// particles of their cell (reference order inside a cell).
#include "tsph_internal.h"
#include "tsph_physics.h"
#include "tsph_tiles.h"

namespace tsph {

namespace {

using namespace tiles;

// constants of the FP64 pass
struct Rale64 {
  double h, ih, awen, bwen, cs, ics, cs2, ics2, rho0, irho0, cb, dp, gx, gy;
};
__host__ __device__ __forceinline__ Rale64 rale64(const Consts &k) {
  return {k.h, k.ih, k.awen, k.bwen, k.cs, 1. / k.cs, k.cs * k.cs, 1. / (k.cs * k.cs), k.rho0,
          1. / k.rho0, k.cb, k.dp, k.gx, k.gy};
}

// one particle of the FP64 pass
struct RaleP {
  double2 r, v, n;
  double rho, omega;
  int t;
};

// the terms of one RALE pair (d omega, d omega rho, d omega v) in the reference
// operand order, zeros beyond the exact support; bit 0 of the result: inside
// it, bit 1: its gamma term W m / rho_j is not 0 (W is 0 only at qq = 2)
__device__ __forceinline__ int rale_pair64(const Rale64 &k, const RaleP &o, const RaleP &b,
                                           double (&t)[4]) {
  const double c0 = k.cs, dp = k.dp, rho0 = k.rho0;
  const double drx = o.r.x - b.r.x, dry = o.r.y - b.r.y;
  const Root64 rt = sqrt64((drx * drx) + (dry * dry));
  const double qq = quot64(rt.s, k.h, k.ih);
  const KW64 kw = wendland64(rt, qq, k.awen, k.bwen);
  const double W = kw.w;
  const double dWx = drx * kw.f, dWy = dry * kw.f;
  const double dvx = o.v.x - b.v.x, dvy = o.v.y - b.v.y;
  const double dvdW = dvx * dWx + dvy * dWy;
  const double inv = quot64(1., rt.s, recip_of_root64(rt));
  const double drnx = drx * inv * (-1), drny = dry * inv * (-1);
  const double vL = o.v.x * drnx + o.v.y * drny;
  const double vR = b.v.x * drnx + b.v.y * drny;
  const double avgrho = 0.5 * (o.rho + b.rho);
  const double vss = 0.5 * (vR + vL) - quot64_any(0.5 * (b.rho - o.rho) * c0, avgrho, recip64(avgrho));
  const double dd = vL - vR;
  const double mx = dd > 0 ? dd : 0;
  const double e = 3. * mx;
  const double beta = e < c0 ? e : c0;
  const double rhos = 0.5 * (o.rho + b.rho) +
                      quot64_any(0.5 * beta * (vL - vR) * (0.5 * (o.rho + b.rho)), k.cs2, k.ics2);
  const double vsx = drnx * vss + ((o.v.x + b.v.x) * 0.5 - drnx * (vL + vR) * 0.5);
  const double vsy = drny * vss + ((o.v.y + b.v.y) * 0.5 - drny * (vL + vR) * 0.5);
  if (b.t == TSPH_WALL) {
    const double nbx = b.n.x * (-1), nby = b.n.y * (-1);
    const double rw = o.rho - quot64_any(((0 - o.v.x) * nbx + (0 - o.v.y) * nby) * o.rho, c0, k.ics);
    const double pw = c0 * c0 * (rw - rho0) * 1;
    const double dvn = dvx * nbx + dvy * nby;
    t[0] = 0. - dvn * W * dp;
    t[1] = 0.;
    t[2] = 0. - 2 * W * dp * (pw * nbx);
    t[3] = 0. - 2 * W * dp * (pw * nby);
  } else {
    // Compute_Pressure (tait64)
    const double ps = k.cb * (pow7(quot64_any(rhos, rho0, k.irho0)) - 1);
    const double vsdW = (vsx - o.v.x) * dWx + (vsy - o.v.y) * dWy;
    t[0] = 0. - dvdW * b.omega;
    t[1] = 0. - 2 * rhos * b.omega * vsdW;
    t[2] = 0. - 2 * b.omega * ((rhos * vsx * (vsx - o.v.x) + ps) * dWx + (rhos * vsx * (vsy - o.v.y)) * dWy);
    t[3] = 0. - 2 * b.omega * ((rhos * vsy * (vsx - o.v.x)) * dWx + (rhos * vsy * (vsy - o.v.y) + ps) * dWy);
  }
  if (!(qq <= 2.0)) t[0] = t[1] = t[2] = t[3] = 0.;
  return (int)(qq <= 2.0) | ((int)((qq < 2.0) & (fabs(b.rho) != INFINITY)) << 1);
}

// outputs for a particle whose own gamma sum is non-zero (:271-273), or the
// all-zero branch (:265-267) pending k_rale_isolated
template <class D, class K>
__device__ __forceinline__ void rale_finish(const D &d, const K &k, int i, double ao,
                                           double arho, double dom, double domrho, double dovx,
                                           double dovy, bool nonzero, uint8_t *gflag) {
  if (nonzero) {
    d.domega[i] = dom * ao;
    d.domegarho[i] = domrho * ao;
    d.domegav[i] = make_double2(dovx * ao - k.gx * ao * arho, dovy * ao - k.gy * ao * arho);
  } else {
    d.domega[i] = 0.;
    d.domegarho[i] = 0.;
    d.domegav[i] = make_double2(0., 0.);
  }
  gflag[i] = nonzero;
}

// FP64: the cell walk's policy (cells64, tsph_tiles.h)
struct RalePtr {
  const double2 *r, *v, *n;
  const double *rho, *omega;
  const uint8_t *type;
  double *domega, *domegarho;
  double2 *domegav;
  uint8_t *gflag;
};

template <int H>
struct RaleCell64 {
  RalePtr d;
  Rale64 k;
  static constexpr int kSums = 4, kSlotBytes = 4 * 16 + 1, kWaves = H == 2 ? 4 : 2;
  static constexpr int kSlots = cell_slots_of<H>();
  static constexpr bool kFlag = true, kSkip = false;
  struct Lds {
    double2 *r, *v, *rw, *n;  // rw = {rho, omega}
    uint8_t *t;
  };
  using Rec = RaleP;
  static __device__ __forceinline__ Lds lds(unsigned char *b, int cap) {
    double2 *p = reinterpret_cast<double2 *>(b);
    return {p, p + cap, p + 2 * cap, p + 3 * cap, reinterpret_cast<uint8_t *>(p + 4 * cap)};
  }
  __device__ __forceinline__ void set(const Consts &) {}  // (no batched ALE contexts)
  __device__ __forceinline__ Rec load(int j) const {
    return {d.r[j], d.v[j], d.n ? d.n[j] : make_double2(0., 0.), d.rho[j], d.omega[j], d.type[j]};
  }
  __device__ __forceinline__ void store(const Lds &L, int l, const Rec &q) const {
    L.r[l] = q.r;
    L.v[l] = q.v;
    L.rw[l] = make_double2(q.rho, q.omega);
    L.n[l] = q.n;
    L.t[l] = (uint8_t)q.t;
  }
  static __device__ __forceinline__ Rec slot(const Lds &L, int l) {
    const double2 rw = L.rw[l];
    return {L.r[l], L.v[l], L.n[l], rw.x, rw.y, L.t[l]};
  }
  __device__ __forceinline__ bool act_lds(const Lds &L, int l) const { return L.t[l] == TSPH_FLUID; }
  __device__ __forceinline__ bool skip_lds(const Lds &, int) const { return false; }
  __device__ __forceinline__ double2 pos_lds(const Lds &L, int l) const { return L.r[l]; }
  __device__ __forceinline__ int terms(const Lds &L, int p, int l, double (&t)[kSums]) const {
    return rale_pair64(k, slot(L, p), slot(L, l), t);
  }
  __device__ __forceinline__ void sums(const Lds &L, int p, int i, const double (&s)[kSums],
                                       bool some) const {
    const double2 rw = L.rw[p];
    rale_finish(d, k, i, rw.y, rw.x, s[0], s[1], s[2], s[3], some, d.gflag);
  }
  __device__ __forceinline__ void far(int i, const int *cs, const CellGrid &g, int c, unsigned &npair,
                                      unsigned &ncand, unsigned &nact) const {
    const Rec o = load(i);
    if (o.t != TSPH_FLUID) return;
    ++nact;
    const int cx = c / g.ncy, cy = c - cx * g.ncy;
    double s[kSums] = {0., 0., 0., 0.};
    bool some = false;
    for (int q = 0; q < 9; ++q) {
      int dx, dy;
      stencil_dxy(q, dx, dy);
      if (cx + dx < 0 || cx + dx >= g.ncx || cy + dy < 0 || cy + dy >= g.ncy) continue;
      const int cl = c + dy + dx * g.ncy;
      for (int j = cs[cl]; j < cs[cl + 1]; ++j) {
        if (j == i) continue;
        ++ncand;
        const Rec b = load(j);
        const double drx = o.r.x - b.r.x, dry = o.r.y - b.r.y;
        if (drx * drx + dry * dry > g.c2) continue;
        double t[kSums];
        const int got = rale_pair64(k, o, b, t);
        npair += got & 1;
        some |= (got & 2) != 0;
        for (int u = 0; u < kSums; ++u) s[u] += t[u];
      }
    }
    rale_finish(d, k, i, o.omega, o.rho, s[0], s[1], s[2], s[3], some, d.gflag);
  }
};

template <class P>
__global__ __launch_bounds__(P::kWaves * kWave, cell_halves<P>() == 2 ? 3 : 2) void k_rale_cells64(
    P pol, CellGrid g, const int *__restrict__ cell_start, CellSource src,
    unsigned long long *__restrict__ counters) {
  cells64(pol, g, cell_start, nullptr, 1, src, counters);
}

// --------------------------------------------------------------------------
// mixed form: FP32 fluxes (positions staged relative to the tile, computed in
// FP64 and rounded once; density as rho - rho0), FP64 outputs
// --------------------------------------------------------------------------
struct AccA32 {
  float dom = 0, domrho = 0, dovx = 0, dovy = 0, gamma = 0;
};

struct CA32 {
  float h, ih, m, c0, ic0, rho0, dp, r2cut, awen, bwen, btait;
};

__device__ __forceinline__ void rale_pair32(const CA32 &c, AccA32 &s, float drx, float dry, float r2,
                                            float2 vi, float adev, float2 vj, float ndev, float no,
                                            int nt, float2 n) {
#pragma clang fp contract(fast)
  const float drs = __builtin_amdgcn_sqrtf(r2);
  const float inv = __builtin_amdgcn_rcpf(drs);
  const float qq = drs * c.ih;
  const float wq1 = 1.f - 0.5f * qq;
  const float wq2 = wq1 * wq1;
  const float W = c.awen * (qq + qq + 1.f) * wq2 * wq2;
  const float f = c.bwen * wq2 * wq1 * c.ih;
  const float dWx = drx * f, dWy = dry * f;
  const float dvx = vi.x - vj.x, dvy = vi.y - vj.y;
  const float dvdW = dvx * dWx + dvy * dWy;
  const float drnx = -drx * inv, drny = -dry * inv;
  const float vL = vi.x * drnx + vi.y * drny;
  const float vR = vj.x * drnx + vj.y * drny;
  const float arho = c.rho0 + adev, nrho = c.rho0 + ndev;
  const float avgrho = c.rho0 + 0.5f * (adev + ndev);
  const float vss = 0.5f * (vR + vL) - 0.5f * (ndev - adev) * c.c0 * __builtin_amdgcn_rcpf(avgrho);
  const float dd = vL - vR;
  const float beta = fminf(3.f * fmaxf(dd, 0.f), c.c0);
  const float rsdev = 0.5f * (adev + ndev) + 0.5f * beta * dd * avgrho * (c.ic0 * c.ic0);
  const float vsx = drnx * vss + (0.5f * (vi.x + vj.x) - 0.5f * drnx * (vL + vR));
  const float vsy = drny * vss + (0.5f * (vi.y + vj.y) - 0.5f * drny * (vL + vR));
  if (nt == TSPH_WALL) {
    const float nbx = -n.x, nby = -n.y;
    // wall state rho_w - rho0 = (rho_i - rho0) + (v_i . nb) rho_i / c0, linear EOS
    const float pw = c.c0 * c.c0 * (adev + (vi.x * nbx + vi.y * nby) * arho * c.ic0);
    s.dovx -= 2.f * W * c.dp * (pw * nbx);
    s.dovy -= 2.f * W * c.dp * (pw * nby);
    s.dom -= (dvx * nbx + dvy * nby) * W * c.dp;
  } else {
    // Tait from the density deviation: B((1+x)^7 - 1), binomial expansion
    const float x = rsdev * (1.f / c.rho0);
    const float ps = c.btait * x * (7.f + x * (21.f + x * (35.f + x * (35.f + x * (21.f + x * (7.f + x))))));
    const float rhos = c.rho0 + rsdev;
    const float ex = vsx - vi.x, ey = vsy - vi.y;
    s.dovx -= 2.f * no * ((rhos * vsx * ex + ps) * dWx + (rhos * vsx * ey) * dWy);
    s.dovy -= 2.f * no * ((rhos * vsy * ex) * dWx + (rhos * vsy * ey + ps) * dWy);
    s.dom -= dvdW * no;
    s.domrho -= 2.f * rhos * no * (ex * dWx + ey * dWy);
  }
  s.gamma += W * c.m * __builtin_amdgcn_rcpf(nrho);
}

__global__ __launch_bounds__(kWave * kPoolWaves) void k_rale32(Soa d, const int *__restrict__ cell_start,
                                                  const int *__restrict__ cellof, Consts k, int rows,
                                                  int *__restrict__ scal,
                                                  const int *__restrict__ tile_list, int cap,
                                                  int lds_wave,
                                                  uint8_t *__restrict__ gflag,
                                                  unsigned long long *__restrict__ counters) {
#pragma clang fp contract(fast)
  extern __shared__ __align__(16) unsigned char smem[];
  unsigned char *wl = wave_lds<false>(smem, lds_wave);
  int *tab = reinterpret_cast<int *>(wl);
  float2 *s_pos = reinterpret_cast<float2 *>(wl + kTabBytes);
  float2 *s_vel = s_pos + cap;
  float2 *s_dw = s_vel + cap;  // {rho - rho0, omega}
  float2 *s_n = s_dw + cap;
  uint16_t *s_list = reinterpret_cast<uint16_t *>(s_n + cap);
  uint8_t *s_t = reinterpret_cast<uint8_t *>(s_list + kList * kWave);

  CA32 c;
  c.h = (float)k.h; c.ih = 1.f / c.h; c.m = (float)k.m; c.c0 = (float)k.cs; c.ic0 = 1.f / c.c0;
  c.rho0 = (float)k.rho0; c.dp = (float)k.dp; c.r2cut = 4.f * c.h * c.h;
  c.awen = (float)k.awen; c.bwen = (float)k.bwen; c.btait = (float)(k.cs * k.cs * k.rho0 / 7.);

  if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&counters[C_PASSES], 1ull);
  unsigned npair = 0, ncand = 0, nact = 0;
  TileQueue tq = tq_begin<false>(scal, nullptr, tile_list, smem);
  for (int it = tq_take<false>(tq, 0); it >= 0;) {
    wave_sync();
    const int entry = tile_list[it];
    Tile t;
    tile_begin(k, cell_start, entry_tile(entry), rows, tab, t);
    entry_part(entry, t);
    const bool staged = t.lq[3] <= cap;
    const int mid = t.row_lo + (t.nrows >> 1);
    const double ox = k.x0 - k.of + t.cx * k.kh, oy = k.y0 - k.of + mid * k.kh;
    if (staged) {
      for (int l = tile_lane(); l < t.lq[3]; l += kWave) {
        const int j = l - sel3(t.base, slice_of(t, l));
        const double2 r = d.r[j], v = d.v[j];
        s_pos[l] = make_float2((float)(r.x - ox), (float)(r.y - oy));
        s_vel[l] = make_float2((float)v.x, (float)v.y);
        s_dw[l] = make_float2((float)(d.rho[j] - k.rho0), (float)d.omega[j]);
        s_t[l] = d.type[j];
        s_n[l] = d.n ? make_float2((float)d.n[j].x, (float)d.n[j].y) : make_float2(0.f, 0.f);
      }
    }
    wave_sync();
    const int next = tq_take<false>(tq, 0);
    const int lane = tile_lane();
    uint16_t *my_list = s_list + lane;
    for (int i0 = t.own0; i0 < t.own1; i0 += kWave) {
      const int i = i0 + lane;
      int li = 0, ri = 0;
      bool act = false;
      if (i < t.own1) {
        li = i + t.base[1];
        act = d.type[i] == TSPH_FLUID;
        ri = cellof[i] - t.cx * k.ncy - t.row_lo;
      }
      nact += act;
      const double2 ar = act ? d.r[i] : make_double2(0., 0.);
      const double2 av = act ? d.v[i] : make_double2(0., 0.);
      const float2 pi = make_float2((float)(ar.x - ox), (float)(ar.y - oy));
      const float2 vi = make_float2((float)av.x, (float)av.y);
      const double arho = act ? d.rho[i] : 1.;
      const float adev = (float)(arho - k.rho0);
      AccA32 s;
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
                const double2 r = d.r[j];
                const float drx = pi.x - (float)(r.x - ox), dry = pi.y - (float)(r.y - oy);
                const float r2 = drx * drx + dry * dry;
                if (!(r2 < c.r2cut)) continue;
                ++npair;
                const double2 v = d.v[j];
                const float2 nn = d.n ? make_float2((float)d.n[j].x, (float)d.n[j].y) : make_float2(0.f, 0.f);
                rale_pair32(c, s, drx, dry, r2, vi, adev, make_float2((float)v.x, (float)v.y),
                            (float)(d.rho[j] - k.rho0), (float)d.omega[j], d.type[j], nn);
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
        int cur = 0;
        while (__any(cur < tot)) {
          int cnt = 0;
          while (cur < tot && cnt < kList) {
            const int j = cur < n0 ? a0 + cur : (cur < n0 + n1 ? a1 + (cur - n0) : a2 + (cur - n0 - n1));
            ++cur;
            if (j == li) continue;
            ++ncand;
            const float2 pj = s_pos[j];
            const float drx = pi.x - pj.x, dry = pi.y - pj.y;
            if (drx * drx + dry * dry < c.r2cut) my_list[(cnt++) * kWave] = (uint16_t)j;
          }
          npair += cnt;
          for (int e = 0; e < cnt; ++e) {
            const int j = my_list[e * kWave];
            const float2 pj = s_pos[j], dw = s_dw[j];
            const float drx = pi.x - pj.x, dry = pi.y - pj.y;
            rale_pair32(c, s, drx, dry, drx * drx + dry * dry, vi, adev, s_vel[j], dw.x, dw.y, s_t[j],
                        s_n[j]);
          }
        }
      }
      if (act) {
        const double ao = d.omega[i];
        rale_finish(d, k, i, ao, arho, (double)s.dom, (double)s.domrho, (double)s.dovx,
                    (double)s.dovy, s.gamma != 0.f, gflag);
      }
    }
    it = next;
  }
  wave_count(npair, ncand, nact, counters);
}

// settles fluid particles without neighbours: the reference's cell-wide
// gamma_sum is non-zero for them iff an earlier fluid particle of the same cell
// had neighbours (src/RALESPH_interaction.h:263-274)
__global__ void k_rale_isolated(Soa d, const int *__restrict__ cell_start,
                                const int *__restrict__ cellof, const int *__restrict__ scal,
                                const uint8_t *__restrict__ gflag, Consts k) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= scal[S_NP] || d.type[i] != TSPH_FLUID || gflag[i]) return;
  const int c = cellof[i];
  bool earlier = false;
  for (int j = cell_start[c]; j < i; ++j) earlier |= d.type[j] == TSPH_FLUID && gflag[j];
  if (!earlier) return;
  const double ao = d.omega[i], arho = d.rho[i];
  const double z = 0.;
  d.domega[i] = z * ao;
  d.domegarho[i] = z * ao;
  d.domegav[i] = make_double2(z * ao - k.gx * ao * arho, z * ao - k.gy * ao * arho);
}

// ALESPH_Add_particle's volume variables: omega = dp^2, omega*rho, omega*v
__global__ void k_ale_init(Soa d, const int *__restrict__ scal, double dp) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= scal[S_NP]) return;
  const double w = dp * dp;
  const double2 v = d.v[i];
  const double orho = d.rho[i] * (dp * dp);
  const double2 ov = make_double2(v.x * (dp * dp), v.y * (dp * dp));
  d.omega[i] = w;
  d.omegarho[i] = orho;
  d.omegav[i] = ov;
  d.omega_o[i] = w;
  d.omegarho_o[i] = orho;
  d.omegav_o[i] = ov;
  d.domega[i] = 0.;
  d.domegarho[i] = 0.;
  d.domegav[i] = make_double2(0., 0.);
  d.gradrho[i] = d.gradvx[i] = d.gradvy[i] = make_double2(0., 0.);
}

// Integrate_LeapFrog_partOne, src/RALESPH_integration.h:10-36
__global__ void k_rale_lf1(Soa d, const int *__restrict__ scal, double dt) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= scal[S_NP] || d.type[p] != TSPH_FLUID) return;
  const double om = d.omega[p], orho = d.omegarho[p];
  const double2 ov = d.omegav[p], dov = d.domegav[p];
  d.omega_o[p] = om;
  d.omegarho_o[p] = orho;
  d.omegav_o[p] = ov;
  const double om1 = om + d.domega[p] * dt * 0.5;
  const double orho1 = orho + d.domegarho[p] * dt * 0.5;
  const double2 ov1 = make_double2(ov.x + dov.x * dt * 0.5, ov.y + dov.y * dt * 0.5);
  d.omega[p] = om1;
  d.omegarho[p] = orho1;
  d.omegav[p] = ov1;
  const double rho = orho1 / (om1);
  d.rho[p] = rho;
  d.v[p] = make_double2(ov1.x / (rho * om1), ov1.y / (rho * om1));
}

// Integrate_LeapFrog_partTwo, src/RALESPH_integration.h:38-107
__global__ void k_rale_lf2(Soa d, const int *__restrict__ scal, double dt, int first) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= scal[S_NP] || d.type[p] != TSPH_FLUID) return;
  const double2 dov = d.domegav[p];
  if (first) {
    const double om = d.omega[p], orho = d.omegarho[p];
    const double2 ov = d.omegav[p];
    d.omega_o[p] = om;
    d.omegarho_o[p] = orho;
    d.omegav_o[p] = ov;
    const double om1 = om + d.domega[p] * dt * 0.5;
    const double orho1 = orho + d.domegarho[p] * dt * 0.5;
    const double2 ov1 = make_double2(ov.x + dov.x * dt * 0.5, ov.y + dov.y * dt * 0.5);
    d.omega[p] = om1;
    d.omegarho[p] = orho1;
    d.omegav[p] = ov1;
    const double rho = orho1 / (om1);
    d.rho[p] = rho;
    const double2 v = make_double2(ov1.x / (rho * om1), ov1.y / (rho * om1));
    d.v[p] = v;
    const double2 r = d.r[p];
    d.r[p] = make_double2(r.x + v.x * dt * 0.5, r.y + v.y * dt * 0.5);
  } else {
    const double2 r = d.r[p], v0 = d.v[p];
    d.r[p] = make_double2(r.x + v0.x * dt, r.y + v0.y * dt);
    const double om1 = d.omega_o[p] + d.domega[p] * dt;
    const double orho1 = d.omegarho_o[p] + d.domegarho[p] * dt;
    const double2 ovo = d.omegav_o[p];
    const double2 ov1 = make_double2(ovo.x + dov.x * dt, ovo.y + dov.y * dt);
    d.omega[p] = om1;
    d.omegarho[p] = orho1;
    d.omegav[p] = ov1;
    const double rho = orho1 / (om1);
    d.rho[p] = rho;
    d.v[p] = make_double2(ov1.x / (rho * om1), ov1.y / (rho * om1));
  }
}

}  // namespace

int launch_ale_init(tsph_ctx *c) {
  hipLaunchKernelGGL(k_ale_init, dim3(grid_for(c->n_ub, 256)), dim3(256), 0, c->stream, c->cur,
                     c->scal, c->k.dp);
  TSPH_HIP(hipGetLastError());
  return 0;
}

template <int H>
static int launch_rale_cells(tsph_ctx *c) {
  using P = RaleCell64<H>;
  constexpr int lds = cell_lds_bytes<P>();
  const Soa &d = c->cur;
  const int groups = cell_groups(c, k_rale_cells64<P>, P::kWaves, lds, c->ale_fit[7]);
  return launch_timed(c, [&] {
    hipLaunchKernelGGL(k_rale_cells64<P>, dim3(groups), dim3(P::kWaves * kWave), lds, c->stream,
                       P{{d.r, d.v, d.n, d.rho, d.omega, d.type, d.domega, d.domegarho, d.domegav,
                          c->ale_flag}, rale64(c->k)},
                       cell_grid(c->k), c->cell_start, cell_source(c), c->counters);
  });
}

int launch_rale_forces(tsph_ctx *c) {
  const Consts &k = c->k;
  const int rows = c->tile_rows;
  const int cap = 3 * (rows + 2) * kCellCap;
  hipStream_t s = c->stream;
  const size_t list = sizeof(uint16_t) * kList * kWave;
  int e = 0;
  if (c->prm.precision == TSPH_PREC_MIXED) {
    // the ALE passes stride (see launch_pass, tsph_alemuscl.hip)
    const TileGrid tg =
        tile_grid(c, true, kTabBytes + list + (size_t)cap * (4 * sizeof(float2) + 1), false);
    if ((e = ensure_tile_list(c, 0))) return e;
    e = launch_timed(c, [&] {
      hipLaunchKernelGGL(k_rale32, tg.grid, tg.block, tg.lds, s, c->cur, c->cell_start,
                           c->cellof, k, rows, c->scal, c->tile_list, cap, tg.lds_wave,
                            c->ale_flag, c->counters);
    });
  } else {
    if ((e = ensure_cell_entries(c))) return e;
    e = cells_wide(c) ? launch_rale_cells<4>(c) : launch_rale_cells<2>(c);
  }
  if (e) return e;
  hipLaunchKernelGGL(k_rale_isolated, dim3(grid_for(c->n_ub, 256)), dim3(256), 0, s, c->cur,
                     c->cell_start, c->cellof, c->scal, c->ale_flag, k);
  TSPH_HIP(hipGetLastError());
  return 0;
}

int launch_rale_leapfrog_one(tsph_ctx *c, double dt) {
  hipLaunchKernelGGL(k_rale_lf1, dim3(grid_for(c->n_ub, 256)), dim3(256), 0, c->stream, c->cur,
                     c->scal, dt);
  TSPH_HIP(hipGetLastError());
  c->records_valid = false;
  c->marks_valid = false;
  return 0;
}

int launch_rale_leapfrog_two(tsph_ctx *c, double dt, int step) {
  hipLaunchKernelGGL(k_rale_lf2, dim3(grid_for(c->n_ub, 256)), dim3(256), 0, c->stream, c->cur,
                     c->scal, dt, (int)(step == 1));
  TSPH_HIP(hipGetLastError());
  c->records_valid = false;
  c->marks_valid = false;
  return 0;
}

}  // namespace tsph
