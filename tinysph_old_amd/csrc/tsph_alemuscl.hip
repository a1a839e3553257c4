// ALE-SPH with MUSCL reconstruction: the pipeline of the ALE dam-break driver
// cases/ALESPH_dambreakLong/SPH_simulation.h:78-125,
//   Integrate_LeapFrog_partOne_ALESPH  src/ALESPH_integration.h:9-31
//   Compute_Density                    src/ALESPH_density_and_omega_bt.h:9-281
//   Kernel_gradient_approx             src/ALESPH_kernel_gradient.h:10-190
//   Integrate_density_compute_pressure src/ALESPH_integration.h:86-135
//   Compute_Acceleration_BT            src/ALESPH_acceleration_bt.h:12-295
//   Integrate_LeapFrog_partTwo_ALESPH  src/ALESPH_integration.h:33-83
//
// The three pair passes are policies: in FP64 of the cell walk of tsph_tiles.h
// (the reference's neighbour and operand order; the tile walk's 27 KB of
// records per wavefront left a compute unit four wavefronts, and each of them
// two or three tiles of 183k particles), and of its tile walk in a mixed form with FP32 fluxes on tile-frame positions and densities carried as
// deviations from rho0 (the linear EOS makes the pressure of a deviation exact).
//
// MUSCL states (src/ALESPH_riemann_solver.h:195-235): A_L = A_i + a/2 gA_i.dr,
// A_R = A_j - a/2 gA_j.dr with dr = r_i - r_j; a = 1 as the reference calls
// them, or the minmod weight of src/ALESPH_riemann_solver.h:180-191 per variable
// when limited (r_CD from the reconstructing particle to the other one; phi = 0
// where the two values are equal).
//
// Reference quirk kept: Compute_Density reads `dvdW` for fluid neighbours but
// never assigns it (src/ALESPH_density_and_omega_bt.h:135,237); the reference's
// own build evaluates that volume-flux term as zero, so only wall neighbours
// change omega in that pass.
#include <algorithm>

#include "tsph_internal.h"
#include "tsph_physics.h"
#include "tsph_tiles.h"

namespace tsph {

namespace {

using namespace tiles;

constexpr int kOutletF = 17;  // outletf, src/SPH_defs.h:44-65

// ---------------------------------------------------------------------------
// shared pieces
// ---------------------------------------------------------------------------
// constants of the FP64 passes
struct Ale64 {
  double h, ih, awen, bwen, cs, ics, cs2, ics2, rho0, irho0, m, dp, gx, gy;
};
__host__ __device__ __forceinline__ Ale64 ale64(const Consts &k) {
  return {k.h, k.ih, k.awen, k.bwen, k.cs, 1. / k.cs, k.cs * k.cs, 1. / (k.cs * k.cs), k.rho0,
          1. / k.rho0, k.m, k.dp, k.gx, k.gy};
}

// velRiemannLinearized, src/ALESPH_riemann_solver.h:86-96 (iavg: recip64(rhoAvg))
__device__ __forceinline__ double vel_riemann64(double rhoL, double rhoR, double vL, double vR,
                                                double rhoAvg, double iavg, double c) {
  return 0.5 * (vR + vL) - quot64_any(0.5 * (rhoR - rhoL) * c, rhoAvg, iavg);
}
// densRiemannLinearizedWithLimiter, src/ALESPH_riemann_solver.h:20-34 (c2 = c c, ic2 = 1/c2)
__device__ __forceinline__ double dens_riemann_lim64(double rhoL, double rhoR, double vL, double vR,
                                                     double rhoAvg, double c, double c2, double ic2) {
  const double d = vL - vR;
  const double mx = d > 0 ? d : 0;
  const double e = 3. * mx;
  const double beta = e < c ? e : c;
  return 0.5 * (rhoL + rhoR) + quot64_any(0.5 * beta * (vL - vR) * rhoAvg, c2, ic2);
}
// minmod weights of a pair's two sides for one variable
// (src/ALESPH_riemann_solver.h:161-191): r = 2 (grad.r_CD) / (aD - aC) - 1 on
// either side; the two denominators are each other's negative, so one
// reciprocal serves both.  r_CD: rij from o to b, dr back.  (A denominator so
// small that its reciprocal overflows takes the general division.)
__device__ __forceinline__ void minmod_weights64(double ao, double ab, double2 go, double2 gb,
                                                 double2 rij, double2 dr, double &po, double &pb) {
  const double d = ab - ao;
  const double no = 2. * (go.x * rij.x + go.y * rij.y), nb = 2. * (gb.x * dr.x + gb.y * dr.y);
  const double y = recip64(d);
  double qo = quot64_any(no, d, y), qb = quot64_any(nb, -d, -y);
  if (fabs(d) < 0x1p-960) {
    qo = no / d;
    qb = nb / -d;
  }
  const double ro = qo - 1., rb = qb - 1.;
  const double mo = 1. < ro ? 1. : ro, mb = 1. < rb ? 1. : rb;
  po = d == 0. ? 0. : (0. > mo ? 0. : mo);
  pb = d == 0. ? 0. : (0. > mb ? 0. : mb);
}
template <typename T, typename V>
__device__ __forceinline__ T minmod_phi(T aC, T aD, V g, V rCD) {
  if (aD - aC == T(0)) return T(0);
  const T r = T(2) * (g.x * rCD.x + g.y * rCD.y) / (aD - aC) - T(1);
  const T mn = T(1) < r ? T(1) : r;
  return T(0) > mn ? T(0) : mn;
}

// the fields the FP64 passes read and write
struct AlePtr {
  const double2 *r, *v, *n;
  const double *rho, *omega;
  const uint8_t *type;
  double2 *gradrho, *gradvx, *gradvy;
  double *domega, *domegarho;
  double2 *domegav;
};

// one particle of the FP64 passes (own or neighbour; G: with its gradients)
template <bool G>
struct P64;
template <>
struct P64<false> {
  double2 r, v, n;
  double rho, omega;
  int t;
};
template <>
struct P64<true> : P64<false> {
  double2 gr, gx, gy;
};

// a pair's geometry: dr = r_i - r_j, its length, the kernel (0 beyond the
// exact support) and whether the pair is inside it (qq <= 2)
struct Geo64 {
  double2 dr;
  Root64 rt;
  KW64 kw;
  bool in, some;  // some: the kernel is not 0 (qq < 2)
};
__device__ __forceinline__ Geo64 geometry64(const Ale64 &k, double2 a, double2 b) {
  Geo64 g;
  g.dr = make_double2(a.x - b.x, a.y - b.y);
  g.rt = sqrt64((g.dr.x * g.dr.x) + (g.dr.y * g.dr.y));
  const double qq = quot64(g.rt.s, k.h, k.ih);
  g.in = qq <= 2.0;
  g.some = qq < 2.0;
  g.kw = wendland64(g.rt, qq, k.awen, k.bwen);
  return g;
}

// reconstructed left/right states (FP64, reference operand order)
struct LR64 {
  double rhoL, rhoR;
  double2 vL, vR;
};
template <bool LIM>
__device__ __forceinline__ LR64 states64(const P64<false> &o, const P64<false> &b, double2) {
  return {o.rho, b.rho, o.v, b.v};
}
template <bool LIM>
__device__ __forceinline__ LR64 states64(const P64<true> &o, const P64<true> &b, double2 dr) {
  LR64 s;
  double a1 = 1, a2 = 1, a3 = 1, a4 = 1, a5 = 1, a6 = 1;
  if (LIM) {
    const double2 rij = make_double2(0. - dr.x, 0. - dr.y);
    minmod_weights64(o.rho, b.rho, o.gr, b.gr, rij, dr, a1, a2);
    minmod_weights64(o.v.x, b.v.x, o.gx, b.gx, rij, dr, a3, a5);
    minmod_weights64(o.v.y, b.v.y, o.gy, b.gy, rij, dr, a4, a6);
  }
  s.rhoL = o.rho + a1 * 0.5 * (o.gr.x * dr.x + o.gr.y * dr.y);
  s.rhoR = b.rho - a2 * 0.5 * (b.gr.x * dr.x + b.gr.y * dr.y);
  s.vL.x = o.v.x + a3 * 0.5 * (o.gx.x * dr.x + o.gx.y * dr.y);
  s.vL.y = o.v.y + a4 * 0.5 * (o.gy.x * dr.x + o.gy.y * dr.y);
  s.vR.x = b.v.x - a5 * 0.5 * (b.gx.x * dr.x + b.gx.y * dr.y);
  s.vR.y = b.v.y - a6 * 0.5 * (b.gy.x * dr.x + b.gy.y * dr.y);
  return s;
}

// ---------------------------------------------------------------------------
// FP64 passes: policies of the cell walk (cells64, tsph_tiles.h).  The
// reference's gamma sum is only compared with zero; its terms W m / rho are
// zero exactly where W is (qq = 2) or rho is infinite, so a flag stands for it.
// ---------------------------------------------------------------------------
// Kernel_gradient_approx (fluid only): gradients of rho, vx, vy
struct Grad64 {
  static constexpr bool kG = false, kSound = false;
  static constexpr int kSums = 6;
  static __device__ __forceinline__ bool active(int t) { return t == TSPH_FLUID; }
  static __device__ __forceinline__ void pair(const Ale64 &k, const P64<false> &o, const P64<false> &b,
                                              const Geo64 &g, double, double, double (&s)[kSums]) {
    const double W = g.kw.w;
    const double dWx = g.dr.x * g.kw.f, dWy = g.dr.y * g.kw.f;
    const double drho = b.rho - o.rho, dvx = b.v.x - o.v.x, dvy = b.v.y - o.v.y;
    if (b.t == TSPH_WALL) {
      const double nbx = b.n.x * (-1), nby = b.n.y * (-1);
      s[0] = drho * nbx * W * k.dp;
      s[1] = drho * nby * W * k.dp;
      s[2] = dvx * nbx * W * k.dp;
      s[3] = dvx * nby * W * k.dp;
      s[4] = dvy * nbx * W * k.dp;
      s[5] = dvy * nby * W * k.dp;
    } else {
      s[0] = drho * b.omega * dWx;
      s[1] = drho * b.omega * dWy;
      s[2] = dvx * b.omega * dWx;
      s[3] = dvx * b.omega * dWy;
      s[4] = dvy * b.omega * dWx;
      s[5] = dvy * b.omega * dWy;
    }
  }
  static __device__ __forceinline__ void write(const Ale64 &, const AlePtr &d, const P64<false> &, int i,
                                               const double (&s)[kSums], bool some) {
    double2 gr = make_double2(0., 0.), gx = gr, gy = gr;
    if (some) {
      gr = make_double2(s[0] * 2., s[1] * 2.);
      gx = make_double2(s[2] * 2., s[3] * 2.);
      gy = make_double2(s[4] * 2., s[5] * 2.);
    }
    d.gradrho[i] = gr;
    d.gradvx[i] = gx;
    d.gradvy[i] = gy;
  }
};

// Compute_Density: d(omega), d(omega rho)
template <bool G, bool LIM>
struct Dens64 {
  static constexpr bool kG = G, kSound = false;
  static constexpr int kSums = 2;
  static __device__ __forceinline__ bool active(int t) {
    return t != kOutletF && t != TSPH_OUTLET && t != TSPH_INLET && t != TSPH_WALL && t != kRemoved;
  }
  static __device__ __forceinline__ void pair(const Ale64 &k, const P64<G> &o, const P64<G> &b,
                                              const Geo64 &g, double, double, double (&t)[kSums]) {
    const double2 dr = g.dr;
    const double dvx = o.v.x - b.v.x, dvy = o.v.y - b.v.y;
    const double inv = quot64(1., g.rt.s, recip_of_root64(g.rt));
    const double drnx = dr.x * inv * (-1), drny = dr.y * inv * (-1);
    const double W = g.kw.w;
    const double dWx = dr.x * g.kw.f, dWy = dr.y * g.kw.f;
    const LR64 s = states64<LIM>(o, b, dr);
    const double vl = s.vL.x * drnx + s.vL.y * drny;
    const double vr = s.vR.x * drnx + s.vR.y * drny;
    const double avg = 0.5 * (s.rhoL + s.rhoR);
    const double rhos = dens_riemann_lim64(s.rhoL, s.rhoR, vl, vr, avg, k.cs, k.cs2, k.ics2);
    const double vss = vel_riemann64(s.rhoL, s.rhoR, vl, vr, avg, recip64(avg), k.cs);
    const double vsx = drnx * vss + ((o.v.x + b.v.x) * 0.5 - drnx * (vl + vr) * 0.5);
    const double vsy = drny * vss + ((o.v.y + b.v.y) * 0.5 - drny * (vl + vr) * 0.5);
    const double vsdW = (vsx - o.v.x) * dWx + (vsy - o.v.y) * dWy;
    const bool wall = b.t == TSPH_WALL;
    const double nbx = b.n.x * (-1), nby = b.n.y * (-1);
    const double dvn = dvx * nbx + dvy * nby;
    // the fluid volume flux term is zero as the reference build evaluates it
    t[0] = wall ? 0. - dvn * W * k.dp : 0.;
    t[1] = wall ? 0. : 0. - 2 * rhos * b.omega * vsdW;
  }
  static __device__ __forceinline__ void write(const Ale64 &, const AlePtr &d, const P64<false> &o, int i,
                                               const double (&s)[kSums], bool some) {
    d.domega[i] = some ? s[0] * o.omega : 0.;
    d.domegarho[i] = some ? s[1] * o.omega : 0.;
  }
};

// Compute_Acceleration_BT: d(omega v)
template <bool G, bool LIM>
struct Acc64P {
  static constexpr bool kG = G, kSound = true;
  static constexpr int kSums = 2;
  static __device__ __forceinline__ bool active(int t) { return t == TSPH_FLUID; }
  // co, cb: the particles' sound speeds c0 (rho/rho0)^(1/2)
  // (src/ALESPH_riemann_solver.h:148-159), summed (:178)
  static __device__ __forceinline__ void pair(const Ale64 &k, const P64<G> &o, const P64<G> &b,
                                              const Geo64 &g, double co, double cb,
                                              double (&t)[kSums]) {
    const double c0 = k.cs, rho0 = k.rho0;
    const double2 dr = g.dr;
    const double inv = quot64(1., g.rt.s, recip_of_root64(g.rt));
    const double drnx = dr.x * inv * (-1), drny = dr.y * inv * (-1);
    const double W = g.kw.w;
    const double dWx = dr.x * g.kw.f, dWy = dr.y * g.kw.f;
    const LR64 s = states64<LIM>(o, b, dr);
    const double vl = s.vL.x * drnx + s.vL.y * drny;
    const double vr = s.vR.x * drnx + s.vR.y * drny;
    const double avgc = co + cb, c2 = avgc * avgc;
    const double avg = 0.5 * (s.rhoL + s.rhoR);
    const double rhos = dens_riemann_lim64(s.rhoL, s.rhoR, vl, vr, avg, avgc, c2, recip64(c2));
    const double vss = vel_riemann64(o.rho, b.rho, vl, vr, avg, recip64(avg), avgc);
    const double vsx = drnx * vss + ((o.v.x + b.v.x) * 0.5 - drnx * (vl + vr) * 0.5);
    const double vsy = drny * vss + ((o.v.y + b.v.y) * 0.5 - drny * (vl + vr) * 0.5);
    if (b.t == TSPH_WALL) {
      const double nbx = b.n.x * (-1), nby = b.n.y * (-1);
      const double rw = s.rhoL - quot64_any(((0 - s.vL.x) * nbx + (0 - s.vL.y) * nby) * s.rhoL, c0, k.ics);
      const double pw = c0 * c0 * (rw - 1000.) * 1;
      t[0] = 0. - 2 * W * k.dp * (pw * nbx);
      t[1] = 0. - 2 * W * k.dp * (pw * nby);
    } else {
      const double ps = c0 * c0 * (rhos - rho0);
      t[0] = 0. - 2 * b.omega * ((rhos * vsx * (vsx - o.v.x) + ps) * dWx + (rhos * vsx * (vsy - o.v.y)) * dWy);
      t[1] = 0. - 2 * b.omega * ((rhos * vsy * (vsx - o.v.x)) * dWx + (rhos * vsy * (vsy - o.v.y) + ps) * dWy);
    }
  }
  static __device__ __forceinline__ void write(const Ale64 &k, const AlePtr &d, const P64<false> &o, int i,
                                               const double (&s)[kSums], bool some) {
    const double gx = k.gx * o.omega * o.rho, gy = k.gy * o.omega * o.rho;
    d.domegav[i] = some ? make_double2(s[0] * o.omega - gx, s[1] * o.omega - gy)
                        : make_double2(0. - gx, 0. - gy);
  }
};

// the cell walk's policy of pass A
template <class A, int H>
struct AleCell64 {
  AlePtr d;
  Ale64 k;
  static constexpr bool G = A::kG;
  static constexpr int kSums = A::kSums;
  static constexpr int kSlotBytes = (G ? 7 : 4) * 16 + (A::kSound ? 8 : 0) + 1;
  static constexpr int kWaves = (G ? 2 : 4) / (H / 2);
  static constexpr int kSlots = cell_slots_of<H>();
  static constexpr bool kFlag = true, kSkip = false;
  struct Lds {
    double2 *r, *v, *ro, *n, *gr, *gx, *gy;  // ro = {rho, omega}
    double *cs;
    uint8_t *t;
  };
  using Rec = P64<G>;
  static __device__ __forceinline__ Lds lds(unsigned char *b, int cap) {
    double2 *p = reinterpret_cast<double2 *>(b);
    Lds L;
    L.r = p; L.v = p + cap; L.ro = p + 2 * cap; L.n = p + 3 * cap;
    L.gr = p + 4 * cap; L.gx = p + 5 * cap; L.gy = p + 6 * cap;
    L.cs = reinterpret_cast<double *>(p + (G ? 7 : 4) * cap);
    L.t = reinterpret_cast<uint8_t *>(L.cs + (A::kSound ? cap : 0));
    return L;
  }
  __device__ __forceinline__ void set(const Consts &) {}  // (no batched ALE contexts)
  __device__ __forceinline__ Rec load(int j) const {
    Rec q;
    q.r = d.r[j];
    q.v = d.v[j];
    q.rho = d.rho[j];
    q.omega = d.omega[j];
    q.n = d.n ? d.n[j] : make_double2(0., 0.);
    q.t = d.type[j];
    if constexpr (G) {
      q.gr = d.gradrho[j];
      q.gx = d.gradvx[j];
      q.gy = d.gradvy[j];
    }
    return q;
  }
  __device__ __forceinline__ double sound(double rho) const {
    return A::kSound ? k.cs * sqrt(quot64_any(rho, k.rho0, k.irho0)) : 0.;
  }
  __device__ __forceinline__ void store(const Lds &L, int l, const Rec &q) const {
    L.r[l] = q.r;
    L.v[l] = q.v;
    L.ro[l] = make_double2(q.rho, q.omega);
    L.n[l] = q.n;
    L.t[l] = (uint8_t)q.t;
    if (A::kSound) L.cs[l] = sound(q.rho);
    if constexpr (G) {
      L.gr[l] = q.gr;
      L.gx[l] = q.gx;
      L.gy[l] = q.gy;
    }
  }
  static __device__ __forceinline__ Rec slot(const Lds &L, int l) {
    Rec q;
    q.r = L.r[l];
    q.v = L.v[l];
    q.n = L.n[l];
    const double2 ro = L.ro[l];
    q.rho = ro.x;
    q.omega = ro.y;
    q.t = L.t[l];
    if constexpr (G) {
      q.gr = L.gr[l];
      q.gx = L.gx[l];
      q.gy = L.gy[l];
    }
    return q;
  }
  __device__ __forceinline__ bool act_lds(const Lds &L, int l) const { return A::active(L.t[l]); }
  __device__ __forceinline__ bool skip_lds(const Lds &, int) const { return false; }
  __device__ __forceinline__ double2 pos_lds(const Lds &L, int l) const { return L.r[l]; }
  // the terms; bit 0: inside the support, bit 1: its gamma term is not 0
  __device__ __forceinline__ int pair(const Rec &o, const Rec &b, double co, double cb,
                                      double (&t)[kSums]) const {
    const Geo64 g = geometry64(k, o.r, b.r);
    A::pair(k, o, b, g, co, cb, t);
    if (!g.in) {
#pragma unroll
      for (int q = 0; q < kSums; ++q) t[q] = 0.;
    }
    return (int)g.in | ((int)(g.some & (fabs(b.rho) != INFINITY)) << 1);
  }
  __device__ __forceinline__ int terms(const Lds &L, int p, int l, double (&t)[kSums]) const {
    return pair(slot(L, p), slot(L, l), A::kSound ? L.cs[p] : 0., A::kSound ? L.cs[l] : 0., t);
  }
  __device__ __forceinline__ void sums(const Lds &L, int p, int i, const double (&s)[kSums],
                                       bool some) const {
    A::write(k, d, slot(L, p), i, s, some);
  }
  __device__ __forceinline__ void far(int i, const int *cs, const CellGrid &g, int c, unsigned &npair,
                                      unsigned &ncand, unsigned &nact) const {
    const Rec o = load(i);
    if (!A::active(o.t)) return;
    ++nact;
    const int cx = c / g.ncy, cy = c - cx * g.ncy;
    double s[kSums];
#pragma unroll
    for (int q = 0; q < kSums; ++q) s[q] = 0.;
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
        const int got = pair(o, b, sound(o.rho), sound(b.rho), t);
        npair += got & 1;
        some |= (got & 2) != 0;
#pragma unroll
        for (int u = 0; u < kSums; ++u) s[u] += t[u];
      }
    }
    A::write(k, d, o, i, s, some);
  }
};

// ---------------------------------------------------------------------------
// mixed passes: FP32 fluxes, tile-frame positions, densities as rho - rho0
// ---------------------------------------------------------------------------
template <bool G>
struct Lds32 {
  float2 *p, *v, *dw, *n, *gr, *gx, *gy;  // dw = {rho - rho0, omega}
  uint8_t *t;
};
template <bool G>
__device__ __forceinline__ Lds32<G> carve32(unsigned char *b, int cap) {
  float2 *p = reinterpret_cast<float2 *>(b);
  Lds32<G> L;
  L.p = p; L.v = p + cap; L.dw = p + 2 * cap; L.n = p + 3 * cap;
  L.gr = G ? p + 4 * cap : nullptr;
  L.gx = G ? p + 5 * cap : nullptr;
  L.gy = G ? p + 6 * cap : nullptr;
  L.t = reinterpret_cast<uint8_t *>(p + (G ? 7 : 4) * cap);
  return L;
}
template <bool G>
constexpr int slot_bytes32() { return (G ? 7 : 4) * 8 + 1; }

__device__ __forceinline__ float2 f2(double2 a) { return make_float2((float)a.x, (float)a.y); }

struct Nb32 {
  float2 v, n, gr, gx, gy;
  float dev, omega;
  int t;
};
template <bool G>
__device__ __forceinline__ void stage32(const Soa &d, const Consts &k, const Lds32<G> &L, int l, int j,
                                        double ox, double oy) {
  const double2 r = d.r[j];
  L.p[l] = make_float2((float)(r.x - ox), (float)(r.y - oy));
  L.v[l] = f2(d.v[j]);
  L.dw[l] = make_float2((float)(d.rho[j] - k.rho0), (float)d.omega[j]);
  L.n[l] = d.n ? f2(d.n[j]) : make_float2(0.f, 0.f);
  L.t[l] = d.type[j];
  if (G) {
    L.gr[l] = f2(d.gradrho[j]);
    L.gx[l] = f2(d.gradvx[j]);
    L.gy[l] = f2(d.gradvy[j]);
  }
}
template <bool G>
__device__ __forceinline__ Nb32 nb_lds32(const Lds32<G> &L, int l) {
  Nb32 b;
  b.v = L.v[l]; b.n = L.n[l];
  const float2 dw = L.dw[l];
  b.dev = dw.x; b.omega = dw.y; b.t = L.t[l];
  if (G) { b.gr = L.gr[l]; b.gx = L.gx[l]; b.gy = L.gy[l]; }
  return b;
}
template <bool G>
__device__ __forceinline__ Nb32 nb_glob32(const Soa &d, const Consts &k, int j) {
  Nb32 b;
  b.v = f2(d.v[j]);
  b.n = d.n ? f2(d.n[j]) : make_float2(0.f, 0.f);
  b.dev = (float)(d.rho[j] - k.rho0); b.omega = (float)d.omega[j]; b.t = d.type[j];
  if (G) { b.gr = f2(d.gradrho[j]); b.gx = f2(d.gradvx[j]); b.gy = f2(d.gradvy[j]); }
  return b;
}

struct Own32 {
  float2 p, v, gr, gx, gy;
  float dev;
  double rho, omega;
};
template <bool G>
__device__ __forceinline__ Own32 own32(const Soa &d, const Consts &k, int i, double ox, double oy) {
  Own32 o;
  if (i >= 0) {
    const double2 r = d.r[i];
    o.p = make_float2((float)(r.x - ox), (float)(r.y - oy));
    o.v = f2(d.v[i]);
    o.rho = d.rho[i];
    o.omega = d.omega[i];
    o.dev = (float)(o.rho - k.rho0);
    if (G) { o.gr = f2(d.gradrho[i]); o.gx = f2(d.gradvx[i]); o.gy = f2(d.gradvy[i]); }
  } else {
    o.p = o.v = make_float2(0.f, 0.f);
    o.rho = 1.; o.omega = 0.; o.dev = 0.f;
    o.gr = o.gx = o.gy = make_float2(0.f, 0.f);
  }
  return o;
}

struct C32A {
  float ih, m, c0, ic0, rho0, dp, awen, bwen, pw0;
};
__host__ __device__ __forceinline__ C32A make_c32a(const Consts &k) {
  C32A c;
  c.ih = (float)(1. / k.h); c.m = (float)k.m; c.c0 = (float)k.cs; c.ic0 = (float)(1. / k.cs);
  c.rho0 = (float)k.rho0; c.dp = (float)k.dp; c.awen = (float)k.awen; c.bwen = (float)k.bwen;
  c.pw0 = (float)(k.rho0 - 1000.);  // the wall pressure is taken against 1000 (:242)
  return c;
}

struct KW32 {
  float w, f, inv;
};
__device__ __forceinline__ KW32 wendland32(const C32A &c, float r2) {
#pragma clang fp contract(fast)
  const float drs = __builtin_amdgcn_sqrtf(r2);
  const float qq = drs * c.ih;
  const float wq1 = 1.f - 0.5f * qq;
  const float wq2 = wq1 * wq1;
  KW32 k;
  k.w = c.awen * (qq + qq + 1.f) * wq2 * wq2;
  k.f = c.bwen * wq2 * wq1 * c.ih;
  k.inv = __builtin_amdgcn_rcpf(drs);
  return k;
}

// reconstructed states as deviations (rho - rho0) and velocities
struct LR32 {
  float aL, nR;
  float2 vL, vR;
};
template <bool G, bool LIM>
__device__ __forceinline__ LR32 states32(const Own32 &o, const Nb32 &b, float drx, float dry) {
#pragma clang fp contract(fast)
  LR32 s;
  if (!G) {
    s.aL = o.dev; s.nR = b.dev; s.vL = o.v; s.vR = b.v;
    return s;
  }
  float a1 = 1.f, a2 = 1.f, a3 = 1.f, a4 = 1.f, a5 = 1.f, a6 = 1.f;
  const float2 dr = make_float2(drx, dry), rij = make_float2(-drx, -dry);
  if (LIM) {
    a1 = minmod_phi(o.dev, b.dev, o.gr, rij);
    a2 = minmod_phi(b.dev, o.dev, b.gr, dr);
    a3 = minmod_phi(o.v.x, b.v.x, o.gx, rij);
    a4 = minmod_phi(o.v.y, b.v.y, o.gy, rij);
    a5 = minmod_phi(b.v.x, o.v.x, b.gx, dr);
    a6 = minmod_phi(b.v.y, o.v.y, b.gy, dr);
  }
  s.aL = o.dev + a1 * 0.5f * (o.gr.x * drx + o.gr.y * dry);
  s.nR = b.dev - a2 * 0.5f * (b.gr.x * drx + b.gr.y * dry);
  s.vL.x = o.v.x + a3 * 0.5f * (o.gx.x * drx + o.gx.y * dry);
  s.vL.y = o.v.y + a4 * 0.5f * (o.gy.x * drx + o.gy.y * dry);
  s.vR.x = b.v.x - a5 * 0.5f * (b.gx.x * drx + b.gx.y * dry);
  s.vR.y = b.v.y - a6 * 0.5f * (b.gy.x * drx + b.gy.y * dry);
  return s;
}

struct Grad32 {
  Soa d;
  Consts k;
  C32A c;
  using Lds = Lds32<false>;
  using Own = Own32;
  struct Acc {
    float grx = 0, gry = 0, gxx = 0, gxy = 0, gyx = 0, gyy = 0, gamma = 0;
  };
  static __device__ Lds lds(unsigned char *b, int cap) { return carve32<false>(b, cap); }
  __device__ void stage(const Lds &L, int l, int j, double ox, double oy) const { stage32<false>(d, k, L, l, j, ox, oy); }
  __device__ bool active(int i) const { return d.type[i] == TSPH_FLUID; }
  __device__ Own own(int i, double ox, double oy) const { return own32<false>(d, k, i, ox, oy); }
  __device__ float2 pos_lds(const Lds &L, int l) const { return L.p[l]; }
  __device__ float2 pos_glob(int j, double ox, double oy) const {
    const double2 r = d.r[j];
    return make_float2((float)(r.x - ox), (float)(r.y - oy));
  }
  __device__ void pair(Acc &a, const Own &o, const Nb32 &b, float drx, float dry, float r2) const {
#pragma clang fp contract(fast)
    const KW32 kw = wendland32(c, r2);
    const float dWx = drx * kw.f, dWy = dry * kw.f;
    const float drho = b.dev - o.dev, dvx = b.v.x - o.v.x, dvy = b.v.y - o.v.y;
    if (b.t == TSPH_WALL) {
      const float s = kw.w * c.dp;
      a.grx -= drho * b.n.x * s;
      a.gry -= drho * b.n.y * s;
      a.gxx -= dvx * b.n.x * s;
      a.gxy -= dvx * b.n.y * s;
      a.gyx -= dvy * b.n.x * s;
      a.gyy -= dvy * b.n.y * s;
    } else {
      a.grx += drho * b.omega * dWx;
      a.gry += drho * b.omega * dWy;
      a.gxx += dvx * b.omega * dWx;
      a.gxy += dvx * b.omega * dWy;
      a.gyx += dvy * b.omega * dWx;
      a.gyy += dvy * b.omega * dWy;
    }
    a.gamma += kw.w * c.m * __builtin_amdgcn_rcpf(c.rho0 + b.dev);
  }
  __device__ void pair_lds(Acc &a, const Own &o, const Lds &L, int l, float drx, float dry, float r2) const {
    pair(a, o, nb_lds32<false>(L, l), drx, dry, r2);
  }
  __device__ void pair_glob(Acc &a, const Own &o, int j, float drx, float dry, float r2) const {
    pair(a, o, nb_glob32<false>(d, k, j), drx, dry, r2);
  }
  __device__ void finish(const Acc &a, const Own &, int i) const {
    if (a.gamma == 0.f) {
      d.gradrho[i] = d.gradvx[i] = d.gradvy[i] = make_double2(0., 0.);
    } else {
      d.gradrho[i] = make_double2(2. * a.grx, 2. * a.gry);
      d.gradvx[i] = make_double2(2. * a.gxx, 2. * a.gxy);
      d.gradvy[i] = make_double2(2. * a.gyx, 2. * a.gyy);
    }
  }
};

template <bool G, bool LIM>
struct Dens32 {
  Soa d;
  Consts k;
  C32A c;
  using Lds = Lds32<G>;
  using Own = Own32;
  struct Acc {
    float dom = 0, domrho = 0, gamma = 0;
  };
  static __device__ Lds lds(unsigned char *b, int cap) { return carve32<G>(b, cap); }
  __device__ void stage(const Lds &L, int l, int j, double ox, double oy) const { stage32<G>(d, k, L, l, j, ox, oy); }
  __device__ bool active(int i) const {
    const int t = d.type[i];
    return t != kOutletF && t != TSPH_OUTLET && t != TSPH_INLET && t != TSPH_WALL && t != kRemoved;
  }
  __device__ Own own(int i, double ox, double oy) const { return own32<G>(d, k, i, ox, oy); }
  __device__ float2 pos_lds(const Lds &L, int l) const { return L.p[l]; }
  __device__ float2 pos_glob(int j, double ox, double oy) const {
    const double2 r = d.r[j];
    return make_float2((float)(r.x - ox), (float)(r.y - oy));
  }
  __device__ void pair(Acc &a, const Own &o, const Nb32 &b, float drx, float dry, float r2) const {
#pragma clang fp contract(fast)
    const KW32 kw = wendland32(c, r2);
    const float dWx = drx * kw.f, dWy = dry * kw.f;
    const float drnx = -drx * kw.inv, drny = -dry * kw.inv;
    const LR32 s = states32<G, LIM>(o, b, drx, dry);
    const float vl = s.vL.x * drnx + s.vL.y * drny;
    const float vr = s.vR.x * drnx + s.vR.y * drny;
    const float avg = c.rho0 + 0.5f * (s.aL + s.nR);
    const float dd = vl - vr;
    const float beta = fminf(3.f * fmaxf(dd, 0.f), c.c0);
    const float rsdev = 0.5f * (s.aL + s.nR) + 0.5f * beta * dd * avg * (c.ic0 * c.ic0);
    const float vss = 0.5f * (vr + vl) - 0.5f * (s.nR - s.aL) * c.c0 * __builtin_amdgcn_rcpf(avg);
    const float vsx = drnx * vss + (0.5f * (o.v.x + b.v.x) - 0.5f * drnx * (vl + vr));
    const float vsy = drny * vss + (0.5f * (o.v.y + b.v.y) - 0.5f * drny * (vl + vr));
    if (b.t == TSPH_WALL) {
      const float dvn = -((o.v.x - b.v.x) * b.n.x + (o.v.y - b.v.y) * b.n.y);
      a.dom -= dvn * kw.w * c.dp;
    } else {
      const float vsdW = (vsx - o.v.x) * dWx + (vsy - o.v.y) * dWy;
      a.domrho -= 2.f * (c.rho0 + rsdev) * b.omega * vsdW;
    }
    a.gamma += kw.w * c.m * __builtin_amdgcn_rcpf(c.rho0 + b.dev);
  }
  __device__ void pair_lds(Acc &a, const Own &o, const Lds &L, int l, float drx, float dry, float r2) const {
    pair(a, o, nb_lds32<G>(L, l), drx, dry, r2);
  }
  __device__ void pair_glob(Acc &a, const Own &o, int j, float drx, float dry, float r2) const {
    pair(a, o, nb_glob32<G>(d, k, j), drx, dry, r2);
  }
  __device__ void finish(const Acc &a, const Own &o, int i) const {
    if (a.gamma == 0.f) {
      d.domega[i] = 0.;
      d.domegarho[i] = 0.;
    } else {
      d.domega[i] = (double)a.dom * o.omega;
      d.domegarho[i] = (double)a.domrho * o.omega;
    }
  }
};

template <bool G, bool LIM>
struct Acc32P {
  Soa d;
  Consts k;
  C32A c;
  using Lds = Lds32<G>;
  using Own = Own32;
  struct Acc {
    float ax = 0, ay = 0, gamma = 0;
  };
  static __device__ Lds lds(unsigned char *b, int cap) { return carve32<G>(b, cap); }
  __device__ void stage(const Lds &L, int l, int j, double ox, double oy) const { stage32<G>(d, k, L, l, j, ox, oy); }
  __device__ bool active(int i) const { return d.type[i] == TSPH_FLUID; }
  __device__ Own own(int i, double ox, double oy) const { return own32<G>(d, k, i, ox, oy); }
  __device__ float2 pos_lds(const Lds &L, int l) const { return L.p[l]; }
  __device__ float2 pos_glob(int j, double ox, double oy) const {
    const double2 r = d.r[j];
    return make_float2((float)(r.x - ox), (float)(r.y - oy));
  }
  __device__ void pair(Acc &a, const Own &o, const Nb32 &b, float drx, float dry, float r2) const {
#pragma clang fp contract(fast)
    const KW32 kw = wendland32(c, r2);
    const float dWx = drx * kw.f, dWy = dry * kw.f;
    const float drnx = -drx * kw.inv, drny = -dry * kw.inv;
    const LR32 s = states32<G, LIM>(o, b, drx, dry);
    const float vl = s.vL.x * drnx + s.vL.y * drny;
    const float vr = s.vR.x * drnx + s.vR.y * drny;
    const float ir0 = 1.f / c.rho0;
    const float avgc = c.c0 * (__builtin_amdgcn_sqrtf(1.f + o.dev * ir0) + __builtin_amdgcn_sqrtf(1.f + b.dev * ir0));
    const float avg = c.rho0 + 0.5f * (s.aL + s.nR);
    const float dd = vl - vr;
    const float beta = fminf(3.f * fmaxf(dd, 0.f), avgc);
    const float rsdev = 0.5f * (s.aL + s.nR) + 0.5f * beta * dd * avg * __builtin_amdgcn_rcpf(avgc * avgc);
    const float vss = 0.5f * (vr + vl) - 0.5f * (b.dev - o.dev) * avgc * __builtin_amdgcn_rcpf(avg);
    const float vsx = drnx * vss + (0.5f * (o.v.x + b.v.x) - 0.5f * drnx * (vl + vr));
    const float vsy = drny * vss + (0.5f * (o.v.y + b.v.y) - 0.5f * drny * (vl + vr));
    if (b.t == TSPH_WALL) {
      const float nbx = -b.n.x, nby = -b.n.y;
      // wall state rho_w - rho0 = aL + (vL . nb) (rho0 + aL) / c0
      const float rwdev = s.aL + (s.vL.x * nbx + s.vL.y * nby) * (c.rho0 + s.aL) * c.ic0;
      const float pw = c.c0 * c.c0 * (c.pw0 + rwdev);
      a.ax -= 2.f * kw.w * c.dp * (pw * nbx);
      a.ay -= 2.f * kw.w * c.dp * (pw * nby);
    } else {
      const float ps = c.c0 * c.c0 * rsdev;
      const float rhos = c.rho0 + rsdev;
      const float ex = vsx - o.v.x, ey = vsy - o.v.y;
      a.ax -= 2.f * b.omega * ((rhos * vsx * ex + ps) * dWx + (rhos * vsx * ey) * dWy);
      a.ay -= 2.f * b.omega * ((rhos * vsy * ex) * dWx + (rhos * vsy * ey + ps) * dWy);
    }
    a.gamma += kw.w * c.m * __builtin_amdgcn_rcpf(c.rho0 + b.dev);
  }
  __device__ void pair_lds(Acc &a, const Own &o, const Lds &L, int l, float drx, float dry, float r2) const {
    pair(a, o, nb_lds32<G>(L, l), drx, dry, r2);
  }
  __device__ void pair_glob(Acc &a, const Own &o, int j, float drx, float dry, float r2) const {
    pair(a, o, nb_glob32<G>(d, k, j), drx, dry, r2);
  }
  __device__ void finish(const Acc &a, const Own &o, int i) const {
    const double gx = k.gx * o.omega * o.rho, gy = k.gy * o.omega * o.rho;
    if (a.gamma == 0.f)
      d.domegav[i] = make_double2(0. - gx, 0. - gy);
    else
      d.domegav[i] = make_double2((double)a.ax * o.omega - gx, (double)a.ay * o.omega - gy);
  }
};

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
template <class P>
__global__ __launch_bounds__(P::kWaves * kWave, 2) void k_ale_cells64(
    P pol, CellGrid g, const int *__restrict__ cell_start, CellSource src,
    unsigned long long *__restrict__ counters) {
  cells64(pol, g, cell_start, nullptr, 1, src, counters);
}

template <class P>
__global__ __launch_bounds__(kWave * kPoolWaves) void k_ale_pass32(P pol, const int *__restrict__ cell_start,
                                                      const int *__restrict__ cellof, int rows,
                                                      int *__restrict__ scal,
                                                      const int *__restrict__ tile_list,
                                                      int cap, int lds_wave,
                                                      unsigned long long *__restrict__ counters) {
  walk32(pol, pol.k, cell_start, cellof, rows, scal, tile_list, cap, lds_wave, counters);
}

// Integrate_density_compute_pressure, src/ALESPH_integration.h:86-135 (fluid
// only; linear EOS src/SPH_pressure.h:24-34, pressure clamped at zero)
__global__ void k_ale_density_pressure(Soa d, const int *__restrict__ scal, Consts k, double dt,
                                       unsigned long long *__restrict__ counters) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= scal[S_NP] || d.type[p] != TSPH_FLUID) return;
  const double om = d.omega[p] + d.domega[p] * dt;
  const double orho = d.omegarho[p] + d.domegarho[p] * dt;
  d.omega[p] = om;
  d.omegarho[p] = orho;
  const double rho = orho / (om);
  d.rho[p] = rho;
  if (rho > 1500. || rho < 0.) atomicAdd(&counters[C_BADRHO], 1ull);
  double pr = k.cs * k.cs * (rho - k.rho0);
  if (pr < 0) pr = 0;
  d.p[p] = pr;
}

// Integrate_LeapFrog_partOne_ALESPH, src/ALESPH_integration.h:9-31
__global__ void k_ale_lf1(Soa d, const int *__restrict__ scal, double dt) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= scal[S_NP] || d.type[p] != TSPH_FLUID) return;
  const double2 ov = d.omegav[p], dov = d.domegav[p];
  const double2 ov1 = make_double2(ov.x + dov.x * dt * 0.5, ov.y + dov.y * dt * 0.5);
  d.omegav[p] = ov1;
  const double ro = d.rho[p] * d.omega[p];
  d.v[p] = make_double2(ov1.x / ro, ov1.y / ro);
}

// Integrate_LeapFrog_partTwo_ALESPH, src/ALESPH_integration.h:33-83
__global__ void k_ale_lf2(Soa d, const int *__restrict__ scal, double dt, int first) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= scal[S_NP] || d.type[p] != TSPH_FLUID) return;
  const double2 ov = d.omegav[p], dov = d.domegav[p];
  const double ro = d.rho[p] * d.omega[p];
  const double2 r = d.r[p];
  if (first) {
    const double2 ov1 = make_double2(ov.x + dov.x * dt * 0.5, ov.y + dov.y * dt * 0.5);
    d.omegav[p] = ov1;
    const double2 v = make_double2(ov1.x / ro, ov1.y / ro);
    d.v[p] = v;
    d.r[p] = make_double2(r.x + v.x * dt * 0.5, r.y + v.y * dt * 0.5);
  } else {
    const double2 ov1 = make_double2(ov.x + dov.x * dt, ov.y + dov.y * dt);
    d.omegav[p] = ov1;
    const double2 v = make_double2(ov1.x / ro, ov1.y / ro);
    d.v[p] = v;
    d.r[p] = make_double2(r.x + v.x * dt, r.y + v.y * dt);
  }
}

// launch of one mixed pair pass on the persistent tile grid
template <class P, int SLOT>
int launch_pass32(tsph_ctx *c, const P &pol) {
  const int rows = c->tile_rows;
  // Slots per tile.  The ALE records are large (57 B with the MUSCL gradients)
  // and the waves that a compute unit holds pay, so the budget is at least
  // kAleCellCap records per cell (the lattice's), and beyond that what the waves
  // leave over that it holds at once: those that fit with kAleCellCap records, no
  // more than the launch has, and no more than the system has tiles for; up to
  // kCellCap records per cell.  (A tile beyond its budget is taken in runs of
  // rows.)  us per step, at the start and after 1500 steps, against 10 records
  // for every pass, of which a compute unit held 11 of the gradient pass's 12
  // waves: 727k particles 767 and 800, now 729 and 760; 324k 362 and 379, 341 and
  // 353; 183k 227 and 235, 224 and 234; 47k 118 and 129, 118 and 129.
  constexpr int kAleCellCap = 9;
  constexpr int kFixed = kTabBytes + sizeof(uint16_t) * kList * kWave;
  const int most = std::min(3 * (rows + 2) * kCellCap, (65536 - kPoolHdr - kFixed) / SLOT);
  const int base = std::min(3 * (rows + 2) * kAleCellCap, most);
  const int lds = kStaticHdr + kFixed + 32;  // (with the rounding to allocation granules below)
  const int fit = std::max(1, c->lds_cu / (lds + base * SLOT));
  const int want = std::max(1, grid_for(c->n_ub, 48 * c->num_cu));
  const int share = c->lds_cu / std::min({fit, want, c->waves_per_cu}) / kLdsGranule * kLdsGranule;
  const int cap = std::max(base, std::min(most, (share - lds) / SLOT));
  // the static walk: a cell build serves several passes of different cost
  // profiles, and the dam breaks these passes run on give each wave about ten
  // tiles, too few for the pooled walk to pay for its chunk cut
  const TileGrid tg = tile_grid(c, true, kFixed + (size_t)cap * SLOT, false);
  if (int e = ensure_tile_list(c, 0)) return e;
  return launch_timed(c, [&] {
    hipLaunchKernelGGL(k_ale_pass32<P>, tg.grid, tg.block, tg.lds, c->stream, pol,
                       c->cell_start, c->cellof, rows, c->scal, c->tile_list, cap, tg.lds_wave,
                        c->counters);
  });
}

// launch of one FP64 pair pass by cells
template <class A, int H>
int launch_pass64(tsph_ctx *c, int slot) {
  using P = AleCell64<A, H>;
  constexpr int lds = cell_lds_bytes<P>();
  const Soa &d = c->cur;
  if (int e = ensure_cell_entries(c)) return e;
  const int groups = cell_groups(c, k_ale_cells64<P>, P::kWaves, lds, c->ale_fit[slot]);
  return launch_timed(c, [&] {
    hipLaunchKernelGGL(k_ale_cells64<P>, dim3(groups), dim3(P::kWaves * kWave), lds, c->stream,
                       P{{d.r, d.v, d.n, d.rho, d.omega, d.type, d.gradrho, d.gradvx, d.gradvy,
                          d.domega, d.domegarho, d.domegav}, ale64(c->k)},
                       cell_grid(c->k), c->cell_start, cell_source(c), c->counters);
  });
}

template <class A>
int launch_pass64(tsph_ctx *c, int slot) {
  return cells_wide(c) ? launch_pass64<A, 4>(c, slot) : launch_pass64<A, 2>(c, slot);
}

}  // namespace

// muscl: 0 no gradients (first order), 1 gradients with alpha = 1, 2 minmod-limited
int launch_ale_density(tsph_ctx *c, int muscl) {
  const bool mixed = c->prm.precision == TSPH_PREC_MIXED;
  if (mixed) {
    const C32A cc = make_c32a(c->k);
    if (muscl == 0) return launch_pass32<Dens32<false, false>, slot_bytes32<false>()>(c, {c->cur, c->k, cc});
    if (muscl == 1) return launch_pass32<Dens32<true, false>, slot_bytes32<true>()>(c, {c->cur, c->k, cc});
    return launch_pass32<Dens32<true, true>, slot_bytes32<true>()>(c, {c->cur, c->k, cc});
  }
  if (muscl == 0) return launch_pass64<Dens64<false, false>>(c, 0);
  if (muscl == 1) return launch_pass64<Dens64<true, false>>(c, 1);
  return launch_pass64<Dens64<true, true>>(c, 2);
}

int launch_ale_acceleration(tsph_ctx *c, int muscl) {
  const bool mixed = c->prm.precision == TSPH_PREC_MIXED;
  if (mixed) {
    const C32A cc = make_c32a(c->k);
    if (muscl == 0) return launch_pass32<Acc32P<false, false>, slot_bytes32<false>()>(c, {c->cur, c->k, cc});
    if (muscl == 1) return launch_pass32<Acc32P<true, false>, slot_bytes32<true>()>(c, {c->cur, c->k, cc});
    return launch_pass32<Acc32P<true, true>, slot_bytes32<true>()>(c, {c->cur, c->k, cc});
  }
  if (muscl == 0) return launch_pass64<Acc64P<false, false>>(c, 3);
  if (muscl == 1) return launch_pass64<Acc64P<true, false>>(c, 4);
  return launch_pass64<Acc64P<true, true>>(c, 5);
}

int launch_ale_gradient(tsph_ctx *c) {
  if (c->prm.precision == TSPH_PREC_MIXED)
    return launch_pass32<Grad32, slot_bytes32<false>()>(c, {c->cur, c->k, make_c32a(c->k)});
  return launch_pass64<Grad64>(c, 6);
}

int launch_ale_density_pressure(tsph_ctx *c, double dt) {
  hipLaunchKernelGGL(k_ale_density_pressure, dim3(grid_for(c->n_ub, 256)), dim3(256), 0, c->stream,
                     c->cur, c->scal, c->k, dt, c->counters);
  TSPH_HIP(hipGetLastError());
  c->records_valid = false;
  return 0;
}

int launch_ale_leapfrog_one(tsph_ctx *c, double dt) {
  hipLaunchKernelGGL(k_ale_lf1, dim3(grid_for(c->n_ub, 256)), dim3(256), 0, c->stream, c->cur,
                     c->scal, dt);
  TSPH_HIP(hipGetLastError());
  c->records_valid = false;
  return 0;
}

int launch_ale_leapfrog_two(tsph_ctx *c, double dt, int step) {
  hipLaunchKernelGGL(k_ale_lf2, dim3(grid_for(c->n_ub, 256)), dim3(256), 0, c->stream, c->cur,
                     c->scal, dt, (int)(step == 1));
  TSPH_HIP(hipGetLastError());
  c->records_valid = false;
  c->marks_valid = false;
  return 0;
}

}  // namespace tsph
