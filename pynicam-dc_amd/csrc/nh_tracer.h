// Tracer transport of the last RK stage: MIURA2004 flux form with the
// Thuburn (1996) limiters (nhm/dynamics/mod_src_tracer.py:83-1228).
//
//   vertical half step   TrcFlux (fluxes, density), TrcVert1 (every column, all
//                        tracers in place)
//   horizontal step      TrcHFlux (arc mass fluxes, mass centroids), TrcRhog2,
//                        then for one or two tracers TrcGradQ -> halo -> TrcRemap
//                        and for each TrcQout -> halo -> TrcApply (both as column
//                        tiles where the limiter is on, nh_trccol.h)
//   vertical half step   TrcVert2 (compute cells, a group of tracers)
//
// The face mass fluxes of the reference's flx_h(i, j, face) are formed on the
// fly from one value per hexagon arc: face 0/1/2 of (i, j) is the AI/AIJ/AJ arc
// of (i, j); faces 3/4/5 are the same arcs of (i-1, j), (i-1, j-1), (i, j-1)
// with the sign flipped and this cell's area.  The limiter's inflow bounds
// (Qin) are recomputed from q on the 7-point stencil instead of being stored.
#pragma once

#include "nh_step.h"

NH_BEGIN

// CONST_EPS / CONST_HUGE of the field precision (np.finfo(rdtype).eps / .max,
// mod_const.py:170-172)
template <class T> struct Lim;
template <> struct Lim<double> {
  static constexpr double eps = 2.220446049250313e-16, big = 1.7976931348623157e308;   // NH_KEEP64
};
template <> struct Lim<float> {
  static constexpr float eps = 1.1920928955078125e-07f, big = 3.4028234663852886e+38f;
};
#define NH_EPS (Lim<real>::eps)
#define NH_BIG (Lim<real>::big)

NH_HD inline real dmin(real a, real b) { return (a < b) ? a : b; }
NH_HD inline real dmax(real a, real b) { return (a > b) ? a : b; }
NH_HD inline real clip(real x, real lo, real hi) { return dmin(dmax(x, lo), hi); }
NH_HD inline real upwind_mask(real ch) { return real(0.5) - nsign(real(0.5), ch - NH_EPS); }

// ----------------------------------------------------------------------------
// vertical half step of one tracer column (mod_src_tracer.py:420-533 and the
// limiter mod_src_tracer.py:1909-2074), streamed in k.  A column is a serial
// chain over its levels; the loads of level k + 3 go out while level k is formed
// (in place is allowed: every element is loaded once, before its store).
// den(k), flx(k): density and vertical mass flux; fr(k): the density tendency,
// from which dvk(fr, den) forms the divergence term.
// ----------------------------------------------------------------------------
template <class DEN, class FLX, class FR, class DVK>
NH_HD inline void vert_sweep(const Geo& G, int kmin, int kmax, const real* in, real* out, long base, long ks,
                             DEN den, FLX flx, FR fr, DVK dvk, bool limiter, bool clipneg) {
  struct Lev {
    real r, den, flx, fr;   // tracer, density, flux at kk; tendency at kk - 1
  };
  auto load = [&](int kk) {
    const int k2 = (kk > kmax + 1) ? kmax + 1 : kk;   // past the top: not used
    return Lev{ld_own(in + base + (long)k2 * ks), den(k2), flx(k2), fr(k2 - 1)};
  };
  auto ck0 = [&](int k, real f, real dn) -> real {
    return (k >= kmin && k <= kmax) ? -f / dn * G.rdgz[k] : real(0.0);
  };
  Lev n1 = load(kmin + 1), n2 = load(kmin + 2), n3 = load(kmin + 3);
  const real r_km1 = ld_own(in + base + (long)(kmin - 1) * ks);
  real r_k = ld_own(in + base + (long)kmin * ks);
  real den_k = den(kmin);
  real q_km1 = r_km1 / den(kmin - 1);
  real q_k = r_k / den_k;
  real omin_prev = real(0.0), omax_prev = real(0.0);
  real qh_prev = real(0.0);      // limited face value at k-1 (zero at kmin)
  real r_prev = r_km1;
  real f_km1 = real(0.0), f_k = flx(kmin);
  real c0_k = ck0(kmin, f_k, den_k);
  for (int k = kmin; k <= kmax; ++k) {
    const Lev c = n1;
    n1 = n2;
    n2 = n3;
    n3 = load(k + 4);
    const real q_kp1 = c.r / c.den;
    const real c0_kp1 = ck0(k + 1, c.flx, c.den);
    const real c1_k = c.flx / den_k * G.rdgz[k];
    real qh = G.afact[k] * q_k + G.bfact[k] * q_km1;
    real omin = real(0.0), omax = real(0.0);
    if (limiter) {
      const real inL = real(0.5) - nsign(real(0.5), c0_k);
      const real inU = real(0.5) + nsign(real(0.5), c0_kp1);
      const real minL = (inL == real(1.0)) ? dmin(q_k, q_km1) : NH_BIG;
      const real minU = (inU == real(1.0)) ? dmin(q_k, q_kp1) : NH_BIG;
      const real maxL = (inL == real(1.0)) ? dmax(q_k, q_km1) : -NH_BIG;
      const real maxU = (inU == real(1.0)) ? dmax(q_k, q_kp1) : -NH_BIG;
      const real nmin = dmin(dmin(minL, minU), q_k);
      const real nmax = dmax(dmax(maxL, maxU), q_k);
      const real Cin = inL * c0_k + inU * c1_k;
      const real Cout = (real(1.0) - inL) * c0_k + (real(1.0) - inU) * c1_k;
      const real CQmin = inL * c0_k * minL + inU * c1_k * minU;
      const real CQmax = inL * c0_k * maxL + inU * c1_k * maxU;
      const real zsw = real(0.5) - nsign(real(0.5), nabs(Cout) - NH_EPS);
      const real dk = dvk(c.fr, den_k);
      omin = ((q_k - nmax) + nmax * (Cin + Cout - dk) - CQmax) / (Cout + zsw) * (real(1.0) - zsw) + q_k * zsw;
      omax = ((q_k - nmin) + nmin * (Cin + Cout - dk) - CQmin) / (Cout + zsw) * (real(1.0) - zsw) + q_k * zsw;
      if (k > kmin) qh = inL * clip(qh, omin_prev, omax_prev) + (real(1.0) - inL) * clip(qh, omin, omax);
    }
    if (k == kmin) qh = real(0.0);
    if (k > kmin) {
      // update of level k-1 with the face values at k-1 and k
      real o = r_prev - (f_k * qh - f_km1 * qh_prev) * G.rdgz[k - 1];
      if (clipneg && o > -real(1.0e-10) && o < real(0.0)) o = real(0.0);
      out[base + (long)(k - 1) * ks] = o;
    }
    omin_prev = omin;
    omax_prev = omax;
    qh_prev = qh;
    r_prev = r_k;
    r_k = c.r;
    q_km1 = q_k;
    q_k = q_kp1;
    c0_k = c0_kp1;
    den_k = c.den;
    f_km1 = f_k;
    f_k = c.flx;
  }
  {
    // f_k, f_km1: the fluxes at kmax + 1 and kmax
    real o = r_prev - (f_k * real(0.0) - f_km1 * qh_prev) * G.rdgz[kmax];
    if (clipneg && o > -real(1.0e-10) && o < real(0.0)) o = real(0.0);
    out[base + (long)kmax * ks] = o;
  }
  out[base + (long)(kmin - 1) * ks] = real(0.0);
  out[base + (long)(kmax + 1) * ks] = real(0.0);
}

// the vertical mass flux of a half step from the mean flux rw (zero at the
// boundaries), and the density after the first one
NH_HD inline real half_flux(const Dims& d, const real* rw, long b, long ks, int k, real dt) {
  return (k >= d.kmin + 1 && k <= d.kmax) ? (real(0.0) + ldc(rw + b + (long)k * ks) * real(1.0)) * real(0.5) * dt
                                          : real(0.0);
}

// Phase 1, one thread per point: vertical flux of the mean mass flux and the
// half-step density (kernels/tracervertflux.py:44-122), on every column
struct TrcFlux {
  static constexpr const char* kName = "trc_flux";
  Dims d; Geo G;
  real dt;
  const real* rw_mean;    // time-mean rhogw
  const real* rhog_in;    // density at the start of the large step
  const real* frhog;      // hyperdiffusion density tendency
  real* flxv;             // out
  real* rhog1;            // out
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p)) return;
    const long a = p.a, ks = p.ks, b = a - (long)p.k * ks;
    const int k = p.k;
    const real f = half_flux(d, rw_mean, b, ks, k, dt);
    real r;
    if (k < d.kmin) r = rhog_in[a + ks];
    else if (k > d.kmax) r = rhog_in[a - ks];
    else r = rhog_in[a] - (half_flux(d, rw_mean, b, ks, k + 1, dt) - f) * G.rdgz[k] + real(0.0) * frhog[a] * dt;
    flxv[a] = f;
    rhog1[a] = r;
  }
};

// Phase 1: first vertical half step of every tracer, on every column (the
// horizontal step reads halo values; computing them here equals filling
// them), one thread per column and tracer.
struct TrcVert1 {
  static constexpr const char* kName = "trc_vert1";
  Dims d; Consts c; Geo G;
  real dt;
  const real* rw_mean;    // time-mean rhogw
  const real* rhog_in;    // density at the start of the large step
  const real* frhog;      // hyperdiffusion density tendency
  real* rhogq;            // nq tracer fields, in place
  int limiter;
  NH_HD long columns() const { return d.nreg + 12; }
  // t < nq * columns()
  NH_HD void operator()(long t) const {
    const long q = t / columns();
    const Cell cl = cell_of(d, t - q * columns());
    const long ks = cl.ks, b = cl.base;
    real* f = rhogq + q * d.NF;
    vert_sweep(G, d.kmin, d.kmax, f, f, b, ks, [&](int k) { return ldc(rhog_in + b + (long)k * ks); },
               [&](int k) { return half_flux(d, rw_mean, b, ks, k, dt); },
               [&](int k) { return ldc(frhog + b + (long)k * ks); },
               [&](real fr, real den) { return real(0.0) * fr / den * dt; }, limiter != 0, false);
  }
};

// Phase 2: second vertical half step of nq tracers on the compute cells, with
// the density after the horizontal step, and the small-negative clip
// (mod_src_tracer.py:947-1204), one thread per column and tracer.
struct TrcVert2 {
  static constexpr const char* kName = "trc_vert2";
  Dims d; Consts c; Geo G;
  real dt;
  const real* flxv;
  const real* rhog2;
  const real* frhog;
  const real* in;     // nq tracers after the horizontal step
  real* out;          // nq tracer fields
  int limiter;
  NH_HD long columns() const { return d.nreg + 12; }
  // t < nq * columns()
  NH_HD void operator()(long t) const {
    const long q = t / columns();
    const Cell cl = cell_of(d, t - q * columns());
    if (cl.pole ? cl.v != 0 : !cl.inner) return;
    const long ks = cl.ks, b = cl.base;
    vert_sweep(G, d.kmin, d.kmax, in + q * d.NF, out + q * d.NF, b, ks,
               [&](int k) { return ldc(rhog2 + b + (long)k * ks); },
               [&](int k) { return ldc(flxv + b + (long)k * ks); },
               [&](int k) { return ldc(frhog + b + (long)k * ks); },
               [&](real fr, real den) { return real(0.0) * fr / den * dt; }, limiter != 0, true);
  }
};

// ----------------------------------------------------------------------------
// horizontal mass fluxes (mod_src_tracer.py:1376-1533)
// ----------------------------------------------------------------------------
// field layout of the arc quantities: fa[arc] (0.5 * rhov.HN of the arc), xc[arc*3+d]
//
// One thread per column and KC levels: its 30 coefficients stay in registers,
// each of the four triangles is formed once for the arcs that share it, and all
// loads of a level come before its 12 stores.  16 fields, 96 us at the streaming
// rate at gl07 z40 mixed.  As points with triangles formed per arc, as points with
// shared triangles, and so: gl07 mixed 223, 188, 166 us; gl07 FP64 448, 362, 299;
// gl06 z60 FP64 184, 147, 118.
struct TrcHFlux {
  static constexpr const char* kName = "trc_hflux";
  Dims d; Geo G;
  real dt;
  const real* pm;   // rhog, rhogvx, rhogvy, rhogvz (field stride NF)
  real* fa[3];
  real* xc[9];
  int KC;           // levels per thread
  long threads() const { return (d.nreg + 2) * ((d.kall + KC - 1) / KC); }
  NH_HD void operator()(long t) const {
    const long NF = d.NF, nc = d.nreg + 2;
    const long chunk = t / nc, c = t - chunk * nc;
    const int k0 = (int)chunk * KC, k1 = (k0 + KC < d.kall) ? k0 + KC : d.kall;
    if (c >= d.nreg) {
      const int lp = (int)(c - d.nreg);
      for (int k = k0; k < k1; ++k) pole(lp, d.R + (long)(lp * d.kall + k) * 6);
      return;
    }
    const int g = d.g, gg = g * g;
    const long ci = c;
    const int l = (int)(ci / gg), h = (int)(ci - (long)l * gg), j = h / g, i = h - j * g;
    if (i > g - 2 || j > g - 2) return;
    const long nreg = d.nreg;
    // the four triangles of a point's arcs: TI and TJ of the point, TJ of
    // (i, j-1) and TI of (i-1, j) (the point's own where there is none: the
    // arc is then dropped)
    const int south = j >= 1 ? -g : 0, west = i >= 1 ? -1 : 0;
    real wi[3], wj[3], ws[3], ww[3], hn[9], xr[9];
    for (int m = 0; m < 3; ++m) {
      wi[m] = rcp(G.twt, nreg, m, ci);
      wj[m] = rcp(G.twt, nreg, 3 + m, ci);
      ws[m] = rcp(G.twt, nreg, 3 + m, ci + south);
      ww[m] = rcp(G.twt, nreg, m, ci + west);
    }
    for (int m = 0; m < 9; ++m) {
      hn[m] = rcp(G.ahn, nreg, m, ci);
      xr[m] = rcp(G.axr, nreg, m, ci);
    }
    for (int k = k0; k < k1; ++k) {
      const long a = ((long)l * d.kall + k) * gg + h;
      const unsigned o = byte_off(a);
      real f[4][6];
      for (int q = 0; q < 4; ++q) {
        const real* pq = pm + q * NF;
        f[q][0] = at_off(pq, o);
        f[q][1] = at_off(pq + 1, o);
        f[q][2] = at_off(pq + 1 + g, o);
        f[q][3] = at_off(pq + g, o);
        f[q][4] = at_off(pq, o + (unsigned)(south * (int)sizeof(real)));
        f[q][5] = at_off(pq, o + (unsigned)(west * (int)sizeof(real)));
      }
      // arcs: AI (TJ(i, j-1) + TI(i, j)), AIJ (TI(i, j) + TJ(i, j)), AJ (TJ(i, j) + TI(i-1, j))
      real s[3][4];
      for (int q = 0; q < 4; ++q) {
        const real* e = f[q];
        real ti = (e[0] * wi[0] + e[1] * wi[1]) + e[2] * wi[2];
        const real tj = e[0] * wj[0] + (e[2] * wj[1] + e[3] * wj[2]);
        const real ts = e[4] * ws[0] + (e[1] * ws[1] + e[0] * ws[2]);
        real tw = (e[5] * ww[0] + e[0] * ww[1]) + e[3] * ww[2];
        if (j == 0 && i <= 1) {
          // the (0, 0) TI triangle is replaced by TJ(1, 0) on pentagon regions (arithmetic mask, all regions)
          const real m0 = G.sgp[l] ? real(0.0) : real(1.0), m1 = G.sgp[l] ? real(1.0) : real(0.0);
          const real* b = pm + q * NF + a + (1 - i);
          const long c1 = ci + (1 - i);
          const real t1 = b[0] * rcp(G.twt, nreg, 3, c1)
                          + (b[1 + g] * rcp(G.twt, nreg, 4, c1) + b[g] * rcp(G.twt, nreg, 5, c1));
          if (i == 0) ti = ti * m0 + t1 * m1;
          else tw = tw * m0 + t1 * m1;
        }
        s[0][q] = ts + ti;
        s[1][q] = ti + tj;
        s[2][q] = tj + tw;
      }
      for (int arc = 0; arc < 3; ++arc) {
        const bool valid = arc == 1 || (arc == 0 ? j >= 1 : i >= 1);
        const real* v2 = s[arc] + 1;
        const real rr = real(1.0) / dmax(s[arc][0], NH_EPS);
        const real fl = real(0.5) * (v2[0] * hn[arc * 3] + v2[1] * hn[arc * 3 + 1] + v2[2] * hn[arc * 3 + 2]);
        at_off(fa[arc], o) = valid ? fl : real(0.0);
        for (int dd = 0; dd < 3; ++dd) {
          const real xv = xr[arc * 3 + dd] - v2[dd] * rr * dt * real(0.5);
          at_off(xc[arc * 3 + dd], o) = valid ? xv : real(0.0);
        }
      }
    }
  }
  NH_HD void pole(int lp, long a0) const {
    const long NF = d.NF;
    real rt[6][4];
    for (int v = 1; v <= 5; ++v) {
      int vp = (v == 5) ? 1 : v + 1;
      const real* w = G.twt_pl + (v * 2 + lp) * 3;
      for (int q = 0; q < 4; ++q) {
        const real* f = pm + q * NF;
        rt[v][q] = f[a0] * w[0] + f[a0 + v] * w[1] + f[a0 + vp] * w[2];
      }
    }
    for (int v = 1; v <= 5; ++v) {
      int vm = (v == 1) ? 5 : v - 1;
      const real rr = real(1.0) / dmax(rt[vm][0] + rt[v][0], NH_EPS);
      const real v2x = rt[vm][1] + rt[v][1], v2y = rt[vm][2] + rt[v][2], v2z = rt[vm][3] + rt[v][3];
      const real* hn = G.ahn_pl + (v * 2 + lp) * 3;
      fa[0][a0 + v] = real(0.5) * (v2x * hn[0] + v2y * hn[1] + v2z * hn[2]);
      const real* xr = G.axr_pl + (v * 2 + lp) * 3;
      xc[0][a0 + v] = xr[0] - v2x * rr * dt * real(0.5);
      xc[1][a0 + v] = xr[1] - v2y * rr * dt * real(0.5);
      xc[2][a0 + v] = xr[2] - v2z * rr * dt * real(0.5);
    }
  }
};

// face mass flux of face m (0..5) of regional cell at address a / column ci
NH_HD inline real face_flux(const Geo& G, const Dims& d, const real* const* fa, long a, long ci, int i, int j,
                              int l, int m, real dt) {
  const int g = d.g;
  const real ra = rcp(G.rarea, d.nreg, 0, ci);
  switch (m) {
    case 0: return fa[0][a] * ra * dt;
    case 1: return fa[1][a] * ra * dt;
    case 2: return fa[2][a] * ra * dt;
    case 3: return -fa[0][a - 1] * ra * dt;
    case 4: return -fa[1][a - 1 - g] * ra * dt;
    default: {
      real f = -fa[2][a - g] * ra * dt;
      if (i == 1 && j == 1) f *= (G.sgp[l] ? real(0.0) : real(1.0));
      return f;
    }
  }
}

// density after the horizontal step (mod_src_tracer.py:889-929)
struct TrcRhog2 {
  static constexpr const char* kName = "trc_rhog2";
  Dims d; Consts c; Geo G;
  real dt;
  const real* fa[3];
  const real* rhog1;
  const real* frhog;
  real* rhog2;
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (pt_of(d, plane, x, p)) levels(cell_of_pt(p), p.k, p.k + 1);
  }
  NH_HD void levels(const Cell& cl, int k0, int k1) const {
    if (cl.pole ? cl.v != 0 : !cl.inner) return;
    for (int k = k0; k < k1; ++k) {
      const long a = cl.base + k * cl.ks;
      if (cl.pole) {
        real r = rhog1[a];
        for (int v = 1; v <= 5; ++v) r -= fa[0][a + v] * G.rarea_pl[cl.lp] * dt;
        r += real(1.0) * frhog[a] * dt;
        rhog2[a] = r;
      } else {
        real f[6];
        for (int m = 0; m < 6; ++m) f[m] = face_flux(G, d, fa, a, cl.ci, cl.i, cl.j, cl.l, m, dt);
        rhog2[a] = rhog1[a] - ((((f[0] + f[1]) + f[2]) + f[3]) + f[4] + f[5] - (real(1.0) * frhog[a] * dt));
      }
    }
  }
};

// gradient of q = rhogq / rhog1 (OPRT_gradient, kernels/oprtgradient.py:45-88)
// the pole centres (the regional points run as Oper7C over SrcRatio)
struct TrcGradQ {
  static constexpr const char* kName = "trc_gradq";
  Dims d; Geo G;
  const real* rq;
  const real* rhog1;
  real* gq[3];
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p) || !p.pole || p.v != 0) return;
    real qv[6];
    for (int v = 0; v < 6; ++v) qv[v] = rq[p.a + v] / rhog1[p.a + v];
    for (int dd = 0; dd < 3; ++dd) {
      real acc = real(0.0);
      for (int v = 0; v < 6; ++v) {
        const real pv = G.cgrad_pl[(v * 2 + p.lp) * 3 + dd] * qv[v];
        acc = (v == 0) ? pv : acc + pv;
      }
      gq[dd][p.a] = acc;
    }
  }
};

// ----------------------------------------------------------------------------
// upwind face values (horizontal_remap, mod_src_tracer.py:1642-1843)
// ----------------------------------------------------------------------------
// N tracers (1 or 2) per launch: the nine centroid fields and the three fluxes,
// two thirds of what one tracer reads, are read once for both.  Every load of a
// point is issued before the first use and an arc that does not exist is a
// select (its operands are in bounds), so a point waits once for memory.
// gl06 z60 FP64, two tracers: 274 us as two point launches of one, 121 as a pair
// (28 fields, 131 us at the streaming rate from memory); gl07 z40 mixed, one
// tracer: 176 -> 148 us.
template <int N>
struct TrcRemap {
  static constexpr const char* kName = "trc_remap";
  Dims d; Geo G;
  real dt;
  const real* rq[N];
  const real* rhog1;
  const real* gq[N][3];
  const real* fa[3];
  const real* xc[9];
  real* qa[N][3];
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p)) return;
    if (p.pole) {
      if (p.v == 0) return;
      // pole arc v: upwind value from the pole centre or spoke v
      const int lp = p.lp, v = p.v;
      const real* xp0 = G.gx_pl + (0 * 2 + lp) * 3;
      const real* xpv = G.gx_pl + (v * 2 + lp) * 3;
      const long av = p.a, a0 = av - v;
      const real xcx = xc[0][av], xcy = xc[1][av], xcz = xc[2][av];
      const real ch = fa[0][av] * G.rarea_pl[lp] * dt / rhog1[a0];
      const real cm = upwind_mask(ch);
      for (int n = 0; n < N; ++n) {
        const real* const* gn = gq[n];
        const real q0 = rq[n][a0] / rhog1[a0], qv = rq[n][av] / rhog1[av];
        const real qap = q0 + gn[0][a0] * (xcx - xp0[0]) + gn[1][a0] * (xcy - xp0[1]) + gn[2][a0] * (xcz - xp0[2]);
        const real qam = qv + gn[0][av] * (xcx - xpv[0]) + gn[1][av] * (xcy - xpv[1]) + gn[2][av] * (xcz - xpv[2]);
        qa[n][0][av] = cm * qam + (real(1.0) - cm) * qap;
      }
      return;
    }
    const int g = d.g, i = p.i, j = p.j;
    if (i > g - 2 || j > g - 2) return;
    const long nreg = d.nreg, ci = p.ci;
    const unsigned o = byte_off(p.a);
    // neighbour across each arc: AI (i+1, j), AIJ (i+1, j+1), AJ (i, j+1)
    const int noff[3] = {1, 1 + g, g};
    real xv[9], fv[3], r[4], xg[4][3], q[N][4], gv[N][4][3];
    for (int m = 0; m < 9; ++m) xv[m] = at_off(xc[m], o);
    for (int m = 0; m < 3; ++m) fv[m] = at_off(fa[m], o);
    const real ra = rcp(G.rarea, nreg, 0, ci);
    for (int m = 0; m < 4; ++m) {
      const int of = m ? noff[m - 1] : 0;
      r[m] = at_off(rhog1 + of, o);
      for (int dd = 0; dd < 3; ++dd) xg[m][dd] = rcp(G.gx, nreg, dd, ci + of);
      for (int n = 0; n < N; ++n) {
        q[n][m] = at_off(rq[n] + of, o);
        for (int dd = 0; dd < 3; ++dd) gv[n][m][dd] = at_off(gq[n][dd] + of, o);
      }
    }
    for (int n = 0; n < N; ++n)
      for (int m = 0; m < 4; ++m) q[n][m] = q[n][m] / r[m];
    for (int arc = 0; arc < 3; ++arc) {
      const real ch = fv[arc] * ra * dt / r[0];
      const real cm = upwind_mask(ch);
      const bool valid = arc == 1 || (arc == 0 ? j >= 1 : i >= 1);
      const real* xa = xv + arc * 3;
      for (int n = 0; n < N; ++n) {
        const real* g0 = gv[n][0];
        const real* g1 = gv[n][arc + 1];
        const real* x1 = xg[arc + 1];
        const real qap = q[n][0] + g0[0] * (xa[0] - xg[0][0]) + g0[1] * (xa[1] - xg[0][1]) + g0[2] * (xa[2] - xg[0][2]);
        const real qam = q[n][arc + 1] + g1[0] * (xa[0] - x1[0]) + g1[1] * (xa[1] - x1[1]) + g1[2] * (xa[2] - x1[2]);
        const real s = cm * qam + (real(1.0) - cm) * qap;
        at_off(qa[n][arc], o) = valid ? s : real(0.0);
      }
    }
  }
};

// ----------------------------------------------------------------------------
// Thuburn horizontal limiter (horizontal_limiter_thuburn, mod_src_tracer.py:2190-2660)
// ----------------------------------------------------------------------------
// q on the 7-point stencil of one regional cell, and the inflow bounds of the
// six faces.  Stencil: 0 (i,j) 1 (i+1,j) 2 (i+1,j+1) 3 (i,j+1) 4 (i-1,j)
// 5 (i-1,j-1) 6 (i,j-1).
struct FaceBounds {
  real mn[6], mx[6];      // min/max of q over the four cells around each face
  real cm[6];             // upwind mask of the face's owner
  bool pent;                // face 4 uses the pentagon override
};

NH_HD inline void face_bounds(const real q[7], const real cmo[6], bool pentagon, FaceBounds& fb) {
  // owner sets: own AI {0,6,1,2}, own AIJ {0,1,2,3}, own AJ {0,2,3,4},
  // (i-1,j) AI {4,5,0,3}, (i-1,j-1) AIJ {5,6,0,4} (pentagon: {5,0,1,4}), (i,j-1) AJ {6,1,0,5}
  const int sets[6][4] = {{0, 6, 1, 2}, {0, 1, 2, 3}, {0, 2, 3, 4}, {4, 5, 0, 3}, {5, 6, 0, 4}, {6, 1, 0, 5}};
  for (int m = 0; m < 6; ++m) {
    const int* s = sets[m];
    int s1 = s[1], s2 = s[2];
    if (m == 4 && pentagon) { s1 = 0; s2 = 1; }
    const real a = q[s[0]], b = q[s1], c = q[s2], e = q[s[3]];
    fb.mn[m] = dmin(dmin(dmin(a, b), c), e);
    fb.mx[m] = dmax(dmax(dmax(a, b), c), e);
    fb.cm[m] = cmo[m];
  }
  fb.pent = pentagon;
}

// inflow bounds as seen from this cell (Qin(i, j, *, m)): faces 0..2 are owned by the
// cell, faces 3..5 by the neighbour and see the complementary mask
NH_HD inline void qin_of_cell(const FaceBounds& fb, int m, real& lo, real& hi) {
  const real c = fb.cm[m];
  if (m < 3) {
    lo = c * fb.mn[m] + (real(1.0) - c) * NH_BIG;
    hi = c * fb.mx[m] + (real(1.0) - c) * (-NH_BIG);
  } else if (m == 4 && fb.pent) {
    lo = (c == real(1.0)) ? NH_BIG : fb.mn[m];
    hi = (c == real(1.0)) ? -NH_BIG : fb.mx[m];
  } else {
    lo = c * NH_BIG + (real(1.0) - c) * fb.mn[m];
    hi = c * (-NH_BIG) + (real(1.0) - c) * fb.mx[m];
  }
}

// inflow bounds of the same face as seen from its owner (m >= 3 only)
NH_HD inline void qin_of_owner(const FaceBounds& fb, int m, real& lo, real& hi) {
  const real c = fb.cm[m];
  if (m == 4 && fb.pent) {
    lo = (c == real(1.0)) ? fb.mn[m] : NH_BIG;
    hi = (c == real(1.0)) ? fb.mx[m] : -NH_BIG;
  } else {
    lo = c * fb.mn[m] + (real(1.0) - c) * NH_BIG;
    hi = c * fb.mx[m] + (real(1.0) - c) * (-NH_BIG);
  }
}

// shared per-cell setup: q on the stencil, owner masks, own Courant numbers
struct TrcCellCtx {
  real q[7];
  real cmo[6];    // owner mask per face
  real ch[6];     // this cell's Courant numbers
  real f[6];      // this cell's face fluxes
};

NH_HD inline void trc_cell(const Geo& G, const Dims& d, const Cell& cl, long a, real dt, const real* rq,
                           const real* rhog1, const real* const* fa, TrcCellCtx& x) {
  long off[7];
  stencil_offsets(d.g, off);
  for (int m = 0; m < 7; ++m) x.q[m] = rq[a + off[m]] / rhog1[a + off[m]];
  for (int m = 0; m < 6; ++m) x.f[m] = face_flux(G, d, fa, a, cl.ci, cl.i, cl.j, cl.l, m, dt);
  for (int m = 0; m < 6; ++m) x.ch[m] = x.f[m] / rhog1[a];
  for (int m = 0; m < 3; ++m) x.cmo[m] = upwind_mask(x.ch[m]);
  // faces 3..5: the owner's face 0/1/2 mask with the owner's own flux and density
  const long nreg = d.nreg;
  const long o3 = a - 1, o4 = a - 1 - d.g, o5 = a - d.g;
  const long c3 = cl.ci - 1, c4 = cl.ci - 1 - d.g, c5 = cl.ci - d.g;
  x.cmo[3] = upwind_mask(fa[0][o3] * rcp(G.rarea, nreg, 0, c3) * dt / rhog1[o3]);
  x.cmo[4] = upwind_mask(fa[1][o4] * rcp(G.rarea, nreg, 0, c4) * dt / rhog1[o4]);
  x.cmo[5] = upwind_mask(fa[2][o5] * rcp(G.rarea, nreg, 0, c5) * dt / rhog1[o5]);
}

// outflow bounds of a regional cell
NH_HD inline void trc_qout_cell(const TrcCellCtx& x, bool pentagon, real dk, real& o0, real& o1) {
  FaceBounds fb;
  face_bounds(x.q, x.cmo, pentagon, fb);
  real nmin = x.q[0], nmax = x.q[0];
  real lo[6], hi[6];
  for (int m = 0; m < 6; ++m) {
    qin_of_cell(fb, m, lo[m], hi[m]);
    nmin = dmin(nmin, lo[m]);
    nmax = dmax(nmax, hi[m]);
  }
  real Cin = -real(0.0), Cout = -real(0.0), CQmin = -real(0.0), CQmax = -real(0.0);
  for (int m = 0; m < 6; ++m) {
    const real chm = (x.ch[m] < real(0.0)) ? x.ch[m] : real(0.0);
    Cin = Cin + chm;
    Cout = Cout + (x.ch[m] - chm);
    CQmin = CQmin + chm * lo[m];
    CQmax = CQmax + chm * hi[m];
  }
  const real zsw = real(0.5) - nsign(real(0.5), nabs(Cout) - NH_EPS);
  const real qq = x.q[0];
  o0 = (qq - CQmax - nmax * (real(1.0) - Cin - Cout + dk)) / (Cout + zsw) * (real(1.0) - zsw) + qq * zsw;
  o1 = (qq - CQmin - nmin * (real(1.0) - Cin - Cout + dk)) / (Cout + zsw) * (real(1.0) - zsw) + qq * zsw;
}

// the pole centres (the regional cells run as TrcQoutC)
struct TrcQout {
  static constexpr const char* kName = "trc_qout";
  Dims d; Geo G;
  real dt;
  const real* rq;
  const real* rhog1;
  const real* frhog;
  const real* fa[3];
  real* qout[2];
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p) || !p.pole || p.v != 0) return;
    const long a = p.a;
    const real dk = real(1.0) * frhog[a] / rhog1[a] * dt;
    const real ra = G.rarea_pl[p.lp];
    const real q0 = rq[a] / rhog1[a];
    real qv[6];
    for (int v = 1; v <= 5; ++v) qv[v] = rq[a + v] / rhog1[a + v];
    real nmin = q0, nmax = q0, Cin = real(0.0), Cout = real(0.0), CQmin = real(0.0), CQmax = real(0.0);
    for (int v = 1; v <= 5; ++v) {
      const int vp = (v == 5) ? 1 : v + 1, vm = (v == 1) ? 5 : v - 1;
      const real mn = dmin(dmin(dmin(q0, qv[v]), qv[vm]), qv[vp]);
      const real mx = dmax(dmax(dmax(q0, qv[v]), qv[vm]), qv[vp]);
      const real ch = fa[0][a + v] * ra * dt / rhog1[a];
      const real cm = upwind_mask(ch);
      const real lo = (cm == real(1.0)) ? mn : NH_BIG;
      const real hi = (cm == real(1.0)) ? mx : -NH_BIG;
      nmin = dmin(nmin, lo);
      nmax = dmax(nmax, hi);
      const real chm = cm * ch;
      Cin = Cin + chm;
      Cout = Cout + (ch - chm);
      CQmin = CQmin + chm * lo;
      CQmax = CQmax + chm * hi;
    }
    const real zsw = real(0.5) - nsign(real(0.5), nabs(Cout) - NH_EPS);
    const real den = Cout + zsw, fac = real(1.0) - zsw;
    qout[0][a] = (q0 - CQmax - nmax * (real(1.0) - Cin - Cout + dk)) / den * fac + q0 * zsw;
    qout[1][a] = (q0 - CQmin - nmin * (real(1.0) - Cin - Cout + dk)) / den * fac + q0 * zsw;
  }
};

// limited outflow of a regional cell: sum over the faces of flux times limited
// value.  qa: unlimited face values, q0, q1: outflow bounds on the stencil
NH_HD inline real trc_outflow_cell(const TrcCellCtx& x, bool pentagon, const real qa[6], const real q0[7],
                                   const real q1[7]) {
  FaceBounds fb;
  face_bounds(x.q, x.cmo, pentagon, fb);
  // owner cell and downstream cell of the owner's face (stencil indices)
  const int own[6] = {0, 0, 0, 4, 5, 6};
  const int dst[6] = {1, 2, 3, 0, 0, 0};
  real s_face[6];
  for (int m = 0; m < 6; ++m) {
    const real cm = fb.cm[m];
    real loA, hiA, loB, hiB;     // A: owner side, B: downstream side
    if (m < 3) {
      qin_of_cell(fb, m, loA, hiA);
      // the downstream cell sees the complementary mask
      loB = cm * NH_BIG + (real(1.0) - cm) * fb.mn[m];
      hiB = cm * (-NH_BIG) + (real(1.0) - cm) * fb.mx[m];
    } else {
      qin_of_owner(fb, m, loA, hiA);
      qin_of_cell(fb, m, loB, hiB);
    }
    const real s = qa[m];
    const real v1 = cm * clip(s, loA, hiA) + (real(1.0) - cm) * clip(s, loB, hiB);
    const int o = own[m], dn = dst[m];
    s_face[m] = cm * dmax(dmin(v1, q1[dn]), q0[dn]) + (real(1.0) - cm) * dmax(dmin(v1, q1[o]), q0[o]);
  }
  return x.f[0] * s_face[0] + x.f[1] * s_face[1] + x.f[2] * s_face[2] + x.f[3] * s_face[3] + x.f[4] * s_face[4]
         + x.f[5] * s_face[5];
}

// limited face values and the flux-form update of rhogq (mod_src_tracer.py:2536-2660, :838-874)
struct TrcApply {
  static constexpr const char* kName = "trc_apply";
  Dims d; Geo G;
  real dt;
  const real* rq;
  const real* rhog1;
  const real* fa[3];
  const real* qa[3];
  const real* qout[2];
  real* out;
  // limiter off (mod_src_tracer.py:789): the face values go in unlimited; faces
  // 3..5 then take the remap's own values of this cell (:1785), upwind by this
  // cell's mask between the extrapolations from here and from the face's owner
  int limiter;
  const real* gq[3];
  const real* xc[9];
  NH_HD real face_unlimited(const Cell& cl, long a, int m, real fm) const {
    if (m < 3) return qa[m][a];
    const int g = d.g, arc = m - 3;
    const long o = (m == 3) ? a - 1 : (m == 4) ? a - 1 - g : a - g;
    const long co = (m == 3) ? cl.ci - 1 : (m == 4) ? cl.ci - 1 - g : cl.ci - g;
    const long nreg = d.nreg;
    const real* x0 = xc[arc * 3];
    const real* x1 = xc[arc * 3 + 1];
    const real* x2 = xc[arc * 3 + 2];
    const real am = rq[a] / rhog1[a] + gq[0][a] * (x0[o] - rcp(G.gx, nreg, 0, cl.ci))
                    + gq[1][a] * (x1[o] - rcp(G.gx, nreg, 1, cl.ci)) + gq[2][a] * (x2[o] - rcp(G.gx, nreg, 2, cl.ci));
    const real ap = rq[o] / rhog1[o] + gq[0][o] * (x0[o] - rcp(G.gx, nreg, 0, co))
                    + gq[1][o] * (x1[o] - rcp(G.gx, nreg, 1, co)) + gq[2][o] * (x2[o] - rcp(G.gx, nreg, 2, co));
    const real cm = upwind_mask(fm / rhog1[a]);
    return cm * am + (real(1.0) - cm) * ap;
  }
  // with the limiter the pole centres only (the regional cells run as TrcApplyC)
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p) || !pt_compute(p)) return;
    const long a = p.a;
    if (!p.pole) {
      if (limiter) return;
      const Cell cl = cell_of_pt(p);
      real f[6], s[6];
      for (int m = 0; m < 6; ++m) f[m] = face_flux(G, d, fa, a, cl.ci, cl.i, cl.j, cl.l, m, dt);
      for (int m = 0; m < 6; ++m) s[m] = face_unlimited(cl, a, m, f[m]);
      out[a] = rq[a] - (f[0] * s[0] + f[1] * s[1] + f[2] * s[2] + f[3] * s[3] + f[4] * s[4] + f[5] * s[5]);
      return;
    }
    const real ra = G.rarea_pl[p.lp];
    if (!limiter) {
      real r = rq[a];
      for (int v = 1; v <= 5; ++v) r -= fa[0][a + v] * ra * dt * qa[0][a + v];
      out[a] = r;
      return;
    }
    const real q0 = rq[a] / rhog1[a];
    real qv[6];
    for (int v = 1; v <= 5; ++v) qv[v] = rq[a + v] / rhog1[a + v];
    real r = rq[a];
    for (int v = 1; v <= 5; ++v) {
      const int vp = (v == 5) ? 1 : v + 1, vm = (v == 1) ? 5 : v - 1;
      const real mn = dmin(dmin(dmin(q0, qv[v]), qv[vm]), qv[vp]);
      const real mx = dmax(dmax(dmax(q0, qv[v]), qv[vm]), qv[vp]);
      const real fl = fa[0][a + v] * ra * dt;
      const real cm = upwind_mask(fl / rhog1[a]);
      const real lo0 = (cm == real(1.0)) ? mn : NH_BIG, hi0 = (cm == real(1.0)) ? mx : -NH_BIG;
      const real lo1 = (cm == real(1.0)) ? NH_BIG : mn, hi1 = (cm == real(1.0)) ? -NH_BIG : mx;
      real s = qa[0][a + v];
      const real s0 = clip(s, lo0, hi0), s1 = clip(s, lo1, hi1);
      s = cm * s0 + (real(1.0) - cm) * s1;
      const real s2 = dmax(dmin(s, qout[1][a + v]), qout[0][a + v]);
      const real s3 = dmax(dmin(s, qout[1][a]), qout[0][a]);
      s = cm * s2 + (real(1.0) - cm) * s3;
      r -= fl * s;
    }
    out[a] = r;
  }
};

NH_END
