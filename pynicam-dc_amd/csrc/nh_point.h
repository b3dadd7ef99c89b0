// Point kernels of the HEVI step: one thread per (column, level).
//
// Horizontal stencils have no vertical recurrence, so they run one thread per
// point on the 2-D grid of nh_columns.h (plane = region level, x = point in
// the plane).  Vertical couplings that reach only k-2..k+1 (half-level
// interpolation, boundary rows, the tridiagonal coefficients) are recomputed
// by the thread that needs them, which keeps every kernel free of per-thread
// column arrays.  Only the tridiagonal solve (ViMainV) stays a column kernel.
// The arithmetic of every value follows the reference kernels cited per
// functor, in the reference's operation order.
#pragma once

#include "nh_step.h"

NH_BEGIN

// ----------------------------------------------------------------------------
// single operators (tests and callers of the C-ABI): the pole centres; the
// regional points run as Oper7C
// ----------------------------------------------------------------------------
struct OpLapP {
  static constexpr const char* kName = "oprt_laplacian";
  Dims d; Geo G;
  const real* s;
  real* o;
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p) || !p.pole || p.v != 0) return;
    o[p.a] = lap_pl(G, p.lp, s, p.a);
  }
};

struct OpDivP {
  static constexpr const char* kName = "oprt_divergence";
  Dims d; Geo G;
  const real *vx, *vy, *vz;
  real* o;
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p) || !p.pole || p.v != 0) return;
    const long a = p.a;
    o[a] = div_pl(G, p.lp, [&](int v) { return vx[a + v]; }, [&](int v) { return vy[a + v]; },
                  [&](int v) { return vz[a + v]; });
  }
};

struct OpGradP {
  static constexpr const char* kName = "oprt_gradient";
  Dims d; Geo G;
  const real* s;
  real *ox, *oy, *oz;
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p) || !p.pole || p.v != 0) return;
    real o[3];
    grad_pl(G, p.lp, s, p.a, o);
    ox[p.a] = o[0];
    oy[p.a] = o[1];
    oz[p.a] = o[2];
  }
};

// ----------------------------------------------------------------------------
// Pre_Post (kernels/diag.py:53-143, mod_bndcnd.py:153-238, kernels/thrmdyn.py:56-71)
// ----------------------------------------------------------------------------
struct PrePostP {
  static constexpr const char* kName = "prepost";
  Dims d; Consts c; Geo G;
  real* prog;
  const real* rhogq;
  real* diag;
  real* eth;
  struct Th { real rho, ein, tem, pre; };
  NH_HD Th thermo_v(real rhog, real rhoge, real rhogq0) const {
    Th t;
    t.rho = rhog / real(1.0);
    t.ein = rhoge / rhog;
    const real q = rhogq0 / rhog;
    const real qd = real(1.0) - q;
    const real cv = q * c.CVW_qv + qd * c.CVdry;
    t.tem = t.ein / cv;
    t.pre = t.rho * t.tem * (qd * c.Rdry + q * c.Rvap);
    return t;
  }
  NH_HD Th thermo(long a) const { return thermo_v(prog[a], prog[5 * d.NF + a], rhogq[a]); }
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p)) return;
    const long NF = d.NF, a = p.a, ks = p.ks;
    const int kmin = d.kmin, kmax = d.kmax, k = p.k;
    real* rg = prog;
    real* rw = prog + 4 * NF;
    real* pre = diag + I_PRE * NF;
    real* tem = diag + I_TEM * NF;
    real* w = diag + I_W * NF;
    if (k >= kmin && k <= kmax) {
      // every value is read before the first store (the stores could alias
      // the reads for all the compiler knows, which would serialize them)
      const long al = (k > kmin) ? a - ks : a + ks;   // level below, or above at kmin
      const real rhog = rg[a], rhoge = prog[5 * NF + a], q0 = rhogq[a];
      const real v1 = prog[1 * NF + a], v2 = prog[2 * NF + a], v3 = prog[3 * NF + a];
      const real rwa = rw[a], rgl = rg[al], rgel = prog[5 * NF + al], ql = rhogq[al];
      Th t = thermo_v(rhog, rhoge, q0);
      diag[I_VX * NF + a] = v1 / rhog;
      diag[I_VY * NF + a] = v2 / rhog;
      diag[I_VZ * NF + a] = v3 / rhog;
      tem[a] = t.tem;
      pre[a] = t.pre;
      if (k > kmin) {
        w[a] = rwa / (G.c2w0[k] * rhog + G.c2w1[k] * rgl);
      } else {
        // bottom: rigid lid, with the density of the ghost row after the boundary condition
        const Th t1 = thermo_v(rgl, rgel, ql);
        const real pre_b = t1.pre - t.rho * (G.phi[kmin - 1] - G.phi[kmin + 1]);
        const real rho_b = pre_b / (c.Rdry * t.tem);
        rw[a] = real(0.0);
        w[a] = real(0.0) / (G.c2w0[kmin] * rhog + G.c2w1[kmin] * (rho_b * real(1.0)));
      }
      eth[a] = t.ein + t.pre / t.rho;
      return;
    }
    // ghost rows: TEM thermodynamic condition, free-slip top, rigid bottom
    const bool top = (k == kmax + 1);
    const long an = top ? a - ks : a + ks;            // nearest physical level
    const long an2 = top ? a - 2 * ks : a + 2 * ks;    // next one
    const Th tn = thermo(an);
    const Th tn2 = thermo(an2);
    const real tem_g = tn.tem;
    const real pre_g = top ? tn2.pre - tn.rho * (G.phi[kmax + 1] - G.phi[kmax - 1])
                             : tn2.pre - tn.rho * (G.phi[kmin - 1] - G.phi[kmin + 1]);
    const real rho_g = pre_g / (c.Rdry * tem_g);
    const real rg_g = rho_g * real(1.0);
    const real ein_g = c.CVdry * tem_g;
    tem[a] = tem_g;
    pre[a] = pre_g;
    rg[a] = rg_g;
    prog[5 * NF + a] = rg_g * ein_g;
    const real sgn = top ? real(1.0) : -real(1.0);
    for (int q = 0; q < 3; ++q) {
      const real v = sgn * (prog[(1 + q) * NF + an] / rg[an]) * rg_g;
      prog[(1 + q) * NF + a] = v;
      diag[(I_VX + q) * NF + a] = v / rg_g;
    }
    if (top) {
      rw[a] = -real(0.0);
      w[a] = rw[a] / (G.c2w0[kmax + 1] * rg_g + G.c2w1[kmax + 1] * rg[an]);
    } else {
      rw[a] = real(0.0);
      w[a] = real(0.0);
    }
    eth[a] = ein_g + pre_g / rho_g;
  }
};

// ----------------------------------------------------------------------------
// momentum advection, Coriolis, projection (mod_src.py:96-497, kernels/advconvmom.py)
// out[0..2]: momentum tendencies; out[3]: the radial part gwc at full levels
// (the half-level w tendency c2w0*gwc(k) + c2w1*gwc(k-1) is formed by its user)
// ----------------------------------------------------------------------------
// the pole centres (the regional points run as AdvMomC)
struct AdvMomP {
  Dims d; Consts c; Geo G;
  const real* prog;
  const real* diag;
  real* out;
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p) || !p.pole || p.v != 0) return;
    const long NF = d.NF, a = p.a, ks = p.ks;
    const int kmin = d.kmin, kmax = d.kmax, k = p.k;
    if (k < kmin || k > kmax) {
      for (int q = 0; q < 4; ++q) out[q * NF + a] = real(0.0);
      return;
    }
    const real R = c.RADIUS;
    const real* rw = prog + 4 * NF;
    const real* wd = diag + I_W * NF;
    auto pos = [&](int m, real* x3) {
      for (int q = 0; q < 3; ++q) x3[q] = G.gx_pl[(m * 2 + p.lp) * 3 + q];
    };
    // merged velocity v + w_full r/|r| at address b (level kk) with position x
    auto vv3 = [&](long b, int kk, const real* x3, real* o) {
      const real wc = G.cfact[kk] * wd[b + ks] + G.dfact[kk] * wd[b];
      for (int q = 0; q < 3; ++q) o[q] = diag[(I_VX + q) * NF + b] + wc * x3[q] / R;
    };
    real x0[3], vvm0[3], div[3];
    pos(0, x0);
    // divergence of rhogv * vv_q: the directions summed per point, as in div_pl
    for (int m = 0; m < 6; ++m) {
      real xm[3], vv[3];
      pos(m, xm);
      vv3(a + m, k, xm, vv);
      if (m == 0)
        for (int q = 0; q < 3; ++q) vvm0[q] = vv[q];
      const real fx0 = prog[1 * NF + a + m], fy0 = prog[2 * NF + a + m], fz0 = prog[3 * NF + a + m];
      const real* cc = G.cdiv_pl + (m * 2 + p.lp) * 3;
      for (int q = 0; q < 3; ++q) {
        const real pv = cc[0] * (fx0 * vv[q] * real(1.0)) + cc[1] * (fy0 * vv[q] * real(1.0)) +
                        cc[2] * (fz0 * vv[q] * real(1.0));
        div[q] = (m == 0) ? pv : div[q] + pv;
      }
    }
    // vertical fluxes at the half levels k+1 and k (zero at kmin and kmax+1)
    real hi[3] = {real(0.0), real(0.0), real(0.0)}, lo[3] = {real(0.0), real(0.0), real(0.0)};
    if (k + 1 <= kmax) {
      real up[3];
      vv3(a + ks, k + 1, x0, up);
      for (int q = 0; q < 3; ++q)
        hi[q] = real(0.0) * real(1.0) + rw[a + ks] * (G.afact[k + 1] * up[q] + G.bfact[k + 1] * vvm0[q]) * real(1.0);
    }
    if (k >= kmin + 1) {
      real dn[3];
      vv3(a - ks, k - 1, x0, dn);
      for (int q = 0; q < 3; ++q)
        lo[q] = real(0.0) * real(1.0) + rw[a] * (G.afact[k] * vvm0[q] + G.bfact[k] * dn[q]) * real(1.0);
    }
    real dvv[3];
    for (int q = 0; q < 3; ++q) dvv[q] = -div[q] - (hi[q] - lo[q]) * G.rdgz[k];
    const real gxc = x0[0] / R, gyc = x0[1] / R, gzc = x0[2] / R;
    const real rh = prog[a];
    const real dx = dvv[0] - (-real(2.0) * rh * (c.OHM * vvm0[1]));
    const real dy = dvv[1] - (real(2.0) * rh * (c.OHM * vvm0[0]));
    const real dz = dvv[2];
    const real prd = dx * gxc + dy * gyc + dz * gzc;
    out[0 * NF + a] = dx - prd * gxc;
    out[1 * NF + a] = dy - prd * gyc;
    out[2 * NF + a] = dz - prd * gzc;
    out[3 * NF + a] = prd * c.ALPHA;
  }
};

// ----------------------------------------------------------------------------
// hyperdiffusion passes (mod_numfilter.py:1125-1264)
// ----------------------------------------------------------------------------
template <int LAST>
struct HDiffPassP {
  static constexpr const char* kName = LAST ? "hdiff_pass2" : "hdiff_pass1";
  Dims d; Consts c; Geo G;
  const real* in[6];
  real* out[6];
  const real* rhog;
  // first pass: FP64 k-profile subtracted from input f (tem - tem_bs,
  // rho - rho_bs, mod_numfilter.py:1068-1076), or none
  const double* sub[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
  const int* cs = nullptr;   // second pass: source columns of the inputs' halo values
  NH_HD real input(int f, long b, int k) const {
    return sub[f] ? (real)((double)in[f][b] - sub[f][k]) : in[f][b];
  }
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p) || !p.pole || p.v != 0) return;
    if (!LAST) {
      at(p, [&](int f, long b) { return input(f, b, p.k); });
      return;
    }
    const long a = p.a;
    auto pa = [&](int v) { return src_pole(d, cs, p.lp, v, p.k); };
    for (int q = 0; q < 6; ++q) {
      real r;
      if (q >= 4) {
        const real fac = (q == 4) ? c.CVdry : c.HDIFF_FACT_RHO;
        const real* rg = rhog;
        const real gam = c.GAMMA_H;
        auto kh = [rg, fac, gam](long xx) { return rg[xx] * fac * gam; };
        r = diffusion_pl(G, p.lp, in[q], kh, a, pa);
      } else {
        r = lap_pl_at(G, p.lp, in[q], pa);
      }
      out[q][a] = -r;
    }
  }
  // first pass: minus the Laplacian of each field, fields read through ld(f, address)
  template <class LD>
  NH_HD void at(const Pt& p, LD ld) const {
    const long a = p.a;
    for (int q = 0; q < 6; ++q) {
      real r = real(0.0);
      for (int v = 0; v < 6; ++v) {
        const real pv = G.clap_pl[v * 2 + p.lp] * ld(q, a + v);
        r = (v == 0) ? pv : r + pv;
      }
      out[q][a] = -r;
    }
  }
};

// ----------------------------------------------------------------------------
// 3-D divergence damping (kernels/oprt3ddivdamp.py, oprtdivdamp.py, divdamppostcomm.py)
// ----------------------------------------------------------------------------
struct DivDamp1P {
  static constexpr const char* kName = "divdamp_3d";
  Dims d; Consts c; Geo G;
  const real *rvx, *rvy, *rvz, *rw;
  real* out[3];
  const int* cs;   // source columns of the inputs' halo values (read at the poles)
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p) || !p.pole || p.v != 0) return;
    const int kmin = d.kmin, kmax = d.kmax, k = p.k;
    const long ks = p.ks, a = p.a;
    if (k < kmin || k > kmax) {
      for (int q = 0; q < 3; ++q) out[q][a] = real(0.0);
      return;
    }
    auto rwv = [&](long aa, int kk) { return (kk >= kmin + 1 && kk <= kmax) ? (real(0.0) * real(1.0) + rw[aa] * real(1.0)) : real(0.0); };
    real sclt[5];
    auto pa = [&](int v, int kk) { return src_pole(d, cs, p.lp, v, kk); };
    const real* vv[3] = {rvx, rvy, rvz};
    for (int v = 1; v <= 5; ++v) {
      const int vp = (v == 5) ? 1 : v + 1;
      real s = real(0.0);
      for (int dd = 0; dd < 3; ++dd) {
        const real* cI = G.cintp_pl + ((v * 2 + p.lp) * 3 + dd) * 3;
        const real t0 = cI[0] * (vv[dd][a] * real(1.0)), t1 = cI[1] * (vv[dd][pa(v, k)] * real(1.0)),
                     t2 = cI[2] * (vv[dd][pa(vp, k)] * real(1.0));
        s = (dd == 0) ? (t0 + t1 + t2) : (s + t0 + t1 + t2);
      }
      const real up = (rwv(a + ks, k + 1) + rwv(pa(v, k + 1), k + 1) + rwv(pa(vp, k + 1), k + 1));
      const real dn = (rwv(a, k) + rwv(pa(v, k), k) + rwv(pa(vp, k), k));
      sclt[v - 1] = s + (up - dn) / real(3.0) * G.rdgz[k];
    }
    for (int dd = 0; dd < 3; ++dd) {
      real row = real(0.0);
      for (int v = 1; v <= 5; ++v) {
        const int vm = (v == 1) ? 5 : v - 1;
        const real cb = G.cdiff_pl[(v * 2 + p.lp) * 3 + dd] * (sclt[vm - 1] + sclt[v - 1]);
        row = (v == 1) ? cb : row + cb;
      }
      out[dd][a] = row;
    }
  }
};

struct DivDamp2P {
  static constexpr const char* kName = "divdamp_post";
  Dims d; Consts c; Geo G;
  const real* in[3];
  real* out[3];
  const int* cs;   // source columns of the inputs' halo values (read at the poles)
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p) || !p.pole || p.v != 0) return;
    const long a = p.a;
    const int kmin = d.kmin, kmax = d.kmax, k = p.k;
    const real R = c.RADIUS;
    real o[3];
    if (k < kmin || k > kmax) {
      o[0] = o[1] = o[2] = real(0.0);
    } else {
      real sclt[5];
      for (int v = 1; v <= 5; ++v) {
        const int vp = (v == 5) ? 1 : v + 1;
        real s = real(0.0);
        for (int dd = 0; dd < 3; ++dd) {
          const real* cI = G.cintp_pl + ((v * 2 + p.lp) * 3 + dd) * 3;
          const real t0 = cI[0] * (-in[dd][a]), t1 = cI[1] * (-in[dd][src_pole(d, cs, p.lp, v, k)]),
                     t2 = cI[2] * (-in[dd][src_pole(d, cs, p.lp, vp, k)]);
          s = (dd == 0) ? (t0 + t1 + t2) : (s + t0 + t1 + t2);
        }
        sclt[v - 1] = s;
      }
      for (int dd = 0; dd < 3; ++dd) {
        real row = real(0.0);
        for (int v = 1; v <= 5; ++v) {
          const int vm = (v == 1) ? 5 : v - 1;
          const real cb = G.cdiff_pl[(v * 2 + p.lp) * 3 + dd] * (sclt[vm - 1] + sclt[v - 1]);
          row = (v == 1) ? cb : row + cb;
        }
        o[dd] = row;
      }
    }
    const real gd[3] = {c.ALPHA_D * o[0], c.ALPHA_D * o[1], c.ALPHA_D * o[2]};
    const real gx = G.gx_pl[p.lp * 3 + 0], gy = G.gx_pl[p.lp * 3 + 1], gz = G.gx_pl[p.lp * 3 + 2];
    const real prd = gd[0] * gx / R + gd[1] * gy / R + gd[2] * gz / R;
    out[0][a] = gd[0] - prd * gx / R;
    out[1][a] = gd[1] - prd * gy / R;
    out[2][a] = gd[2] - prd * gz / R;
  }
};

// ----------------------------------------------------------------------------
// large-step source terms of the small steps and the tridiagonal coefficients
// (mod_vi.py:132-881, kernels/vimatrix.py:67-136); column quantities of levels
// k-1..k+1 are recomputed per point
// ----------------------------------------------------------------------------
struct ViPath0P {
  static constexpr const char* kName = "vi_path0";
  Dims d; Consts c; Geo G;
  double dt;
  const real* prog;
  const real* diag;
  const real* eth;
  const real* gadv;   // 3 momentum tendencies + gwc at full levels
  const real* vt[6];
  const real* dd[3];
  real* gT;
  double* Mc; double* Mu; double* Ml;   // FP64 in every form
  real* getot;
  real* frhog;
  // the pole centres (the regional points run as ViPath0C)
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p) || !p.pole || p.v != 0) return;
    const long sh = (p.k == d.kmin) ? p.ks : 0;
    at(p, [&](int f, long b) {
      return f < 3 ? prog[(long)(1 + f) * d.NF + b] : f == 3 ? eth[b] : diag[I_PRE * d.NF + b + sh];
    });
  }
  // ld(f, address): rhogvx, rhogvy, rhogvz, eth at the point's level, the
  // pressure at the level of its gradient (kmin -> kmin+1)
  template <class LD>
  NH_HD void at(const Pt& p, LD ld) const {
    const long NF = d.NF, ks = p.ks, a = p.a;
    const int kmin = d.kmin, kmax = d.kmax, k = p.k;
    const real R = c.RADIUS;
    const real* rg = prog;
    const real* rw = prog + 4 * NF;
    const real* pre = diag + I_PRE * NF;
    const long b = a - (long)k * ks;     // column base
    auto lev = [&](int kk) { return b + (long)kk * ks; };
    // the column window k-2 .. k+1 of rhog, pressure, eth and rhogw, loaded
    // first at levels clamped into range (a clamped value is never used: the
    // level tests below are the reference's), read through selects
    real Wrg[4], Wpr[4], Wet[4], Wrw[4];
    for (int jw = 0; jw < 4; ++jw) {
      int kw = k - 2 + jw;
      kw = (kw < 0) ? 0 : ((kw > d.kall - 1) ? d.kall - 1 : kw);
      const long aw = lev(kw);
      Wrg[jw] = rg[aw];
      Wpr[jw] = pre[aw];
      Wet[jw] = eth[aw];
      Wrw[jw] = rw[aw];
    }
    auto win = [&](const real* W, int kk) {
      const int jw = kk - k + 2;
      return (jw <= 0) ? W[0] : (jw == 1) ? W[1] : (jw == 2) ? W[2] : W[3];
    };
    auto RG = [&](int kk) { return win(Wrg, kk); };
    auto PR = [&](int kk) { return win(Wpr, kk); };
    // pregd = (pre - pre_bs) GSGAM2, rhogd = (rho - rho_bs) GSGAM2 with the basic
    // state in FP64 (mod_dynamics.py:1056-1057); GSGAM2 = 1
    auto PRD = [&](int kk) { return (real)((double)PR(kk) - G.pre_bs[kk]) * real(1.0); };
    auto RGD = [&](int kk) { return (real)((double)(RG(kk) / real(1.0)) - G.rho_bs[kk]) * real(1.0); };
    auto ET = [&](int kk) { return win(Wet, kk); };
    auto RW = [&](int kk) { return win(Wrw, kk); };
    auto rhog_h = [&](int kk) {
      const int k2 = (kk < kmin) ? kmin : kk;
      return G.c2w0[k2] * RG(k2) + G.c2w1[k2] * RG(k2 - 1);
    };
    auto dpgw = [&](int kk) {
      return (kk >= kmin + 1 && kk <= kmax) ? real(1.0) * (PRD(kk) * real(1.0) - PRD(kk - 1) * real(1.0)) * G.rdgzh[kk] : real(0.0);
    };
    auto dbuo = [&](int kk) {
      return (kk >= kmin + 1 && kk <= kmax)
                 ? -c.GRAV * (G.c2w0[kk] * RGD(kk) + G.c2w1[kk] * RGD(kk - 1))
                 : real(0.0);
    };
    auto gzt = [&](int kk) { return c.GRAV - (dpgw(kk) - dbuo(kk)) / rhog_h(kk); };
    auto pwh = [&](int kk) { return -gzt(kk) * RW(kk); };
    const real gx = G.gx_pl[p.lp * 3 + 0], gy = G.gx_pl[p.lp * 3 + 1], gz = G.gx_pl[p.lp * 3 + 2];
    const real Kh = c.GAMMA_H;
    // hyperdiffusion tendency + momentum advection = large-step tendency g0
    const real rgk = RG(k);
    real fvx = -(vt[0][a] * Kh + real(0.0)) * rgk;
    real fvy = -(vt[1][a] * Kh + real(0.0)) * rgk;
    real fvz = -(vt[2][a] * Kh + real(0.0)) * rgk;
    const real rgh = (k >= kmin) ? G.c2w0[k] * rgk + G.c2w1[k] * RG(k - 1) : real(0.0);
    const real fw = -(vt[3][a] * Kh + real(0.0)) * rgh;
    const real fe = -(vt[4][a] + real(0.0));
    const real fr = -(vt[5][a] + real(0.0));
    {
      const real prd = fvx * gx / R + fvy * gy / R + fvz * gz / R;
      fvx = fvx - prd * gx / R; fvy = fvy - prd * gy / R; fvz = fvz - prd * gz / R;
    }
    const real gadv_w = (k > kmin && k <= kmax) ? (G.c2w0[k] * gadv[3 * NF + a] + G.c2w1[k] * gadv[3 * NF + a - ks]) : real(0.0);
    real g0[6];
    g0[0] = real(0.0) + fr;
    g0[1] = gadv[0 * NF + a] + fvx;
    g0[2] = gadv[1 * NF + a] + fvy;
    g0[3] = gadv[2 * NF + a] + fvz;
    g0[4] = gadv_w + fw;
    g0[5] = real(0.0) + fe;
    getot[a] = g0[5];
    frhog[a] = g0[0];
    real drhog = real(0.0), drhoge = real(0.0), pw = real(0.0);
    real dpg[3] = {real(0.0), real(0.0), real(0.0)};
    if (k >= kmin && k <= kmax) {
      // div(rhogv), div(rhogv eth)
      real dvs[2];
      hdiv_multi<2>(G, p, [&](int, long bn, real (*v)[3]) {
        const real e = ld(3, bn);
        const real r3[3] = {ld(0, bn), ld(1, bn), ld(2, bn)};
        for (int q = 0; q < 3; ++q) {
          v[0][q] = r3[q] * real(1.0);
          v[1][q] = r3[q] * e * real(1.0);
        }
      }, dvs);
      const real hd = dvs[0];
      const real vmh_hi = (k + 1 <= kmax) ? real(0.0) * real(1.0) + real(1.0) * RW(k + 1) * real(1.0) : real(0.0);
      const real vmh_lo = (k >= kmin + 1) ? real(0.0) * real(1.0) + real(1.0) * RW(k) * real(1.0) : real(0.0);
      drhog = -hd - (vmh_hi - vmh_lo) * G.rdgz[k];
      const real he = dvs[1];
      const real ws_hi = (k + 1 <= kmax)
          ? real(0.0) * real(1.0) + real(1.0) * (RW(k + 1) * (G.afact[k + 1] * ET(k + 1) + G.bfact[k + 1] * ET(k))) * real(1.0) : real(0.0);
      const real ws_lo = (k >= kmin + 1)
          ? real(0.0) * real(1.0) + real(1.0) * (RW(k) * (G.afact[k] * ET(k) + G.bfact[k] * ET(k - 1))) * real(1.0) : real(0.0);
      drhoge = -he - (ws_hi - ws_lo) * G.rdgz[k];
      // the gradient of pregd at the level the pressure is read from (kmin -> kmin+1)
      const int kg = (k == kmin) ? kmin + 1 : k;
      presgrad_ld(p, [&](int f, long b) {
        return f == 4 ? (real)((double)ld(4, b) - G.pre_bs[kg]) * real(1.0) : ld(f, b);
      }, R, dpg);
      pw = diag[I_VX * NF + a] * dpg[0] + diag[I_VY * NF + a] * dpg[1] + diag[I_VZ * NF + a] * dpg[2]
         + G.w2c0[k] * pwh(k + 1) + G.w2c1[k] * pwh(k);
    }
    gT[0 * NF + a] = g0[0] + drhog;
    gT[1 * NF + a] = g0[1] - dpg[0] + dd[0][a] + real(0.0);
    gT[2 * NF + a] = g0[2] - dpg[1] + dd[1][a] + real(0.0);
    gT[3 * NF + a] = g0[3] - dpg[2] + dd[2][a] + real(0.0);
    gT[4 * NF + a] = g0[4] + real(0.0) * c.ALPHA - dpgw(k) + dbuo(k);
    gT[5 * NF + a] = g0[5] + drhoge + pw;
    if (k >= kmin + 1 && k <= kmax) {
      // tridiagonal coefficients, FP64 in every form: the column quantities of
      // levels k-1..k+1 again, from the stored fields, in double
      const VProf<double>& V = G.v64;
      const ConstsT<double>& C = c.d;
      auto rhog_h64 = [&](int kk) {
        const int k2 = (kk < kmin) ? kmin : kk;
        return V.c2w0[k2] * (double)RG(k2) + V.c2w1[k2] * (double)RG(k2 - 1);
      };
      auto eth_h64 = [&](int kk) {
        const int k2 = (kk < kmin) ? kmin : kk;
        return V.afact[k2] * (double)ET(k2) + V.bfact[k2] * (double)ET(k2 - 1);
      };
      auto dpgw64 = [&](int kk) {
        return (kk >= kmin + 1 && kk <= kmax)
                   ? 1.0 * (((double)PR(kk) - G.pre_bs[kk]) * 1.0 - ((double)PR(kk - 1) - G.pre_bs[kk - 1]) * 1.0)
                         * V.rdgzh[kk]
                   : 0.0;
      };
      auto dbuo64 = [&](int kk) {
        return (kk >= kmin + 1 && kk <= kmax)
                   ? -C.GRAV * (V.c2w0[kk] * (((double)RG(kk) / 1.0 - G.rho_bs[kk]) * 1.0) +
                                V.c2w1[kk] * (((double)RG(kk - 1) / 1.0 - G.rho_bs[kk - 1]) * 1.0))
                   : 0.0;
      };
      auto gzt64 = [&](int kk) { return C.GRAV - (dpgw64(kk) - dbuo64(kk)) / rhog_h64(kk); };
      const double GCVovR = C.GRAV * C.CVdry / C.Rdry;
      const double ACVovRt2 = C.ALPHA * C.CVdry / C.Rdry / (dt * dt);
      const double Ca = (1.0 * V.rdgz[k] + 1.0 * V.rdgz[k - 1]) * 1.0;
      const double Cb = V.dfact[k] - V.cfact[k - 1];
      const double Cu1 = 1.0 * V.rdgz[k] * 1.0;
      const double Cu2 = 1.0 * 1.0 * GCVovR;
      const double Cl1 = 1.0 * V.rdgz[k] * 1.0;
      const double Cl2 = 1.0 * 1.0 * GCVovR;
      Mc[a] = ACVovRt2 / 1.0 + V.rdgzh[k] * (Ca * eth_h64(k) - Cb * (gzt64(k) + GCVovR));
      Mu[a] = -V.rdgzh[k] * (Cu1 * eth_h64(k + 1) + V.cfact[k] * (gzt64(k + 1) + Cu2));
      Ml[a] = -V.rdgzh[k] * (Cl1 * eth_h64(k - 1) - V.dfact[k - 1] * (gzt64(k - 1) + Cl2));
    }
  }
  // horizontal pressure-gradient force at the pole centre with the first-layer
  // remedy, the pressure of the gradient's level read as ld(4, .)
  template <class LD>
  NH_HD void presgrad_ld(const Pt& p, LD ld, real R, real o[3]) const {
    const long a = p.a;
    real gr[3];
    for (int dd2 = 0; dd2 < 3; ++dd2) {
      real acc = real(0.0);
      for (int v = 0; v < 6; ++v) {
        const real pv = G.cgrad_pl[(v * 2 + p.lp) * 3 + dd2] * (ld(4, a + v) * real(1.0) * real(1.0));
        acc = (v == 0) ? pv : acc + pv;
      }
      gr[dd2] = acc;
    }
    for (int q = 0; q < 3; ++q) gr[q] = gr[q] + real(0.0);
    const real gx = G.gx_pl[(0 * 2 + p.lp) * 3 + 0];
    const real gy = G.gx_pl[(0 * 2 + p.lp) * 3 + 1];
    const real gz = G.gx_pl[(0 * 2 + p.lp) * 3 + 2];
    const real prd = gr[0] * gx / R + gr[1] * gy / R + gr[2] * gz / R;
    o[0] = gr[0] - prd * gx / R;
    o[1] = gr[1] - prd * gy / R;
    o[2] = gr[2] - prd * gz / R;
  }
};

// The time-mean mass fluxes of a stage, accumulated over its small steps.  A
// small step reads its input state anyway, which is the previous one's output,
// so the sums are read and written every second small step with both steps'
// terms (two), in the order one step at a time adds them; the first time they
// start from the large-step state itself (in).  Null out: nothing this step.
// Against one accumulation per small step of every stage (the tracer transport
// reads the last stage's only), 80 of the 960 field passes of a step are gone.
struct MeanFlux {
  const real* in = nullptr;   // rhog, rhogvx, rhogvy, rhogvz, rhogw
  real* out = nullptr;
  bool two = false;
  NH_HD real add(real sum, real prev, real cur, real weight) const {
    if (two) sum = sum + prev * weight;
    return sum + cur * weight;
  }
};

// total specific energy of the large-step state; pm (null elsewhere): the start of the
// time-mean fluxes in the last stage under a halo map that leaves columns out, where
// the copy stands for the fill (a full map's small steps start from prog itself)
struct EthTotPMP {
  static constexpr const char* kName = "ethtot_mean";
  Dims d; Consts c; Geo G;
  const real* prog;
  const real* eth;
  real* ethtot;
  real* pm;
  // the column values are read first (levels k-1, k+1 clamped into range;
  // rhogkin_k uses them only where they exist), then the stores
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p)) return;
    const long NF = d.NF, a = p.a, ks = p.ks;
    const int k = p.k;
    const long am = (k > 0) ? a - ks : a, ap = (k < d.kall - 1) ? a + ks : a;
    const real rg[3] = {prog[am], prog[a], prog[ap]};
    const real rv[3] = {prog[NF + a], prog[2 * NF + a], prog[3 * NF + a]};
    const real rw[2] = {prog[4 * NF + a], prog[4 * NF + ap]};
    const real e = eth[a];
    auto get = [&](int kk, int q) {
      if (q == 0) return rg[kk - k + 1];
      if (q == 4) return rw[kk - k];
      return rv[q - 1];
    };
    const real kin0 = rhogkin_k(G, d.kmin, d.kmax, k, get);
    ethtot[a] = e + kin0 / rg[1] + G.phi[k];
    if (pm) {
      pm[a] = rg[1];
      for (int q = 0; q < 3; ++q) pm[(1 + q) * NF + a] = rv[q];
      pm[4 * NF + a] = rw[0];
    }
  }
};

// ----------------------------------------------------------------------------
// small step path1 (kernels/vipath1.py:68-160); the ghost rows recompute the
// nearest physical level
// ----------------------------------------------------------------------------
struct Path1P {
  static constexpr const char* kName = "vi_path1";
  // the split rhoge is read on the stencil, at the level whose pressure
  // gradient the point needs (stage_shift levels above the point's own).  The
  // regional points run as column tiles (Path1C), this form the pole centres
  Dims d; Consts c; Geo G;
  real dt, rweight;
  const real* prog;
  const real* ps[6];
  const real* gT;
  const real* dd[3];
  real* dv[3];
  MeanFlux mf;
  const int* cs;   // source columns of the split rhoge's halo values
  // level of the gradient for a point at level k: kmin -> kmin+1 (first-layer
  // remedy); the ghost rows use the nearest physical level's value, kmin-1 ->
  // kmin (gradient at kmin+1) and kmax+1 -> kmax
  NH_HD int stage_shift(int k) const {
    const int kmin = d.kmin, kmax = d.kmax;
    if (k == kmin || k == kmin - 1) return kmin + 1 - k;
    if (k == kmax + 1) return -1;
    return 0;
  }
  // a pole level
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p) || !p.pole || p.v != 0) return;
    at(p, [&](int v) { return ps[I_RHOGE][src_pole(d, cs, p.lp, v, p.k + stage_shift(p.k))]; });
  }
  // momentum of the small step at level k (column address a); the gradient of
  // the split pressure comes through grad(dir)
  template <class GR>
  NH_HD void level(const Pt& p, long a, GR grad, real out[3]) const {
    const long NF = d.NF;
    const real R = c.RADIUS;
    real gr[3];
    for (int dd2 = 0; dd2 < 3; ++dd2) gr[dd2] = grad(dd2);
    for (int q = 0; q < 3; ++q) gr[q] = gr[q] + real(0.0);
    real Pg[3];
    const real gx = G.gx_pl[p.lp * 3 + 0], gy = G.gx_pl[p.lp * 3 + 1], gz = G.gx_pl[p.lp * 3 + 2];
    const real prd = gr[0] * gx / R + gr[1] * gy / R + gr[2] * gz / R;
    Pg[0] = gr[0] - prd * gx / R; Pg[1] = gr[1] - prd * gy / R; Pg[2] = gr[2] - prd * gz / R;
    for (int q = 0; q < 3; ++q) {
      const real drv = gT[(1 + q) * NF + a] - Pg[q] + dd[q][a] + real(0.0);
      out[q] = ps[1 + q][a] + drv * dt;
    }
  }
  // ld(v): split rhoge of pole point v at the gradient's level
  template <class LD>
  NH_HD void at(const Pt& p, LD ld) const {
    const long NF = d.NF, a = p.a, ks = p.ks;
    const int kmin = d.kmin, kmax = d.kmax, k = p.k;
    const real RovCV = c.Rdry / c.CVdry;
    auto grad = [&](int dd2) {
      real acc = real(0.0);
      for (int v = 0; v < 6; ++v) {
        const real pv = G.cgrad_pl[(v * 2 + p.lp) * 3 + dd2] * ((ld(v) * RovCV) * real(1.0) * real(1.0));
        acc = (v == 0) ? pv : acc + pv;
      }
      return acc;
    };
    real v[3];
    if (k >= kmin && k <= kmax) {
      level(p, a, grad, v);
    } else {
      // free-slip top / rigid bottom, scaled by the large-step density
      const bool top = (k == kmax + 1);
      const long an = top ? a - ks : a + ks;
      real vn[3];
      level(p, an, grad, vn);
      const real* rg = prog;
      for (int q = 0; q < 3; ++q) v[q] = top ? real(1.0) * (vn[q] / rg[an]) * rg[a] : -real(1.0) * (vn[q] / rg[an]) * rg[a];
    }
    for (int q = 0; q < 3; ++q) {
      const real pmq = mf.out ? mf.in[(1 + q) * NF + a] : real(0.0);
      dv[q][a] = v[q];
      if (mf.out) mf.out[(1 + q) * NF + a] = mf.add(pmq, mf.two ? ps[1 + q][a] : real(0.0), v[q], rweight);
    }
  }
};

// ----------------------------------------------------------------------------
// small step vi_main, horizontal part: the three flux divergences of the new
// momentum (mod_vi.py:1925-2432, kernels/vimain.py:127-262)
//   hv[0] = div(dv), hv[1] = vertical-pressure source gpre, hv[2] = div((prog + dv) * ethtot)
// ----------------------------------------------------------------------------
struct ViMainH {
  static constexpr const char* kName = "vi_main_h";
  Dims d; Consts c; Geo G;
  const real* prog;
  const real* dv[3];
  const real* eth;
  const real* ethtot;
  const real* gT;
  real* hv[3];
  const int* cs;   // source columns of dv's halo values
  // field f at a point of the stencil: address a, of dv am (its halo values' source)
  NH_HD real stage_val(int f, long a, long am) const {
    return f < 3 ? dv[f][am] : (f == 3 ? eth[a] : (f == 4 ? ethtot[a] : prog[(long)(f - 4) * d.NF + a]));
  }
  // a pole level (the regional points run as ViMainHC)
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p) || !p.pole || p.v != 0) return;
    at(p, [&](int f, long b) { return stage_val(f, b, src_pole(d, cs, p.lp, (int)(b - p.a), p.k)); });
  }
  // ld(f, address): field f of the stencil set at an address of the point's stencil
  template <class LD>
  NH_HD void at(const Pt& p, LD ld) const {
    const int kmin = d.kmin, kmax = d.kmax, k = p.k;
    if (k < kmin || k > kmax) return;
    const long NF = d.NF, a = p.a;
    // div(dv), div(dv eth), div((prog + dv) ethtot)
    real dvs[3];
    hdiv_multi<3>(G, p, [&](int, long b, real (*v)[3]) {
      const real e = ld(3, b), et = ld(4, b);
      for (int q = 0; q < 3; ++q) {
        const real dq = ld(q, b);
        v[0][q] = dq * real(1.0);
        v[1][q] = dq * e * real(1.0);
        v[2][q] = (ld(5 + q, b) + dq) * et * real(1.0);
      }
    }, dvs);
    const real divs1 = dvs[0], he = dvs[1], hd = dvs[2];
    const real drhoge = -he - (real(0.0) - real(0.0)) * G.rdgz[k];
    const real grhoge1 = gT[5 * NF + a] + drhoge;
    hv[0][a] = divs1;
    hv[1][a] = grhoge1 * c.Rdry / c.CVdry;
    hv[2][a] = hd;
  }
};

// vertical part, one thread per compute column: source vector of the
// tridiagonal rhogw system and the Thomas sweeps, streamed in k with the
// previous level kept in registers (kernels/virhowsolver.py:42-120).  FP64 in
// every form: the field values are widened on load.  NK > 0 is the number of
// unknowns (kmax - kmin) fixed at compile time: u and gamma of the forward
// sweep then stay in registers; NK = 0 keeps them in the FP64 scratch U, Gm.
// The backward sweep writes the new rhogw split to out on every level.
template <int NK>
struct ViMainV {
  static constexpr const char* kName = "vi_main_v";
  static constexpr int kUnroll = NK > 0 ? NK : 4;
  // rows in flight (the registers of the z40 form leave room for one of 8-byte fields)
  static constexpr int kAhead = (NK > 0 && sizeof(real) == 8) ? 1 : 3;
  Dims d; Consts c; Geo G;
  double dt;
  const real* ps[6];
  const real* gT;
  const double* Mc; const double* Mu; const double* Ml;
  const real* hv[3];
  double* U;
  double* Gm;
  real* out;
  NH_HD void operator()(long t) const {
    Cell cl = cell_of(d, t);
    if (cl.pole ? cl.v != 0 : !cl.inner) return;
    const long NF = d.NF, ks = cl.ks, b = cl.base;
    const int kmin = d.kmin, kmax = d.kmax;
    const VProf<double>& V = G.v64;
    const ConstsT<double>& C = c.d;
    const double RovCV = C.Rdry / C.CVdry;
    const double CVovRt2 = C.CVdry / C.Rdry / (dt * dt);
    const real* __restrict__ pg = ps[I_RHOG];
    const real* __restrict__ pw = ps[I_RHOGW];
    const real* __restrict__ pe = ps[I_RHOGE];
    const real* __restrict__ gT0 = gT;
    const real* __restrict__ gT4 = gT + 4 * NF;
    const real* __restrict__ hv0 = hv[0];
    const real* __restrict__ hv1 = hv[1];
    const double* __restrict__ mc = Mc;
    const double* __restrict__ mu = Mu;
    const double* __restrict__ ml = Ml;
    double* __restrict__ Uo = U;
    double* __restrict__ Go = Gm;
    real* __restrict__ Xo = out;
    const int N = (NK > 0) ? NK : kmax - kmin;
    double ub[NK > 0 ? NK : 1], gb[NK > 0 ? NK : 1];
    // what a level's row needs, loaded kAhead levels before it is formed: the
    // sweep is a serial chain of few waves per SIMD (2.7 at gl07, 0.2 at gl05), so
    // a row must not wait for its loads.  At gl06 the scratch form (NK = 0) 139 -> 75 us
    // mixed with 57 levels, 77 -> 49 FP64 with 33; the z40 form is at the HBM rate
    // at gl07 (90 us mixed, 130 FP64) and at the chain's latency at gl05 (20 us).
    struct Row {
      real pe, hv1, pg, gT0, hv0, gT4, pw;
      double mc, mu, ml;
    };
    auto load = [&](int n) {
      const long a = b + (long)(kmin + 1 + (n < N ? n : N - 1)) * ks;
      return Row{ldc(pe + a), ldc(hv1 + a), ldc(pg + a), ldc(gT0 + a), ldc(hv0 + a), ldc(gT4 + a), ldc(pw + a),
                 ldc(mc + a), ldc(mu + a), ldc(ml + a)};
    };
    Row ahead[kAhead];
    for (int q = 0; q < kAhead; ++q) ahead[q] = load(q);
    // level k-1 values, starting at kmin
    long am = b + (long)kmin * ks;
    double pe_m = pe[am], hv1_m = hv1[am], pg_m = pg[am];
    double gr_m = (double)gT0[am] + (-(double)hv0[am] - (0.0 - 0.0) * V.rdgz[kmin]);
    double beta = 0.0, u_prev = 0.0, mu_m = 0.0;
#pragma unroll kUnroll
    for (int n = 0; n < N; ++n) {
      const int k = kmin + 1 + n;
      const long a = am + ks;
      const Row r = ahead[0];
      for (int q = 0; q + 1 < kAhead; ++q) ahead[q] = ahead[q + 1];
      ahead[kAhead - 1] = load(n + kAhead);
      const double pe_k = r.pe, hv1_k = r.hv1, pg_k = r.pg;
      const double gr_k = (double)r.gT0 + (-(double)r.hv0 - (0.0 - 0.0) * V.rdgz[k]);
      const double sw = (double)r.gT4 + 0.0 * C.ALPHA;
      const double A = ((double)r.pw * C.ALPHA + dt * sw) * 1.0;
      const double B = (pe_k * RovCV + dt * hv1_k) * 1.0 - (pe_m * RovCV + dt * hv1_m) * 1.0;
      const double Cc = (pg_k + dt * gr_k) * 1.0 * V.afact[k] + (pg_m + dt * gr_m) * 1.0 * V.bfact[k];
      double S = (A - B * dt * V.rdgzh[k] - Cc * dt * C.GRAV) * CVovRt2;
      const double mc_k = r.mc, ml_k = r.ml, mu_k = r.mu;
      if (n == 0) S = S - ml_k * (0.0 * 1.0);
      if (n == N - 1) S = S - mu_k * (-0.0 * 1.0);
      double u;
      if (n == 0) {
        beta = mc_k;
        u = S / beta;
      } else {
        const double gm = mu_m / beta;
        beta = mc_k - ml_k * gm;
        u = (S - ml_k * u_prev) / beta;
        if (NK > 0) gb[NK > 0 ? n : 0] = gm;
        else Go[a] = gm;
      }
      if (NK > 0) ub[NK > 0 ? n : 0] = u;
      else Uo[a] = u;
      u_prev = u;
      mu_m = mu_k;
      pe_m = pe_k; hv1_m = hv1_k; pg_m = pg_k; gr_m = gr_k;
      am = a;
    }
    // backward sweep
    long a = b + (long)kmax * ks;
    double xv = u_prev;
    Xo[a] = (real)(xv * 1.0);
    if (NK > 0) {
#pragma unroll
      for (int n = N - 2; n >= 0; --n) {
        a -= ks;
        xv = ub[NK > 0 ? n : 0] - gb[NK > 0 ? n + 1 : 0] * xv;
        Xo[a] = (real)(xv * 1.0);
      }
    } else {
      double gm_next = Go[a];
#pragma unroll 4
      for (int n = N - 2; n >= 0; --n) {
        a -= ks;
        xv = Uo[a] - gm_next * xv;
        gm_next = Go[a];
        Xo[a] = (real)(xv * 1.0);
      }
    }
    Xo[b + (long)kmin * ks] = (real)(0.0 * 1.0);
    Xo[b + (long)(kmax + 1) * ks] = (real)(-0.0 * 1.0);
    Xo[b + (long)(kmin - 1) * ks] = real(0.0);
  }
};

// mass and energy update of the small step from the new rhogw split, one
// thread per point (kernels/vimain.py:190-262, rhogkin.py:38-79)
//
// kin carries the kinetic energy of the state after a small step to the next
// one, whose state before it is the same: with KIN it is read instead of formed
// again from four more fields.
template <bool KIN>
struct ViMainPost {
  static constexpr const char* kName = "vi_main_post";
  Dims d; Consts c; Geo G;
  real dt, rweight;
  const real* prog;
  const real* ps[6];
  const real* dv[3];
  const real* ethtot;
  const real* gT;
  const real* getot;
  const real* hv[3];
  real* we[3];       // we[1] (rhogw split) is read
  real* kin;         // kinetic energy of the state before (KIN: read) and after (written)
  MeanFlux mf;
  // Every value the point needs is loaded first, at levels clamped into
  // 0..kall-1 (a clamped level's value is never used: the level tests below
  // are the reference's), so that the loads issue together instead of one
  // memory round trip per level test.
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p) || !pt_compute(p)) return;
    const long NF = d.NF, ks = p.ks, a = p.a;
    const int kmin = d.kmin, kmax = d.kmax, k = p.k;
    const long b = a - (long)k * ks;
    // window levels k-1 .. k+2 -> index 0..3
    long A[4];
    for (int j = 0; j < 4; ++j) {
      int kk = k - 1 + j;
      kk = (kk < 0) ? 0 : ((kk > d.kall - 1) ? d.kall - 1 : kk);
      A[j] = b + (long)kk * ks;
    }
    const real* pg = ps[I_RHOG];
    const real* rw1 = we[1];
    real P0[3], S0[3], H0[3], T0[3], ET[3], RW[4], P4[2], S4[2], PQ[3], SQ[3], DQ[3];
    for (int j = 0; j < 3; ++j) {
      P0[j] = prog[A[j]];
      S0[j] = pg[A[j]];
      H0[j] = hv[0][A[j]];
      T0[j] = gT[A[j]];
      ET[j] = ethtot[A[j]];
    }
    for (int j = 0; j < 4; ++j) RW[j] = rw1[A[j]];
    for (int j = 0; j < 2; ++j) {
      P4[j] = prog[4 * NF + A[1 + j]];
      if (!KIN) S4[j] = ps[4][A[1 + j]];
    }
    for (int q = 0; q < 3; ++q) {
      PQ[q] = prog[(1 + q) * NF + a];
      if (!KIN) SQ[q] = ps[1 + q][a];
      DQ[q] = dv[q][a];
    }
    const real kin_in = KIN ? kin[a] : real(0.0);
    const real h2 = hv[2][a], ge = getot[a];
    const int ke = (k < kmin) ? kmin : ((k > kmax) ? kmax : k);
    const real pe_k = ps[I_RHOGE][b + (long)ke * ks];
    real pm0 = real(0.0), pm4 = real(0.0), rw0 = real(0.0);
    if (mf.out) {
      pm0 = mf.in[0 * NF + a];
      pm4 = mf.in[4 * NF + a];
      if (mf.two) rw0 = ps[4][a];
    }
    // j: window index of level kk (k - 1 + j)
    auto rs1 = [&](int kk, int j) {
      real drhog2 = real(0.0);
      if (kk >= kmin && kk <= kmax) {
        const real hi = (kk + 1 <= kmax) ? real(0.0) * real(1.0) + real(1.0) * RW[j + 1] * real(1.0) : real(0.0);
        const real lo = (kk >= kmin + 1) ? real(0.0) * real(1.0) + real(1.0) * RW[j] * real(1.0) : real(0.0);
        drhog2 = -H0[j] - (hi - lo) * G.rdgz[kk];
      }
      return S0[j] + (T0[j] + drhog2) * dt;
    };
    auto g10 = [&](int kk, int q) {
      const int j = kk - k + 1;
      if (q == 0) return P0[j] + S0[j];
      if (q == 4) return P4[j - 1] + S4[j - 1];
      return PQ[q - 1] + SQ[q - 1];
    };
    auto g11 = [&](int kk, int q) {
      const int j = kk - k + 1;
      if (q == 0) return P0[j] + rs1(kk, j);
      if (q == 4) return P4[j - 1] + RW[j];
      return PQ[q - 1] + DQ[q - 1];
    };
    const real kin10 = KIN ? kin_in : rhogkin_k(G, kmin, kmax, k, g10);
    const real kin11 = rhogkin_k(G, kmin, kmax, k, g11);
    real dtot = real(0.0);
    if (k >= kmin && k <= kmax) {
      real hi = real(0.0), lo = real(0.0);
      if (k + 1 <= kmax)
        hi = real(0.0) * real(1.0) + real(1.0) * ((P4[1] + RW[2]) * (G.afact[k + 1] * ET[2] + G.bfact[k + 1] * ET[1]))
             * real(1.0);
      if (k >= kmin + 1)
        lo = real(0.0) * real(1.0) + real(1.0) * ((P4[0] + RW[1]) * (G.afact[k] * ET[1] + G.bfact[k] * ET[0]))
             * real(1.0);
      dtot = -h2 - (hi - lo) * G.rdgz[k];
    }
    const real r1 = rs1(k, 1);
    const real re1 = pe_k + (ge + dtot) * dt + (kin10 - kin11) + (S0[1] - r1) * G.phi[k];
    we[0][a] = r1;
    we[2][a] = re1;
    kin[a] = kin11;
    if (mf.out) {
      mf.out[0 * NF + a] = mf.add(pm0, S0[1], r1, rweight);
      mf.out[4 * NF + a] = mf.add(pm4, rw0, RW[1], rweight);
    }
  }
};

// PROG += PROG_split and horizontal projection (mod_vi.py:1572-1586)
struct ProgUpdateP {
  static constexpr const char* kName = "prog_update";
  Dims d; Consts c; Geo G;
  real* prog;
  const real* ps[6];
  NH_HD void operator()(int plane, int x) const {
    Pt p;
    if (!pt_of(d, plane, x, p)) return;
    const long NF = d.NF, a = p.a;
    const real R = c.RADIUS;
    real v[6];
    for (int q = 0; q < 6; ++q) v[q] = prog[q * NF + a] + ps[q][a];
    if (p.pole) {
      const real gx = G.gx_pl[(p.v * 2 + p.lp) * 3 + 0];
      const real gy = G.gx_pl[(p.v * 2 + p.lp) * 3 + 1];
      const real gz = G.gx_pl[(p.v * 2 + p.lp) * 3 + 2];
      const real prd = v[1] * gx / R + v[2] * gy / R + v[3] * gz / R;
      v[1] = v[1] - prd * gx / R; v[2] = v[2] - prd * gy / R; v[3] = v[3] - prd * gz / R;
    } else if (p.inner) {
      const real gx = G.gx[p.ci], gy = G.gx[d.nreg + p.ci], gz = G.gx[2 * d.nreg + p.ci];
      const real prd = (v[1] * gx + v[2] * gy + v[3] * gz) / R;
      v[1] = v[1] - prd * gx / R; v[2] = v[2] - prd * gy / R; v[3] = v[3] - prd * gz / R;
    }
    for (int q = 0; q < 6; ++q) prog[q * NF + a] = v[q];
  }
};

NH_END
