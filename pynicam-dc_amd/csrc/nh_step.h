// Stencil and column helpers of the HEVI large/small step (used by the
// point kernels of nh_point.h and the tracer kernels of nh_tracer.h).
//
// Vertical metrics enter as k-profiles (flat topography: GSQRT = GAM = 1, the
// terrain-following gradient terms vanish); the host verifies this before it
// creates a context.  Operation order follows the reference kernels so that
// the FP64 results track the numpy path to round-off.
#pragma once

#include "nh_columns.h"

NH_BEGIN

// ----------------------------------------------------------------------------
// Operators of the hyperdiffusion and divergence damping at a pole centre (the
// regional cells' are in nh_tile.h and nh_colstencil.h; Laplacian
// oprtlaplacian.py:41-55, divergence damping mod_numfilter.py:2032-2268,
// kernels/oprt3ddivdamp.py, kernels/oprtdivdamp.py, kernels/divdamppostcomm.py)
// ----------------------------------------------------------------------------

// ad(v): address of pole point v at this level
template <class AD>
NH_HD inline real lap_pl_at(const Geo& G, int lp, const real* f, AD ad) {
  real s = real(0.0);
  for (int v = 0; v < 6; ++v) {
    real pv = G.clap_pl[v * 2 + lp] * f[ad(v)];
    s = (v == 0) ? pv : s + pv;
  }
  return s;
}
NH_HD inline real lap_pl(const Geo& G, int lp, const real* f, long a0) {
  // a0: address of pole point v=0 at this level; neighbours at a0 + v
  return lap_pl_at(G, lp, f, [a0](int v) { return a0 + v; });
}

// ----------------------------------------------------------------------------
// Kh-weighted diffusion (kernels/oprtdiffusion.py:59-177)
// ----------------------------------------------------------------------------
// Triangle value of a diffusion-type operator: triangle of type T whose (i, j)
// corner has cell index cj and address a.  TI spans (i,j)(i+1,j)(i+1,j+1),
// TJ spans (i,j)(i+1,j+1)(i,j+1).
NH_HD inline void tri_grad(const Geo& G, long nreg, long cj, int T, const real* s, long a, int g,
                           real out[3]) {
  real s0 = s[a];
  real s1 = (T == 0) ? s[a + 1] : s[a + 1 + g];
  real s2 = (T == 0) ? s[a + 1 + g] : s[a + g];
  for (int dd = 0; dd < 3; ++dd) {
    real c1 = rc(G.cintp, nreg, (dd * 3 + 0) * 2 + T, cj);
    real c2 = rc(G.cintp, nreg, (dd * 3 + 1) * 2 + T, cj);
    real c3 = rc(G.cintp, nreg, (dd * 3 + 2) * 2 + T, cj);
    out[dd] = ((real(2.0) * c1 - c2 - c3) * s0 + (-c1 + real(2.0) * c2 - c3) * s1 + (-c1 - c2 + real(2.0) * c3) * s2) / real(3.0);
  }
}

// s at pole point v is read at ad(v), kh at a0 + v
template <class KH, class AD>
NH_HD inline real diffusion_pl(const Geo& G, int lp, const real* s, KH kh, long a0, AD ad) {
  real vt[5][3];
  for (int v = 1; v <= 5; ++v) {
    int vp = (v == 5) ? 1 : v + 1;
    for (int dd = 0; dd < 3; ++dd) {
      const real* cI = G.cintp_pl + ((v * 2 + lp) * 3 + dd) * 3;
      real c0 = cI[0], c1 = cI[1], c2 = cI[2];
      vt[v - 1][dd] = ((real(2.0) * c0 - c1 - c2) * s[ad(0)] + (-c0 + real(2.0) * c1 - c2) * s[ad(v)]
                       + (-c0 - c1 + real(2.0) * c2) * s[ad(vp)]) / real(3.0);
    }
  }
  real row = real(0.0);
  for (int v = 1; v <= 5; ++v) {
    int vm = (v == 1) ? 5 : v - 1;
    real kavg = real(0.5) * (kh(a0) + kh(a0 + v));
    const real* cd = G.cdiff_pl + (v * 2 + lp) * 3;
    real sum = cd[0] * (vt[vm - 1][0] + vt[v - 1][0]);
    sum = sum + cd[1] * (vt[vm - 1][1] + vt[v - 1][1]);
    sum = sum + cd[2] * (vt[vm - 1][2] + vt[v - 1][2]);
    real cb = kavg * sum;
    row = (v == 1) ? cb : row + cb;
  }
  return row;
}

NH_HD inline void grad_pl(const Geo& G, int lp, const real* s, long a0, real o[3]) {
  for (int dd = 0; dd < 3; ++dd) {
    real acc = real(0.0);
    for (int v = 0; v < 6; ++v) {
      real pv = G.cgrad_pl[(v * 2 + lp) * 3 + dd] * (s[a0 + v] * real(1.0) * real(1.0));
      acc = (v == 0) ? pv : acc + pv;
    }
    o[dd] = acc;
  }
}

// neighbour column bases of a compute cell (7 regional, 6 pole)
NH_HD inline int neighbours(const Dims& d, const Cell& cl, long nb[7]) {
  if (cl.pole) {
    for (int v = 0; v < 6; ++v) nb[v] = d.R + (long)cl.lp * d.kall * 6 + v;
    return 6;
  }
  long off[7];
  stencil_offsets(d.g, off);
  for (int m = 0; m < 7; ++m) nb[m] = cl.base + off[m];
  return 7;
}

// NDIV horizontal divergences at a pole centre, one neighbour at a time:
// f(m, addr, v) fills v[i][dir] for divergence i at neighbour m (address
// addr); per point cx*fx + cy*fy + cz*fz, summed over v, as div_pl.
template <int NDIV, class F>
NH_HD inline void hdiv_multi(const Geo& G, const Pt& p, F f, real out[NDIV]) {
  real v[NDIV][3];
#pragma unroll 1
  for (int m = 0; m < 6; ++m) {
    f(m, p.a + m, v);
    const real* c = G.cdiv_pl + (m * 2 + p.lp) * 3;
    for (int i = 0; i < NDIV; ++i) {
      const real pv = c[0] * v[i][0] + c[1] * v[i][1] + c[2] * v[i][2];
      out[i] = (m == 0) ? pv : out[i] + pv;
    }
  }
}

// kinetic energy at level k of a column given accessors (kernels/rhogkin.py:38-79),
// in the precision T of the vertical profiles V (the field precision, or FP64
// for the global sums)
template <class T, class F>
NH_HD inline T rhogkin_k(const VProf<T>& V, int kmin, int kmax, int k, F get) {
  // get(k, q): q = 0 rhog, 1..3 rhogv, 4 rhogw
  if (k < kmin || k > kmax) return T(0.0);
  T rgk = get(k, 0);
  T vx = get(k, 1), vy = get(k, 2), vz = get(k, 3);
  T kh = T(0.5) * (vx * vx + vy * vy + vz * vz) / rgk;
  T vup = T(0.0), vdn = T(0.0);
  if (k + 1 <= kmax) {
    T w = get(k + 1, 4);
    vup = T(0.5) * (w * w) / (V.c2w0[k + 1] * get(k + 1, 0) + V.c2w1[k + 1] * rgk);
  }
  if (k >= kmin + 1) {
    T w = get(k, 4);
    vdn = T(0.5) * (w * w) / (V.c2w0[k] * rgk + V.c2w1[k] * get(k - 1, 0));
  }
  return kh + V.w2c0[k] * vup + V.w2c1[k] * vdn;
}

// split state at the start of an RK stage: 0 (first stage) or PROG0 - PROG
struct SplitInit {
  static constexpr const char* kName = "split_init";
  long NF;
  const real* prog;
  const real* prog0;
  real* ps[6];
  int zero;
  NH_HD void operator()(long t) const {
    for (int q = 0; q < 6; ++q) ps[q][t] = zero ? real(0.0) : prog0[q * NF + t] - prog[q * NF + t];
  }
};

NH_END
