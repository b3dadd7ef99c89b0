// Column-tile form (nh_colstencil.h) of the small step's transposed pressure
// gradient: the interior points.  Region borders and pole points run the point forms of
// nh_adjoint.h, one thread per border point and level.
//
// A transposed stencil gathers at point x the bars of the compute points whose
// stencil holds x; the coefficient belongs to the source point.  The point
// forms load, per neighbour and level, the source's coefficients, position and
// bars; here a column keeps its seven sources' coefficients (zero where the
// source is not a compute point) and the bars are formed once per point and
// staged.
#pragma once

#include "nh_adjoint.h"
#include "nh_colstencil.h"

NH_BEGIN

// stencil neighbour that is the source x - off(m)
NH_HD inline int opp7(int m) { return (m == 0) ? 0 : (m < 4) ? m + 3 : m - 3; }

// the columns a thread stages: whether it is a compute column, and its position
struct SrcCol {
  bool in;
  real x[3];
};

// is column ci = (l g + j) g + i a compute column
NH_HD inline bool inner_col(const Dims& d, long ci) {
  const long r = ci % ((long)d.g * d.g);
  const int j = (int)(r / d.g), i = (int)(r - (long)j * d.g);
  return i >= 1 && i <= d.g - 2 && j >= 1 && j <= d.g - 2;
}

// coefficients dd * 7 + m of a 3 x 7 operator at the column's seven sources
NH_HD inline void src_coef(const Dims& d, const real* coef, long ci, real c[3][7]) {
  for (int m = 0; m < 7; ++m) {
    const int di = ((4201 >> (2 * m)) & 3) - 1, dj = ((421 >> (2 * m)) & 3) - 1;
    const long co = ci - di - (long)dj * d.g;
    const bool in = inner_col(d, co);
    for (int q = 0; q < 3; ++q) c[q][m] = in ? rc(coef, d.nreg, q * 7 + m, co) : real(0.0);
  }
}

// path1 transposed (Path1A) at the interior points.  With the border launch, per
// small step at gl06: 98 -> 80 us mixed, 157 -> 115 FP64 (20 fields: 30 and 60 us
// of streaming; the border points' edge columns, one value per cache line, cost
// about as much as the interior).  The point form also read and wrote prog's bar
// on every level where only the boundary levels' change.  (vi_main_h's transpose
// the same way was slower, 67 -> 96 us: its border points touch 15 fields.)
struct Path1TC {
  static constexpr const char* kName = Path1A::kName;
  static constexpr int kNS = 3;
  static constexpr bool kMapped = false;
  Path1A pk;
  Dims d;
  struct Col {
    real c[3][7];
  };
  using Stg = SrcCol;
  struct Pre {
    real v[3], ps[3], gT[3], e;
  };
  NH_HD void begin(Pre&) const {}
  NH_HD void init_stage(long ci, Stg& sg) const {
    sg.in = inner_col(d, ci);
    for (int q = 0; q < 3; ++q) sg.x[q] = pk.G.gx[q * d.nreg + ci];
  }
  // the levels that receive a gradient's bar
  NH_HD bool stage_level(int k) const { return k >= d.kmin + 1 && k <= d.kmax; }
  // bars of the gradients taken at level k: the output's own, at kmin+1 also
  // those of kmin and its ghost row, at kmax that of the ghost row above
  NH_HD void stage(int k, unsigned o, unsigned, const Stg& sg, real* v) const {
    v[0] = v[1] = v[2] = real(0.0);
    if (!sg.in) return;
    const long a = (long)(o / (unsigned)sizeof(real)), ks = (long)d.g * d.g;
    pk.grad_bar(a, ks, k, sg.x, v);
    real w[3];
    if (k == d.kmin + 1)
      for (int n = 1; n <= 2; ++n) {
        pk.grad_bar(a - n * ks, ks, k - n, sg.x, w);
        for (int q = 0; q < 3; ++q) v[q] += w[q];
      }
    if (k == d.kmax) {
      pk.grad_bar(a + ks, ks, k + 1, sg.x, w);
      for (int q = 0; q < 3; ++q) v[q] += w[q];
    }
  }
  NH_HD void stage_own(int k, unsigned o, const Stg& sg, const Pre&, real* v) const { stage(k, o, o, sg, v); }
  NH_HD void pre(int k, unsigned o, const Stg&, Pre& p) const {
    if (k < d.kmin || k > d.kmax) return;
    for (int q = 0; q < 3; ++q) {
      p.v[q] = at_off(pk.dv_b[q], o);
      p.ps[q] = at_off(pk.ps_b[1 + q], o);
      p.gT[q] = at_off(pk.gT_b + (1 + q) * d.NF, o);
    }
    p.e = at_off(pk.ps_b[I_RHOGE], o);
  }
  NH_HD void init_col(long ci, Col& col) const {
    src_coef(d, pk.G.cgrad, ci, col.c);
    const real RovCV = pk.c.Rdry / pk.c.CVdry;
    for (int q = 0; q < 3; ++q)
      for (int m = 0; m < 7; ++m) col.c[q][m] = col.c[q][m] * RovCV;
  }
  NH_HD void pole(int) const {}
  template <class NB>
  NH_HD void point(int k, unsigned o, const Col& col, Pre& p, NB nb) const {
    if (k < d.kmin || k > d.kmax) {
      for (int q = 0; q < 3; ++q) at_off(pk.dd_b[q], o) = real(0.0);
      return;
    }
    if (stage_level(k)) {
      real eb = real(0.0);
#pragma unroll
      for (int m = 0; m < 7; ++m)
        for (int q = 0; q < 3; ++q) eb += col.c[q][m] * nb(opp7(m), q);
      at_off(pk.ps_b[I_RHOGE], o) = p.e + eb;
    }
    if (k == d.kmin || k == d.kmax) pk.ghost_terms((long)(o / (unsigned)sizeof(real)), (long)d.g * d.g, k, p.v);
    for (int q = 0; q < 3; ++q) {
      at_off(pk.ps_b[1 + q], o) = p.ps[q] + p.v[q];
      at_off(pk.gT_b + (1 + q) * d.NF, o) = p.gT[q] + p.v[q] * pk.dt;
      at_off(pk.dd_b[q], o) = p.v[q] * pk.dt;
    }
  }
};

NH_END
