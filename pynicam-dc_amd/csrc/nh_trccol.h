// Limiter kernels of the tracer transport as column tiles (see the engine in
// nh_colstencil.h): the outflow bounds (TrcQoutC) and the limited update
// (TrcApplyC).  Each cell needs the mixing ratio at 7 points and the Courant
// masks of its six faces, three of them owned by neighbours; as a point kernel
// that is 16 divisions, 13 of them repeated by neighbours.  Here a cell stages
// its mixing ratio and its three Courant numbers once per level and the tile
// reads the rest from LDS: 7 divisions.
// Bounds and update as points and as tiles: gl06 z60 FP64 70 and 80 -> 56 and
// 70 us, gl07 z40 mixed 119 and 120 -> 78 and 81 us.
#pragma once

#include "nh_colstencil.h"
#include "nh_tracer.h"

NH_BEGIN

template <class P>
struct TrcLimC {
  static constexpr const char* kName = P::kName;
  static constexpr bool kMapped = false;
  P pk;
  Dims d;
  struct Col {
    real ra;
    bool pent;
  };
  struct Stg {
    real ra;
  };
  struct Pre {
    real q, r, f[3], fn[3];   // own rhogq, rhog, owned arc fluxes; the neighbours' arcs
  };
  NH_HD void begin(Pre&) const {}
  NH_HD bool stage_level(int) const { return true; }
  NH_HD void init_stage(long ci, Stg& sg) const { sg.ra = rc(pk.G.rarea, d.nreg, 0, ci); }
  NH_HD void init_col(long ci, Col& col) const {
    col.ra = rc(pk.G.rarea, d.nreg, 0, ci);
    const int g = d.g, h = (int)(ci % ((long)g * g)), l = (int)(ci / ((long)g * g));
    col.pent = h == g + 1 && pk.G.sgp[l];   // i = j = 1 of a pentagon region
  }
  NH_HD void own_loads(unsigned o, Pre& p) const {
    const int g = d.g;
    p.q = at_off(pk.rq, o);
    p.r = at_off(pk.rhog1, o);
    for (int m = 0; m < 3; ++m) p.f[m] = at_off(pk.fa[m], o);
    p.fn[0] = at_off(pk.fa[0] - 1, o);
    p.fn[1] = at_off(pk.fa[1] - 1 - g, o);
    p.fn[2] = at_off(pk.fa[2] - g, o);
  }
  // staged: mixing ratio, Courant numbers of the owned arcs
  NH_HD void courant(real q, real r, const real* f, real ra, real* v) const {
    v[0] = q / r;
    for (int m = 0; m < 3; ++m) v[1 + m] = f[m] * ra * pk.dt / r;
  }
  NH_HD void ring_stage(unsigned o, const Stg& sg, real* v) const {
    const real f[3] = {at_off(pk.fa[0], o), at_off(pk.fa[1], o), at_off(pk.fa[2], o)};
    courant(at_off(pk.rq, o), at_off(pk.rhog1, o), f, sg.ra, v);
  }
  template <class NB>
  NH_HD void cell(const Col& col, const Pre& p, NB nb, TrcCellCtx& x) const {
#pragma unroll
    for (int m = 0; m < 7; ++m) x.q[m] = nb(m, 0);
    for (int m = 0; m < 3; ++m) {
      x.f[m] = p.f[m] * col.ra * pk.dt;
      x.f[3 + m] = -p.fn[m] * col.ra * pk.dt;
    }
    if (col.pent) x.f[5] *= real(0.0);
    for (int m = 0; m < 3; ++m) {
      x.ch[m] = nb(0, 1 + m);
      x.ch[3 + m] = x.f[3 + m] / p.r;
      x.cmo[m] = upwind_mask(x.ch[m]);
      x.cmo[3 + m] = upwind_mask(nb(4 + m, 1 + m));   // the owner's
    }
  }
  NH_HD void pole(int pb) const { pk(d.lall * d.kall + pb, 0); }
};

struct TrcQoutC : TrcLimC<TrcQout> {
  static constexpr int kNS = 4;
  struct Pre : TrcLimC<TrcQout>::Pre {
    real fr;
  };
  NH_HD void begin(Pre&) const {}
  NH_HD void pre(int, unsigned o, const Stg&, Pre& p) const {
    own_loads(o, p);
    p.fr = at_off(pk.frhog, o);
  }
  NH_HD void stage_own(int, unsigned, const Stg& sg, const Pre& p, real* v) const { courant(p.q, p.r, p.f, sg.ra, v); }
  NH_HD void stage(int, unsigned o, unsigned, const Stg& sg, real* v) const { ring_stage(o, sg, v); }
  template <class NB>
  NH_HD void point(int, unsigned o, const Col& col, Pre& p, NB nb) const {
    TrcCellCtx x;
    cell(col, p, nb, x);
    trc_qout_cell(x, col.pent, real(1.0) * p.fr / p.r * pk.dt, at_off(pk.qout[0], o), at_off(pk.qout[1], o));
  }
};

struct TrcApplyC : TrcLimC<TrcApply> {
  static constexpr int kNS = 6;   // and the two outflow bounds
  struct Pre : TrcLimC<TrcApply>::Pre {
    real qa[6], b[2];
  };
  NH_HD void begin(Pre&) const {}
  NH_HD void pre(int, unsigned o, const Stg&, Pre& p) const {
    const int g = d.g;
    own_loads(o, p);
    for (int m = 0; m < 3; ++m) p.qa[m] = at_off(pk.qa[m], o);
    p.qa[3] = at_off(pk.qa[0] - 1, o);
    p.qa[4] = at_off(pk.qa[1] - 1 - g, o);
    p.qa[5] = at_off(pk.qa[2] - g, o);
    for (int m = 0; m < 2; ++m) p.b[m] = at_off(pk.qout[m], o);
  }
  NH_HD void stage_own(int, unsigned, const Stg& sg, const Pre& p, real* v) const {
    courant(p.q, p.r, p.f, sg.ra, v);
    v[4] = p.b[0];
    v[5] = p.b[1];
  }
  NH_HD void stage(int, unsigned o, unsigned, const Stg& sg, real* v) const {
    ring_stage(o, sg, v);
    v[4] = at_off(pk.qout[0], o);
    v[5] = at_off(pk.qout[1], o);
  }
  template <class NB>
  NH_HD void point(int, unsigned o, const Col& col, Pre& p, NB nb) const {
    TrcCellCtx x;
    cell(col, p, nb, x);
    real q0[7], q1[7];
#pragma unroll
    for (int m = 0; m < 7; ++m) {
      q0[m] = nb(m, 4);
      q1[m] = nb(m, 5);
    }
    at_off(pk.out, o) = p.q - trc_outflow_cell(x, col.pent, p.qa, q0, q1);
  }
};

template <class C, class X, class P>
void run_trc_lim(X& x, const P& pk) {
  ColStencil<C> cs;
  cs.op.pk = pk;
  cs.op.d = pk.d;
  cs.cg = st_geom(pk.d);
  x.run_cols(cs, cs.cg.nblocks, ColStencil<C>::lds_elems(cs.cg));
}

template <class X>
void run_trc_qout(X& x, const TrcQout& f) {
  run_trc_lim<TrcQoutC>(x, f);
}

template <class X>
void run_trc_apply(X& x, const TrcApply& f) {
  if (f.limiter) run_trc_lim<TrcApplyC>(x, f);
  else x.run_pts(f, f.d);
}

NH_END
