// Column tiles for 7-point stencil kernels.
//
// A block owns a TX x TY tile of one region's points (st_geom) over a chunk of
// levels.  Each of the first TX TY threads owns one tile column: the
// per-column coefficients of its operator are loaded once into registers, and
// then, level by level, the thread stages its own values of the operator's
// stencil fields into LDS (the first 2 TX + 2 TY + 2 threads also stage one
// point of the ring around the tile), a barrier, and the thread
// forms its point's result from its neighbours' staged values.  The staging
// planes are double-buffered by level parity, so one barrier per level
// suffices.  The point kernels re-read the 21 stencil coefficients (and the
// neighbours' values) per point and level; here each value is loaded from
// memory once per level and each coefficient once per chunk.
//
// An operator Op supplies
//   kName, kNS (stencil fields), Col (per-column registers), d (Dims),
//   Stg (registers of the column a thread stages: its own and its ring column),
//   kMapped (fields read at the source columns cs of their halo values),
//   Pre (registers a point keeps from level to level or loads before the
//   barrier), begin(Pre&) at the start of a chunk and pre(k, o, Stg, Pre&) per
//   level, with o the point's byte offset in a field (at_off),
//   init_stage(col index, Stg&), stage_level(k), stage(k, o, om, Stg, v[kNS])
//   with om the mapped offset (o unless kMapped), stage_own the same for the
//   thread's own point (Pre at hand),
//   init_col(col index, Col&),
//   point(k, o, Col, Pre, nb) with nb(m, f) = field f at stencil neighbour m
//   (0 (0,0) 1 (+1,0) 2 (+1,+1) 3 (0,+1) 4 (-1,0) 5 (-1,-1) 6 (0,-1)),
//   pole(pb): the pole centre of pole level pb (its point kernel).
#pragma once

#include "nh_tile.h"

NH_BEGIN

// tile shape of the stencil engine: TX x TY = 256 points, 64 x 4 where the
// region is wide enough (a wavefront then reads one 64-point row segment;
// measured faster than 32 x 8 and 16 x 16 at gl07)
struct StGeom {
  int TX, TY;       // tile width and height (points)
  int nx, ny;       // tiles per region row and column
  int nchunk, KC;   // level chunks, levels per chunk
  int ntiles;       // lall * nchunk * nx * ny
  int nblocks;      // + 2 * kall pole blocks
};

inline StGeom st_geom(const Dims& d) {
  StGeom c;
  const int W = d.g - 2;
  c.TX = (W < 64) ? W : 64;
  c.TY = (256 / c.TX < W) ? 256 / c.TX : W;
  c.nx = W / c.TX;
  c.ny = W / c.TY;
  c.KC = chunk_levels((long)d.lall * c.nx * c.ny, d.kall, kColLevels);
  c.nchunk = (d.kall + c.KC - 1) / c.KC;
  c.ntiles = d.lall * c.nchunk * c.nx * c.ny;
  c.nblocks = c.ntiles + 2 * d.kall;
  return c;
}

template <class Op>
struct ColStencil {
  using LdsT = real;
  static constexpr const char* kName = Op::kName;
  static constexpr int kThreads = 256;
  static constexpr int NS = Op::kNS;
  static constexpr int kWaves = 1;
  Op op;
  StGeom cg;
  const int* cs = nullptr;   // kMapped: source columns
  static int lds_elems(const StGeom& cg) { return 2 * NS * (cg.TX + 2) * (cg.TY + 2); }
  struct State {
    typename Op::Col col;
    typename Op::Stg sg, rsg;   // staging registers of the own and the ring column
    typename Op::Pre pre;
    unsigned o, ro;    // own and ring offsets at the current level
    unsigned rm;       // kMapped: the ring point's mapped offset
    int k, sidx, ridx;
    bool outp, ring;
  };
  NH_HD int init(int blk, int tid, State& s) const {
    const Dims& d = op.d;
    s.outp = s.ring = false;
    if (blk >= cg.ntiles) {
      if (tid == 0) op.pole(blk - cg.ntiles);
      return 0;
    }
    const int g = d.g, TX = cg.TX, TY = cg.TY, SW = TX + 2, tpr = cg.nx * cg.ny;
    const int tile = blk % tpr, rest = blk / tpr;
    const int chunk = rest % cg.nchunk, l = rest / cg.nchunk;
    const int k0 = chunk * cg.KC;
    const int k1 = (k0 + cg.KC < d.kall) ? k0 + cg.KC : d.kall;
    if (k0 >= k1) return 0;
    const int i0 = 1 + (tile % cg.nx) * TX, j0 = 1 + (tile / cg.nx) * TY;
    s.k = k0;
    if (tid < TX * TY) {
      const int tx = tid % TX, ty = tid / TX;
      const int i = i0 + tx, j = j0 + ty;
      s.outp = true;
      s.sidx = (ty + 1) * SW + tx + 1;
      s.o = byte_off(((long)(l * d.kall + k0) * g + j) * g + i);
      op.init_col(((long)l * g + j) * g + i, s.col);
      op.init_stage(((long)l * g + j) * g + i, s.sg);
      op.begin(s.pre);
    }
    // the ring: row -1 (x = -1..TX-1), row TY (x = 0..TX), columns -1 and TX (y = 0..TY-1)
    if (tid < 2 * TX + 2 * TY + 2) {
      int x, y;
      if (tid < TX + 1) { x = tid - 1; y = -1; }
      else if (tid < 2 * TX + 2) { x = tid - (TX + 1); y = TY; }
      else if (tid < 2 * TX + TY + 2) { x = -1; y = tid - (2 * TX + 2); }
      else { x = TX; y = tid - (2 * TX + TY + 2); }
      s.ring = true;
      s.ridx = (y + 1) * SW + x + 1;
      s.ro = byte_off(((long)(l * d.kall + k0) * g + (j0 + y)) * g + (i0 + x));
      op.init_stage(((long)l * g + (j0 + y)) * g + (i0 + x), s.rsg);
      if constexpr (Op::kMapped) s.rm = byte_off(src_at(d, cs, ((long)l * g + (j0 + y)) * g + (i0 + x), k0));
    }
    return k1 - k0;
  }
  NH_HD void level_a(int step, State& s, real* lds) const {
    if (s.outp) op.pre(s.k, s.o, s.sg, s.pre);
    if (!op.stage_level(s.k)) return;
    const int SW = cg.TX + 2, P = SW * (cg.TY + 2);
    real* buf = lds + (step & 1) * NS * P;
    real v[NS];
    if (s.outp) {
      op.stage_own(s.k, s.o, s.sg, s.pre, v);
      for (int f = 0; f < NS; ++f) buf[f * P + s.sidx] = v[f];
    }
    if (s.ring) {
      op.stage(s.k, s.ro, Op::kMapped ? s.rm : s.ro, s.rsg, v);
      for (int f = 0; f < NS; ++f) buf[f * P + s.ridx] = v[f];
    }
  }
  NH_HD void level_b(int step, State& s, const real* lds) const {
    if (s.outp) {
      const int SW = cg.TX + 2, P = SW * (cg.TY + 2);
      const real* buf = lds + (step & 1) * NS * P;
      const int x = s.sidx;
      op.point(s.k, s.o, s.col, s.pre, [&](int m, int f) {
        const int off = (m == 0) ? 0 : (m == 1) ? 1 : (m == 2) ? 1 + SW : (m == 3) ? SW : (m == 4) ? -1
                      : (m == 5) ? -1 - SW : -SW;
        return buf[f * P + x + off];
      });
    }
    const unsigned ls = byte_off((long)op.d.g * op.d.g);
    s.o += ls;
    s.ro += ls;
    if constexpr (Op::kMapped) {
      if (s.ring) s.rm += src_stride_off(op.d, s.rm);
    }
    s.k += 1;
  }
};

// The single 7-point operators as column operators, P the point kernel that does
// the pole centres: the Laplacian of one field (NC = 1), the gradient of one
// (NC = 3) and the divergence of three, with their 7 or 21 coefficients in
// registers.  A source SRC gives the staged values: src(f, o).  Gradient of a
// tracer's mixing ratio at gl06 z60 FP64: 81 us per launch as points (21 coefficients
// and 7 quotients per level), 39 as tiles; Laplacian, gradient and divergence at gl06
// z40 FP64 in turn: 115 against 73.
template <class P, class SRC, int NC>
struct Oper7C {
  static constexpr const char* kName = P::kName;
  static constexpr bool kDiv = SRC::kFields == 3;
  static constexpr int kNS = SRC::kFields;
  static constexpr bool kMapped = false;
  P pk;
  SRC src;
  Dims d;
  const real* coef;
  real* out[kDiv ? 1 : NC];
  struct Col {
    real c[NC][7];
  };
  struct Stg {};
  struct Pre {};
  NH_HD void begin(Pre&) const {}
  NH_HD void init_stage(long, Stg&) const {}
  NH_HD void pre(int, unsigned, const Stg&, Pre&) const {}
  NH_HD bool stage_level(int) const { return true; }
  NH_HD void stage(int, unsigned o, unsigned, const Stg&, real* v) const {
    for (int f = 0; f < kNS; ++f) v[f] = src(f, o);
  }
  NH_HD void stage_own(int k, unsigned o, const Stg& sg, const Pre&, real* v) const { stage(k, o, o, sg, v); }
  NH_HD void init_col(long ci, Col& col) const {
    for (int dd = 0; dd < NC; ++dd)
      for (int m = 0; m < 7; ++m) col.c[dd][m] = rc(coef, d.nreg, dd * 7 + m, ci);
  }
  NH_HD void pole(int pb) const { pk(d.lall * d.kall + pb, 0); }
  // per direction the sum over the neighbours in stencil order, the divergence's x + y + z
  template <class NB>
  NH_HD void point(int, unsigned o, const Col& col, Pre&, NB nb) const {
    real s[NC];
    for (int dd = 0; dd < NC; ++dd) {
      s[dd] = col.c[dd][0] * nb(0, kDiv ? dd : 0);
#pragma unroll
      for (int m = 1; m < 7; ++m) s[dd] = s[dd] + col.c[dd][m] * nb(m, kDiv ? dd : 0);
    }
    if constexpr (kDiv) {
      at_off(out[0], o) = s[0] + s[1] + s[2];
    } else {
      for (int dd = 0; dd < NC; ++dd) at_off(out[dd], o) = s[dd];
    }
  }
};

// staged as they are: one field or three
template <int N>
struct SrcFields {
  static constexpr int kFields = N;
  const real* f[N];
  NH_HD real operator()(int n, unsigned o) const { return at_off(f[n], o); }
};

// mixing ratio of a tracer mass
struct SrcRatio {
  static constexpr int kFields = 1;
  const real* rq;
  const real* rhog;
  NH_HD real operator()(int, unsigned o) const { return at_off(rq, o) / at_off(rhog, o); }
};

template <int NC, class X, class P, class SRC>
void run_oper7(X& x, const Dims& d, const P& pk, const SRC& src, const real* coef, real* const* out) {
  ColStencil<Oper7C<P, SRC, NC>> cs;
  cs.op.pk = pk;
  cs.op.src = src;
  cs.op.d = d;
  cs.op.coef = coef;
  for (int q = 0; q < (SRC::kFields == 3 ? 1 : NC); ++q) cs.op.out[q] = out[q];
  cs.cg = st_geom(d);
  x.run_cols(cs, cs.cg.nblocks, decltype(cs)::lds_elems(cs.cg));
}

// vi_main, horizontal part (ViMainH) as a column operator: the 21 divergence
// coefficients in registers, the 8 stencil fields staged per level
struct ViMainHC {
  static constexpr const char* kName = "vi_main_h";
  static constexpr int kNS = 8;
  static constexpr bool kMapped = true;
  ViMainH pk;
  Dims d;
  struct Col {
    real c[3][7];
  };
  struct Stg {};
  struct Pre {
    real g5;
  };
  NH_HD void init_stage(long, Stg&) const {}
  NH_HD void begin(Pre&) const {}
  NH_HD void pre(int k, unsigned o, const Stg&, Pre& p) const {
    if (stage_level(k)) p.g5 = at_off(pk.gT + 5 * d.NF, o);
  }
  NH_HD void stage_own(int k, unsigned o, const Stg& sg, const Pre&, real* v) const { stage(k, o, o, sg, v); }
  NH_HD bool stage_level(int k) const { return k >= d.kmin && k <= d.kmax; }
  NH_HD void stage(int, unsigned o, unsigned om, const Stg&, real* v) const {
    for (int q = 0; q < 3; ++q) {
      v[q] = at_off(pk.dv[q], om);
      v[5 + q] = at_off(pk.prog + (long)(1 + q) * d.NF, o);
    }
    v[3] = at_off(pk.eth, o);
    v[4] = at_off(pk.ethtot, o);
  }
  NH_HD void init_col(long ci, Col& col) const {
    for (int dd = 0; dd < 3; ++dd)
      for (int m = 0; m < 7; ++m) col.c[dd][m] = rc(pk.G.cdiv, d.nreg, dd * 7 + m, ci);
  }
  NH_HD void pole(int pb) const { pk(d.lall * d.kall + pb, 0); }
  // ViMainH::at with hdiv_multi<3>, term for term
  template <class NB>
  NH_HD void point(int k, unsigned o, const Col& col, Pre& p, NB nb) const {
    if (k < d.kmin || k > d.kmax) return;
    real s[3][3];
#pragma unroll
    for (int m = 0; m < 7; ++m) {
      real v[3][3];
      const real e = nb(m, 3), et = nb(m, 4);
      for (int q = 0; q < 3; ++q) {
        const real dq = nb(m, q);
        v[0][q] = dq * real(1.0);
        v[1][q] = dq * e * real(1.0);
        v[2][q] = (nb(m, 5 + q) + dq) * et * real(1.0);
      }
      for (int i = 0; i < 3; ++i) {
        const real tx = col.c[0][m] * v[i][0], ty = col.c[1][m] * v[i][1], tz = col.c[2][m] * v[i][2];
        s[i][0] = (m == 0) ? tx : s[i][0] + tx;
        s[i][1] = (m == 0) ? ty : s[i][1] + ty;
        s[i][2] = (m == 0) ? tz : s[i][2] + tz;
      }
    }
    const real divs1 = s[0][0] + s[0][1] + s[0][2];
    const real he = s[1][0] + s[1][1] + s[1][2];
    const real hd = s[2][0] + s[2][1] + s[2][2];
    const real drhoge = -he - (real(0.0) - real(0.0)) * pk.G.rdgz[k];
    const real grhoge1 = p.g5 + drhoge;
    at_off(pk.hv[0], o) = divs1;
    at_off(pk.hv[1], o) = grhoge1 * pk.c.Rdry / pk.c.CVdry;
    at_off(pk.hv[2], o) = hd;
  }
};

// path1 (Path1P) as a column operator: the 21 gradient coefficients and the
// column's position in registers, the split rhoge staged per level at the
// level of its gradient; the nine pointwise values are loaded before the
// barrier, with the staged ones, so that a level waits for memory once.  Bound
// by HBM traffic (13 fields, 19 where the mean fluxes accumulate): 105 us per
// launch at gl07 mixed, 196 FP64; as level-staged points, re-reading the 24
// coefficients per level, 141 and 233; as column tiles with the pointwise loads
// after the barrier slower than those.
struct Path1C {
  static constexpr const char* kName = "vi_path1";
  static constexpr int kNS = 1;
  static constexpr bool kMapped = true;
  Path1P pk;
  Dims d;
  struct Col {
    real c[3][7];
    real x[3];
  };
  struct Stg {};
  struct Pre {
    real g[3], dd[3], ps[3];
    real mq[3], mp[3];   // mean fluxes: the sums and the previous step's momentum
  };
  NH_HD void init_stage(long, Stg&) const {}
  NH_HD bool stage_level(int) const { return true; }
  NH_HD void stage(int k, unsigned, unsigned om, const Stg&, real* v) const {
    v[0] = at_off(pk.ps[I_RHOGE], om + (unsigned)pk.stage_shift(k) * src_stride_off(d, om));
  }
  NH_HD void stage_own(int k, unsigned o, const Stg& sg, const Pre&, real* v) const { stage(k, o, o, sg, v); }
  // values from a point to the physical level it takes its momentum from (ghost rows: the nearest)
  NH_HD long phys(int k) const {
    const long gg = (long)d.g * d.g;
    return (k < d.kmin) ? gg : (k > d.kmax) ? -gg : 0;
  }
  NH_HD void begin(Pre&) const {}
  NH_HD void pre(int k, unsigned o, const Stg&, Pre& p) const {
    const long n = phys(k);
    for (int q = 0; q < 3; ++q) {
      p.g[q] = at_off(pk.gT + (1 + q) * d.NF + n, o);
      p.dd[q] = at_off(pk.dd[q] + n, o);
      p.ps[q] = at_off(pk.ps[1 + q] + n, o);
      if (pk.mf.out) {
        p.mq[q] = at_off(pk.mf.in + (1 + q) * d.NF, o);
        if (pk.mf.two) p.mp[q] = at_off(pk.ps[1 + q], o);
      }
    }
  }
  NH_HD void init_col(long ci, Col& col) const {
    for (int dd = 0; dd < 3; ++dd)
      for (int m = 0; m < 7; ++m) col.c[dd][m] = rc(pk.G.cgrad, d.nreg, dd * 7 + m, ci);
    for (int q = 0; q < 3; ++q) col.x[q] = pk.G.gx[q * d.nreg + ci];
  }
  NH_HD void pole(int pb) const { pk(d.lall * d.kall + pb, 0); }
  // Path1P's arithmetic for a regional point
  template <class NB>
  NH_HD void point(int k, unsigned o, const Col& col, Pre& p, NB nb) const {
    const int kmin = d.kmin, kmax = d.kmax;
    const real R = pk.c.RADIUS, RovCV = pk.c.Rdry / pk.c.CVdry;
    const MeanFlux& mf = pk.mf;
    real pr[7];
    for (int m = 0; m < 7; ++m) pr[m] = (nb(m, 0) * RovCV) * real(1.0);
    real gr[3];
    for (int dd = 0; dd < 3; ++dd) {
      real acc = col.c[dd][0] * pr[0];
      for (int m = 1; m < 7; ++m) acc = acc + col.c[dd][m] * pr[m];
      gr[dd] = acc + real(0.0);
    }
    const real prd = (gr[0] * col.x[0] + gr[1] * col.x[1] + gr[2] * col.x[2]) / R;
    real v[3];
    for (int q = 0; q < 3; ++q) {
      const real Pg = gr[q] - prd * col.x[q] / R;
      const real drv = p.g[q] - Pg + p.dd[q] + real(0.0);
      v[q] = p.ps[q] + drv * pk.dt;
    }
    if (k < kmin || k > kmax) {
      // free-slip top / rigid bottom, scaled by the large-step density
      const real rn = at_off(pk.prog + phys(k), o), ra = at_off(pk.prog, o);
      for (int q = 0; q < 3; ++q) v[q] = (k > kmax) ? real(1.0) * (v[q] / rn) * ra : -real(1.0) * (v[q] / rn) * ra;
    }
    for (int q = 0; q < 3; ++q) {
      at_off(pk.dv[q], o) = v[q];
      if (mf.out) at_off(mf.out + (1 + q) * d.NF, o) = mf.add(p.mq[q], p.mp[q], v[q], pk.rweight);
    }
  }
};

// the large-step source terms and the tridiagonal matrix (ViPath0P) as a column
// operator: the 42 divergence and gradient coefficients in registers, the
// momentum, eth and the pressure staged per level.  A column marches upward and
// carries what levels k and k + 1 share (the effective gravity of the half
// levels, with its divisions, in both precisions, and eth at half levels), where
// the point form forms each three times; all loads of a level go out before
// its barrier.  Bound by memory latency at the 3 (FP64 2) waves per SIMD its
// registers leave: 340 us per launch at gl07 mixed, 533 FP64 (34 fields, 3 FP64
// fields: 222 and 425 us of streaming); one thread per point 454 and 788.
struct ViPath0C {
  static constexpr const char* kName = "vi_path0";
  static constexpr int kNS = 5;
  static constexpr bool kMapped = false;
  ViPath0P pk;
  Dims d;
  struct Col {
    real cd[3][7], cg[3][7];
    real x[3];
  };
  struct Stg {};
  struct Pre {
    bool have;
    real rgm, rg0, rg1, pr0, pr1, et0, et1, rw0, rw1;   // levels k-1, k, k+1
    real dp0, db0, g0, es0;              // half level k: pressure force, buoyancy, gravity, eth
    double gm64, g064, em64, e064;       // half levels k-1, k in FP64: gravity, eth
    real vt[6], ga[3], ga3, ga3m, dd[3], vd[3];
  };
  NH_HD void init_stage(long, Stg&) const {}
  NH_HD void begin(Pre& p) const { p.have = false; }
  NH_HD bool stage_level(int k) const { return k >= d.kmin && k <= d.kmax; }
  NH_HD void stage_own(int k, unsigned o, const Stg& sg, const Pre&, real* v) const { stage(k, o, o, sg, v); }
  NH_HD void stage(int k, unsigned o, unsigned, const Stg&, real* v) const {
    for (int q = 0; q < 3; ++q) v[q] = at_off(pk.prog + (long)(1 + q) * d.NF, o);
    v[3] = at_off(pk.eth, o);
    // the pressure at the level of its gradient (kmin -> kmin+1), pregd
    const int kg = (k == d.kmin) ? k + 1 : k;
    v[4] = (real)((double)at_off(pk.diag + I_PRE * d.NF + (long)(kg - k) * d.g * d.g, o) - pk.G.pre_bs[kg]) * real(1.0);
  }
  NH_HD void init_col(long ci, Col& col) const {
    for (int dd = 0; dd < 3; ++dd)
      for (int m = 0; m < 7; ++m) {
        col.cd[dd][m] = rc(pk.G.cdiv, d.nreg, dd * 7 + m, ci);
        col.cg[dd][m] = rc(pk.G.cgrad, d.nreg, dd * 7 + m, ci);
      }
    for (int q = 0; q < 3; ++q) col.x[q] = pk.G.gx[q * d.nreg + ci];
  }
  NH_HD void pole(int pb) const { pk(d.lall * d.kall + pb, 0); }
  // vertical pressure force, buoyancy and effective gravity at half level kk
  // from rhog and the pressure at kk and kk-1 (ViPath0P's dpgw, dbuo, gzt)
  template <class T>
  NH_HD void half(const VProf<T>& V, T grav, int kk, T rg, T rgl, double pr, double prl, double rgd, double rgld,
                  T& dp, T& db, T& g) const {
    const bool in = kk >= d.kmin + 1 && kk <= d.kmax;
    const Geo& G = pk.G;
    const int k1 = in ? kk : d.kmin + 1;   // a level both profiles have, unused otherwise
    const T prd = (T)(pr - G.pre_bs[k1]) * T(1.0), prdl = (T)(prl - G.pre_bs[k1 - 1]) * T(1.0);
    const T rd = (T)(rgd - G.rho_bs[k1]) * T(1.0), rdl = (T)(rgld - G.rho_bs[k1 - 1]) * T(1.0);
    dp = in ? T(1.0) * (prd * T(1.0) - prdl * T(1.0)) * V.rdgzh[k1] : T(0.0);
    db = in ? -grav * (V.c2w0[k1] * rd + V.c2w1[k1] * rdl) : T(0.0);
    const int k2 = (kk < d.kmin) ? d.kmin : (kk > d.kall - 1) ? d.kall - 1 : kk;
    g = grav - (dp - db) / (V.c2w0[k2] * rg + V.c2w1[k2] * rgl);
  }
  NH_HD void half_both(int kk, real rg, real rgl, real pr, real prl, real& dp, real& db, real& g, double& g64) const {
    half<real>(pk.G, pk.c.GRAV, kk, rg, rgl, (double)pr, (double)prl, (double)(rg / real(1.0)),
               (double)(rgl / real(1.0)), dp, db, g);
    if constexpr (sizeof(real) == 8) {
      g64 = g;
    } else {
      double a, b;
      half<double>(pk.G.v64, pk.c.d.GRAV, kk, (double)rg, (double)rgl, (double)pr, (double)prl, (double)rg, (double)rgl,
                   a, b, g64);
    }
  }
  NH_HD double eth64(int kk, real e, real el) const {
    const VProf<double>& V = pk.G.v64;
    const int k2 = (kk < d.kmin) ? d.kmin : (kk > d.kall - 1) ? d.kall - 1 : kk;
    return V.afact[k2] * (double)e + V.bfact[k2] * (double)el;
  }
  NH_HD real eth_h(int kk, real e, real el) const {
    const int k2 = (kk > d.kall - 1) ? d.kall - 1 : kk;
    return pk.G.afact[k2] * e + pk.G.bfact[k2] * el;
  }
  NH_HD void pre(int k, unsigned o, const Stg&, Pre& p) const {
    const long NF = d.NF, gg = (long)d.g * d.g;
    const real* rg = pk.prog;
    const real* rw = pk.prog + 4 * NF;
    const real* pr = pk.diag + I_PRE * NF;
    if (p.have) {
      p.rgm = p.rg0; p.rg0 = p.rg1;
      p.pr0 = p.pr1; p.et0 = p.et1; p.rw0 = p.rw1;
      p.ga3m = p.ga3;
    } else {
      // levels k-2, k-1, k, clamped into range (a clamped value is not used)
      const long m1 = (k > 0) ? -gg : 0, m2 = (k > 1) ? m1 - gg : m1;
      const real rg2 = at_off(rg + m2, o), pr2 = at_off(pr + m2, o), et2 = at_off(pk.eth + m2, o);
      const real prm = at_off(pr + m1, o), etm = at_off(pk.eth + m1, o);
      p.rgm = at_off(rg + m1, o); p.rg0 = at_off(rg, o);
      p.pr0 = at_off(pr, o); p.et0 = at_off(pk.eth, o); p.rw0 = at_off(rw, o);
      p.ga3m = at_off(pk.gadv + 3 * NF + m1, o);
      real dp, db, g;
      half_both(k - 1, p.rgm, rg2, prm, pr2, dp, db, g, p.gm64);
      half_both(k, p.rg0, p.rgm, p.pr0, prm, p.dp0, p.db0, p.g0, p.g064);
      p.em64 = eth64(k - 1, etm, et2);
      p.e064 = eth64(k, p.et0, etm);
      p.es0 = eth_h(k, p.et0, etm);
      p.have = true;
    }
    const long up = (k < d.kall - 1) ? gg : 0;
    p.rg1 = at_off(rg + up, o); p.pr1 = at_off(pr + up, o); p.et1 = at_off(pk.eth + up, o); p.rw1 = at_off(rw + up, o);
    for (int q = 0; q < 6; ++q) p.vt[q] = at_off(pk.vt[q], o);
    for (int q = 0; q < 3; ++q) {
      p.ga[q] = at_off(pk.gadv + q * NF, o);
      p.dd[q] = at_off(pk.dd[q], o);
      p.vd[q] = at_off(pk.diag + (I_VX + q) * NF, o);
    }
    p.ga3 = at_off(pk.gadv + 3 * NF, o);
  }
  // ViPath0P::at for a regional point, term for term
  template <class NB>
  NH_HD void point(int k, unsigned o, const Col& col, Pre& p, NB nb) const {
    const long NF = d.NF;
    const long a = (long)(o / (unsigned)sizeof(real));   // the FP64 matrix is indexed in 64 bits
    const int kmin = d.kmin, kmax = d.kmax;
    const Geo& G = pk.G;
    const real R = pk.c.RADIUS;
    const real gx = col.x[0], gy = col.x[1], gz = col.x[2];
    const real Kh = pk.c.GAMMA_H;
    real dp1, db1, g1;
    double g164;
    half_both(k + 1, p.rg1, p.rg0, p.pr1, p.pr0, dp1, db1, g1, g164);
    const double e164 = eth64(k + 1, p.et1, p.et0);
    const real es1 = eth_h(k + 1, p.et1, p.et0);
    // hyperdiffusion tendency + momentum advection = large-step tendency
    real fvx = -(p.vt[0] * Kh + real(0.0)) * p.rg0;
    real fvy = -(p.vt[1] * Kh + real(0.0)) * p.rg0;
    real fvz = -(p.vt[2] * Kh + real(0.0)) * p.rg0;
    const real rgh = (k >= kmin) ? G.c2w0[k] * p.rg0 + G.c2w1[k] * p.rgm : real(0.0);
    const real fw = -(p.vt[3] * Kh + real(0.0)) * rgh;
    const real fe = -(p.vt[4] + real(0.0));
    const real fr = -(p.vt[5] + real(0.0));
    {
      const real prd = (fvx * gx + fvy * gy + fvz * gz) / R;
      fvx = fvx - prd * gx / R; fvy = fvy - prd * gy / R; fvz = fvz - prd * gz / R;
    }
    const real gadv_w = (k > kmin && k <= kmax) ? (G.c2w0[k] * p.ga3 + G.c2w1[k] * p.ga3m) : real(0.0);
    const real g00 = real(0.0) + fr, g05 = real(0.0) + fe;
    const real g01 = p.ga[0] + fvx, g02 = p.ga[1] + fvy, g03 = p.ga[2] + fvz;
    const real g04 = gadv_w + fw;
    real drhog = real(0.0), drhoge = real(0.0), pw = real(0.0);
    real dpg[3] = {real(0.0), real(0.0), real(0.0)};
    if (k >= kmin && k <= kmax) {
      // div(rhogv), div(rhogv eth) and the pressure gradient
      real s[2][3], gr[3];
#pragma unroll
      for (int m = 0; m < 7; ++m) {
        const real e = nb(m, 3), pm = nb(m, 4) * real(1.0);
        for (int q = 0; q < 3; ++q) {
          const real r3 = nb(m, q);
          const real t0 = col.cd[q][m] * (r3 * real(1.0)), t1 = col.cd[q][m] * (r3 * e * real(1.0));
          const real tg = col.cg[q][m] * pm;
          s[0][q] = (m == 0) ? t0 : s[0][q] + t0;
          s[1][q] = (m == 0) ? t1 : s[1][q] + t1;
          gr[q] = (m == 0) ? tg : gr[q] + tg;
        }
      }
      const real hd = s[0][0] + s[0][1] + s[0][2], he = s[1][0] + s[1][1] + s[1][2];
      const real vmh_hi = (k + 1 <= kmax) ? real(0.0) * real(1.0) + real(1.0) * p.rw1 * real(1.0) : real(0.0);
      const real vmh_lo = (k >= kmin + 1) ? real(0.0) * real(1.0) + real(1.0) * p.rw0 * real(1.0) : real(0.0);
      drhog = -hd - (vmh_hi - vmh_lo) * G.rdgz[k];
      const real ws_hi = (k + 1 <= kmax) ? real(0.0) * real(1.0) + real(1.0) * (p.rw1 * es1) * real(1.0) : real(0.0);
      const real ws_lo = (k >= kmin + 1) ? real(0.0) * real(1.0) + real(1.0) * (p.rw0 * p.es0) * real(1.0) : real(0.0);
      drhoge = -he - (ws_hi - ws_lo) * G.rdgz[k];
      for (int q = 0; q < 3; ++q) gr[q] = gr[q] + real(0.0);
      const real prd = (gr[0] * gx + gr[1] * gy + gr[2] * gz) / R;
      dpg[0] = gr[0] - prd * gx / R;
      dpg[1] = gr[1] - prd * gy / R;
      dpg[2] = gr[2] - prd * gz / R;
      pw = p.vd[0] * dpg[0] + p.vd[1] * dpg[1] + p.vd[2] * dpg[2] + G.w2c0[k] * (-g1 * p.rw1)
         + G.w2c1[k] * (-p.g0 * p.rw0);
    }
    at_off(pk.getot, o) = g05;
    at_off(pk.frhog, o) = g00;
    at_off(pk.gT + 0 * NF, o) = g00 + drhog;
    at_off(pk.gT + 1 * NF, o) = g01 - dpg[0] + p.dd[0] + real(0.0);
    at_off(pk.gT + 2 * NF, o) = g02 - dpg[1] + p.dd[1] + real(0.0);
    at_off(pk.gT + 3 * NF, o) = g03 - dpg[2] + p.dd[2] + real(0.0);
    at_off(pk.gT + 4 * NF, o) = g04 + real(0.0) * pk.c.ALPHA - p.dp0 + p.db0;
    at_off(pk.gT + 5 * NF, o) = g05 + drhoge + pw;
    if (k >= kmin + 1 && k <= kmax) {
      const VProf<double>& V = G.v64;
      const ConstsT<double>& C = pk.c.d;
      const double GCVovR = C.GRAV * C.CVdry / C.Rdry;
      const double ACVovRt2 = C.ALPHA * C.CVdry / C.Rdry / (pk.dt * pk.dt);
      const double Ca = (1.0 * V.rdgz[k] + 1.0 * V.rdgz[k - 1]) * 1.0;
      const double Cb = V.dfact[k] - V.cfact[k - 1];
      const double Cu1 = 1.0 * V.rdgz[k] * 1.0;
      const double Cu2 = 1.0 * 1.0 * GCVovR;
      const double Cl1 = 1.0 * V.rdgz[k] * 1.0;
      const double Cl2 = 1.0 * 1.0 * GCVovR;
      pk.Mc[a] = ACVovRt2 / 1.0 + V.rdgzh[k] * (Ca * p.e064 - Cb * (p.g064 + GCVovR));
      pk.Mu[a] = -V.rdgzh[k] * (Cu1 * e164 + V.cfact[k] * (g164 + Cu2));
      pk.Ml[a] = -V.rdgzh[k] * (Cl1 * p.em64 - V.dfact[k - 1] * (p.gm64 + Cl2));
    }
    p.dp0 = dp1; p.db0 = db1; p.g0 = g1; p.es0 = es1;
    p.gm64 = p.g064; p.g064 = g164;
    p.em64 = p.e064; p.e064 = e164;
  }
};

// minus the 7-point Laplacian of NFLD fields (HDiffPassP's Laplacians) as a
// column operator: the 7 Laplacian coefficients in registers.  P is the point
// kernel that does the pole centres (all of its fields) unless pole_off.
template <int NFLD, class P>
struct LapC {
  static constexpr const char* kName = (NFLD == 6) ? "hdiff_pass1" : "hdiff_pass2_lap";
  static constexpr int kNS = NFLD;
  static constexpr bool kMapped = NFLD == 4;   // the second pass reads the first's output
  P pk;
  Dims d;
  const real* in[NFLD];
  real* out[NFLD];
  bool pole_off;
  struct Col {
    real c[7];
  };
  struct Stg {};
  struct Pre {};
  NH_HD void init_stage(long, Stg&) const {}
  NH_HD void begin(Pre&) const {}
  NH_HD void pre(int, unsigned, const Stg&, Pre&) const {}
  NH_HD void stage_own(int k, unsigned o, const Stg& sg, const Pre&, real* v) const { stage(k, o, o, sg, v); }
  NH_HD bool stage_level(int) const { return true; }
  NH_HD void stage(int k, unsigned, unsigned om, const Stg&, real* v) const {
    for (int f = 0; f < NFLD; ++f) {
      const real x = at_off(in[f], om);
      v[f] = pk.sub[f] ? (real)((double)x - pk.sub[f][k]) : x;   // HDiffPassP::input
    }
  }
  NH_HD void init_col(long ci, Col& col) const {
    for (int m = 0; m < 7; ++m) col.c[m] = rc(pk.G.clap, d.nreg, m, ci);
  }
  NH_HD void pole(int pb) const {
    if (!pole_off) pk(d.lall * d.kall + pb, 0);
  }
  template <class NB>
  NH_HD void point(int, unsigned o, const Col& col, Pre&, NB nb) const {
    for (int f = 0; f < NFLD; ++f) {
      real r = col.c[0] * nb(0, f);
#pragma unroll
      for (int m = 1; m < 7; ++m) r = r + col.c[m] * nb(m, f);
      at_off(out[f], o) = -r;
    }
  }
};

// the transposed Laplacian of the hyperdiffusion adjoint at the interior
// points: ib(x) += -sum_m clap(x - off(m), m) ob(x - off(m)), summed over
// the interior sources in NegLapGA's order; per column the seven
// coefficients (zero where the source is not interior) in registers, ob
// staged per level.  NegLapGA's 1-D form does the border and pole points.
template <int NFLD>
struct LapTC {
  static constexpr const char* kName = "hdiff_lap_adj";
  static constexpr int kNS = NFLD;
  static constexpr bool kMapped = false;
  Dims d; Geo G;
  const real* ob[NFLD];
  real* ib[NFLD];
  struct Col {
    real c[7];
  };
  struct Stg {};
  struct Pre {
    real ib[NFLD];
  };
  NH_HD void init_stage(long, Stg&) const {}
  NH_HD void begin(Pre&) const {}
  NH_HD void pre(int, unsigned o, const Stg&, Pre& p) const {
    for (int f = 0; f < NFLD; ++f) p.ib[f] = at_off(ib[f], o);
  }
  NH_HD void stage_own(int k, unsigned o, const Stg& sg, const Pre&, real* v) const { stage(k, o, o, sg, v); }
  NH_HD bool stage_level(int) const { return true; }
  NH_HD void stage(int, unsigned o, unsigned, const Stg&, real* v) const {
    for (int f = 0; f < NFLD; ++f) v[f] = at_off(ob[f], o);
  }
  NH_HD void init_col(long ci, Col& col) const {
    const long gg = (long)d.g * d.g;
    const long r = ci % gg;
    const int j = (int)(r / d.g), i = (int)(r - (long)j * d.g);
    for (int m = 0; m < 7; ++m) {
      const int di = ((4201 >> (2 * m)) & 3) - 1, dj = ((421 >> (2 * m)) & 3) - 1;
      const int is = i - di, js = j - dj;
      const bool in = is >= 1 && is <= d.g - 2 && js >= 1 && js <= d.g - 2;
      col.c[m] = in ? rc(G.clap, d.nreg, m, ci - (long)di - (long)dj * d.g) : real(0.0);
    }
  }
  NH_HD void pole(int) const {}
  template <class NB>
  NH_HD void point(int, unsigned o, const Col& col, Pre& p, NB nb) const {
    // the source x - off(m) is staged neighbour opp(m)
    const int opp[7] = {0, 4, 5, 6, 1, 2, 3};
    for (int f = 0; f < NFLD; ++f) {
      real acc = real(0.0);
#pragma unroll
      for (int m = 0; m < 7; ++m) acc += col.c[m] * nb(opp[m], f);
      at_off(ib[f], o) = p.ib[f] + -acc;
    }
  }
};

// momentum advection and Coriolis (AdvMomP) as a column operator: the 21
// divergence coefficients and the column's position in registers; staged per
// level are the merged velocity v + w_full r/|r| (formed once per point, where
// the point kernel forms it once per neighbour) and the three momentum
// components.  A column marches upward and carries its own merged velocity at
// k - 1, k and k + 1; all loads of a level go out before its barrier.  Term for
// term the point kernel's arithmetic; pole centres run the point kernel.  At
// gl07 166 us per launch mixed, 314 FP64 (13 fields: 80 and 155 us of streaming);
// with the neighbouring levels loaded after the barrier 187 mixed, level-staged
// points 464 FP64.
struct AdvMomC {
  static constexpr const char* kName = "adv_mom";
  static constexpr int kNS = 6;
  static constexpr bool kMapped = false;
  AdvMomP pk;
  Dims d;
  struct Col {
    real c[3][7];
    real x[3];
  };
  struct Stg {
    real x[3];
  };
  struct Pre {
    bool have;
    real vm[3], v0[3], v1[3];   // merged velocity at levels k-1, k, k+1
    real w1, w2;                // w at half levels k+1, k+2
    real rw0, rw1, rg;          // rhogw at half levels k, k+1; density
  };
  NH_HD void init_stage(long ci, Stg& sg) const {
    for (int q = 0; q < 3; ++q) sg.x[q] = pk.G.gx[q * d.nreg + ci];
  }
  NH_HD void begin(Pre& p) const { p.have = false; }
  NH_HD bool stage_level(int k) const { return k >= d.kmin && k <= d.kmax; }
  // merged velocity at level kk (up levels above the point's) from w at its half levels
  NH_HD void merged(int kk, long up, unsigned o, const Stg& sg, real whi, real wlo, real* v) const {
    const long NF = d.NF;
    const real R = pk.c.RADIUS;
    const real wc = pk.G.cfact[kk] * whi + pk.G.dfact[kk] * wlo;
    v[0] = at_off(pk.diag + I_VX * NF + up, o) + wc * sg.x[0] / R;
    v[1] = at_off(pk.diag + I_VY * NF + up, o) + wc * sg.x[1] / R;
    v[2] = at_off(pk.diag + I_VZ * NF + up, o) + wc * sg.x[2] / R;
  }
  NH_HD void pre(int k, unsigned o, const Stg& sg, Pre& p) const {
    const long NF = d.NF, gg = (long)d.g * d.g;
    if (!stage_level(k)) return;
    const real* wd = pk.diag + I_W * NF;
    const real* rw = pk.prog + 4 * NF;
    if (p.have) {
      for (int q = 0; q < 3; ++q) { p.vm[q] = p.v0[q]; p.v0[q] = p.v1[q]; }
      p.w1 = p.w2;
      p.rw0 = p.rw1;
    } else {
      const real w0 = at_off(wd, o);
      p.w1 = at_off(wd + gg, o);
      p.rw0 = at_off(rw, o);
      if (k >= d.kmin + 1) merged(k - 1, -gg, o, sg, w0, at_off(wd - gg, o), p.vm);
      merged(k, 0, o, sg, p.w1, w0, p.v0);
      p.have = true;
    }
    if (k + 1 <= d.kmax) {
      p.w2 = at_off(wd + 2 * gg, o);
      merged(k + 1, gg, o, sg, p.w2, p.w1, p.v1);
      p.rw1 = at_off(rw + gg, o);
    }
    p.rg = at_off(pk.prog, o);
  }
  NH_HD void stage(int k, unsigned o, unsigned, const Stg& sg, real* v) const {
    const long NF = d.NF, gg = (long)d.g * d.g;
    const real* wd = pk.diag + I_W * NF;
    merged(k, 0, o, sg, at_off(wd + gg, o), at_off(wd, o), v);
    for (int q = 0; q < 3; ++q) v[3 + q] = at_off(pk.prog + (1 + q) * NF, o);
  }
  NH_HD void stage_own(int, unsigned o, const Stg&, const Pre& p, real* v) const {
    for (int q = 0; q < 3; ++q) {
      v[q] = p.v0[q];
      v[3 + q] = at_off(pk.prog + (1 + q) * d.NF, o);
    }
  }
  NH_HD void init_col(long ci, Col& col) const {
    for (int dd = 0; dd < 3; ++dd)
      for (int m = 0; m < 7; ++m) col.c[dd][m] = rc(pk.G.cdiv, d.nreg, dd * 7 + m, ci);
    for (int q = 0; q < 3; ++q) col.x[q] = pk.G.gx[q * d.nreg + ci];
  }
  NH_HD void pole(int pb) const { pk(d.lall * d.kall + pb, 0); }
  template <class NB>
  NH_HD void point(int k, unsigned o, const Col& col, Pre& p, NB nb) const {
    const long NF = d.NF;
    const int kmin = d.kmin, kmax = d.kmax;
    real* out = pk.out;
    if (k < kmin || k > kmax) {
      for (int q = 0; q < 4; ++q) at_off(out + q * NF, o) = real(0.0);
      return;
    }
    const Geo& G = pk.G;
    const real R = pk.c.RADIUS;
    const real* x0 = col.x;
    real sd[3][3];
#pragma unroll
    for (int m = 0; m < 7; ++m) {
      const real vv[3] = {nb(m, 0), nb(m, 1), nb(m, 2)};
      const real fx0 = nb(m, 3), fy0 = nb(m, 4), fz0 = nb(m, 5);
      const real cx = col.c[0][m], cy = col.c[1][m], cz = col.c[2][m];
      for (int q = 0; q < 3; ++q) {
        const real tx = cx * (fx0 * vv[q] * real(1.0));
        const real ty = cy * (fy0 * vv[q] * real(1.0));
        const real tz = cz * (fz0 * vv[q] * real(1.0));
        sd[0][q] = (m == 0) ? tx : sd[0][q] + tx;
        sd[1][q] = (m == 0) ? ty : sd[1][q] + ty;
        sd[2][q] = (m == 0) ? tz : sd[2][q] + tz;
      }
    }
    real div[3];
    for (int q = 0; q < 3; ++q) div[q] = sd[0][q] + sd[1][q] + sd[2][q];
    real hi[3] = {real(0.0), real(0.0), real(0.0)}, lo[3] = {real(0.0), real(0.0), real(0.0)};
    if (k + 1 <= kmax)
      for (int q = 0; q < 3; ++q)
        hi[q] = real(0.0) * real(1.0) + p.rw1 * (G.afact[k + 1] * p.v1[q] + G.bfact[k + 1] * p.v0[q]) * real(1.0);
    if (k >= kmin + 1)
      for (int q = 0; q < 3; ++q)
        lo[q] = real(0.0) * real(1.0) + p.rw0 * (G.afact[k] * p.v0[q] + G.bfact[k] * p.vm[q]) * real(1.0);
    real dvv[3];
    for (int q = 0; q < 3; ++q) dvv[q] = -div[q] - (hi[q] - lo[q]) * G.rdgz[k];
    const real gxc = x0[0] / R, gyc = x0[1] / R, gzc = x0[2] / R;
    const real rh = p.rg;
    const real dx = dvv[0] - (-real(2.0) * rh * (pk.c.OHM * p.v0[1]));
    const real dy = dvv[1] - (real(2.0) * rh * (pk.c.OHM * p.v0[0]));
    const real dz = dvv[2];
    const real prd = dx * gxc + dy * gyc + dz * gzc;
    at_off(out + 0 * NF, o) = dx - prd * gxc;
    at_off(out + 1 * NF, o) = dy - prd * gyc;
    at_off(out + 2 * NF, o) = dz - prd * gzc;
    at_off(out + 3 * NF, o) = prd * pk.c.ALPHA;
  }
};

NH_END
