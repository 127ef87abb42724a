// sns_rows.h -- source terms of two adjacent rows, two columns per lane (gfx950).
//
// The predictors evaluate the source terms and RK increments of
// src/temperature/update.c:11-122 and src/fluid/update_velocity.c:11-229 for
// pairs of rows.  Lane l of a wave holds columns i, i+1 of a run of adjacent
// column pairs (i odd): one 16-byte access moves both, x neighbours are the
// lane's own other column or come from the adjacent lane (DPP), the y
// neighbours of one row are the centre values of the other, and the column
// metrics serve both rows.
//
// The vector memory path takes a wave's load in about 17 cycles and a store in
// about 40 whatever its width (8 or 16 bytes a lane, measured), so two columns
// per lane halve that time: with one, the row predictor took 0.94 ms at
// 4096x8192 and still 0.50 with every access out of range (no memory traffic
// at all).
#pragma once
#include "sns_fast.h"
#include "sns_fused.h"
#include "sns_buf.h"

namespace sns {

// Columns of a block: two per lane, lanes 0 and 63 hold the neighbours
constexpr int kBlockCols = 124;

// Row pairs of one XCD's run before the next XCD's (xcd_groups): rows that
// share neighbours meet in an L2, and the eight runs stay close in memory.
// 2048x4096 IMP-IMP, us per launch: 234 with an eighth of the grid per XCD,
// 232, 227, 226 and 224 with 1, 4, 8 and 64 pairs, 256 without any order.
constexpr int kPredGroup = 64;

// Waves per SIMD: the two rows' LDS leaves 4 (two workgroups per CU) at the
// widest rows; the folded kernel with the division sequence needs 148
// registers, so it takes 3 (1537x3000: 206 us, 220 with 4 and spilled
// registers), which its widest workgroup, of kFoldDivThreads, still fills.
constexpr int kFoldDivThreads = 256;
template <bool P2, bool FOLD>
constexpr int pred_waves() {
  return FOLD && !P2 ? 3 : 4;
}

// Columns of a lane and their byte offsets: in rows of the cell arrays (c,
// relative to element -1, which the rows' padding holds), of ux (u), of the
// column tables (t) and of the RK history and increments (h).  out0, out1: the
// column is one of the block's own, whose results are stored.
struct LanePos {
  int i, ii;  // first column; its unknown index
  bool out0, out1;
  unsigned c, u, t, h;
  bool low;       // ii < 0: the pair at h is one unknown further right
  bool interior;  // columns i-1..i+2 of all 64 lanes lie in 2..itot-1 (wave-uniform)
};

// Lane position for a run of column pairs whose lane 0 holds column i_first
// (odd, wave-uniform); own columns have unknown indices in [lo, hi) and lie in
// lanes l0..l1-1.
__device__ __forceinline__ LanePos lane_pos(int i_first, int i0, int n, int itot, int lo, int hi,
                                            int l0, int l1) {
  const int lane = threadIdx.x & 63;
  LanePos p;
  p.i = i_first + 2 * lane;
  p.ii = p.i - i0;
  const bool own = lane >= l0 && lane < l1;
  p.out0 = own && p.ii >= lo && p.ii < hi;
  p.out1 = own && p.ii + 1 >= lo && p.ii + 1 < hi;
  const int ic = min(p.i, itot | 1);  // the last pair that holds a column
  p.c = (unsigned)(max(ic, -1) + 1) * 8u;
  p.u = (unsigned)(max(ic, 1) - 1) * 8u;
  p.t = p.u;
  p.low = p.ii < 0;
  p.h = (unsigned)clampi(p.ii, 0, n - 1) * 8u;
  p.interior = i_first >= 3 && i_first + 128 <= itot - 1;
  return p;
}

// The arrays of field F (0: T, 1: ux, 2: uy) for one pair of rows: buffer
// descriptors, and the byte offsets of the rows.  A descriptor of 0 bytes
// reads zeros and drops stores, so an array that a substage does not use
// (the history it does not read or write, T without buoyancy) takes no
// branch.  The cell arrays' descriptors start one element early (LanePos).
template <int F, bool FOLD>
struct RowSrc {
  Buf T, U, V, P, S, hr, hw, pout;
  Buf tab;                       // column tables
  unsigned ts;                   // bytes per table
  unsigned c_am, c_a, c_b, c_bp; // cell rows ja-1, ja, jb, jb+1
  unsigned u_am, u_a, u_b, u_bp; // ux rows
  unsigned h_a, h_b;             // history rows
  unsigned s_mm, p_am;           // psi row ja-2, pressure row ja-1 (folded uy)
};

__device__ __forceinline__ Buf cell_buf(const double *p, unsigned bytes) {
  return buf_of(p - 1, bytes ? bytes + 8u : 0u);
}

template <int F, bool FOLD>
__device__ __forceinline__ RowSrc<F, FOLD> row_src(const PredArgs &a, int ja, int jb, int n) {
  const Geo &g = a.g;
  RowSrc<F, FOLD> r;
  const unsigned wc = (unsigned)g.pc * 8u, wu = (unsigned)g.pu * 8u;
  const unsigned nc = wc * (unsigned)(g.jtot + 2), nu = wu * (unsigned)(g.jtot + 2);
  const unsigned nh = (unsigned)n * 8u * (unsigned)g.jtot;
  double *H = F == 0 ? a.hist_t : (F == 1 ? a.hist_ux : a.hist_uy);
  r.T = cell_buf(a.temp, F == 0 || a.forcing ? nc : 0u);
  r.U = buf_of(a.ux, nu);
  r.V = cell_buf(a.uy, nc);
  r.P = cell_buf(a.p, nc);
  r.S = cell_buf(a.psi, FOLD ? nc : 0u);
  r.hr = buf_of(H, a.read_hist ? nh : 0u);
  r.hw = buf_of(H, a.write_hist ? nh : 0u);
  r.pout = cell_buf(a.p_out, FOLD ? nc : 0u);
  r.ts = (unsigned)a.tb.stride * 8u;
  r.tab = buf_of(a.tb.t, r.ts * (unsigned)kTables);
  r.c_am = (unsigned)(ja - 1) * wc;
  r.c_a = r.c_am + wc;
  r.c_b = r.c_a + wc;
  r.c_bp = r.c_b + wc;
  r.u_am = (unsigned)(ja - 1) * wu;
  r.u_a = r.u_am + wu;
  r.u_b = r.u_a + wu;
  r.u_bp = r.u_b + wu;
  r.h_a = (unsigned)(ja - 1) * (unsigned)n * 8u;
  r.h_b = (unsigned)(jb - 1) * (unsigned)n * 8u;
  r.s_mm = ja >= 2 ? r.c_am - wc : (unsigned)(g.jtot - 1) * wc;
  r.p_am = ja == 1 ? (unsigned)g.jtot * wc : r.c_am;
  return r;
}

// Column metrics of a lane's two columns (tables of sns_fast.h).
struct Metric {
  double2 dxc, rdxc, dxf, rdxf, wm, wp;
};

// The values one lane loads for the two rows: the substage-start fields
// around rows ja, jb and the RK history; folded, also psi.
template <int F>
struct Raw;
template <>
struct Raw<0> {
  // the field's own values, what the increments are added to
  __device__ __forceinline__ double2 own_a() const { return t_a; }
  __device__ __forceinline__ double2 own_b() const { return t_b; }
  double2 t_am, t_a, t_b, t_bp, u_a, u_b, v_a, v_b, v_bp, ba, bb;
  double2 s_am, s_a, s_b, s_bp;
  Metric x;
};
template <>
struct Raw<1> {
  // the field's own values, what the increments are added to
  __device__ __forceinline__ double2 own_a() const { return u_a; }
  __device__ __forceinline__ double2 own_b() const { return u_b; }
  double2 u_am, u_a, u_b, u_bp, v_a, v_b, v_bp, p_a, p_b, t_a, t_b, ba, bb;
  double2 s_am, s_a, s_b, s_bp;
  Metric x;
};
template <>
struct Raw<2> {
  // the field's own values, what the increments are added to
  __device__ __forceinline__ double2 own_a() const { return v_a; }
  __device__ __forceinline__ double2 own_b() const { return v_b; }
  double2 v_am, v_a, v_b, v_bp, u_am, u_a, u_b, p_am, p_a, p_b, ba, bb;
  double2 s_amm, s_am, s_a, s_b, s_bp;
  Metric x;
};

template <int F, bool P2, bool FOLD>
__device__ __forceinline__ Metric metric_load(const Tables &tb, const RowSrc<F, FOLD> &q,
                                              const LanePos &p) {
  Metric x;
  if (p.interior && tb.uniform) {
    auto two = [](double v) { return make_double2(v, v); };
    x.dxc = two(tb.u_dxc);
    x.rdxc = two(tb.u_rdxc);
    x.dxf = two(tb.u_dxf);
    x.rdxf = two(tb.u_rdxf);
    x.wm = x.wp = two(F == 1 ? tb.u_cU : tb.u_cT);
  } else {
    x.dxf = bld2(q.tab, p.t, 0u);
    x.dxc = bld2(q.tab, p.t, q.ts);
    x.rdxf = bld2(q.tab, p.t, 2u * q.ts);
    x.rdxc = bld2(q.tab, p.t, 3u * q.ts);
    x.wm = bld2(q.tab, p.t, (F == 1 ? 6u : 4u) * q.ts);
    x.wp = bld2(q.tab, p.t, (F == 1 ? 7u : 5u) * q.ts);
  }
  return x;
}

// The pair of history values of the lane's columns (F = 1: the first lane's
// pair starts one unknown early; it reads the pair at 0 and takes its first)
template <int F>
__device__ __forceinline__ double2 hist_load(Buf h, const LanePos &p, unsigned row) {
  const double2 v = bld2(h, p.h, row);
  if constexpr (F == 1) return make_double2(v.x, p.low ? v.x : v.y);
  return v;
}

// PART 0: what row ja needs, 1: what row jb needs besides.  k_pred_rows loads and
// evaluates the rows one after the other, which keeps a third fewer values in
// registers than loading both first; k_pred_exp, bound by latency, loads both.
template <int F, bool P2, bool FOLD, int PART>
__device__ __forceinline__ void raw_load(const Tables &tb, const RowSrc<F, FOLD> &q,
                                         const LanePos &p, Raw<F> &r) {
  if constexpr (PART == 0) {
    r.x = metric_load<F, P2, FOLD>(tb, q, p);
    if constexpr (FOLD) {
      if constexpr (F == 2) r.s_amm = bld2(q.S, p.c, q.s_mm);
      r.s_am = bld2(q.S, p.c, q.c_am);
      r.s_a = bld2(q.S, p.c, q.c_a);
      r.s_b = bld2(q.S, p.c, q.c_b);
    }
    r.v_a = bld2(q.V, p.c, q.c_a);
    r.v_b = bld2(q.V, p.c, q.c_b);
    r.u_a = bld2(q.U, p.u, q.u_a);
    if constexpr (F == 0) {
      r.t_am = bld2(q.T, p.c, q.c_am);
      r.t_a = bld2(q.T, p.c, q.c_a);
      r.t_b = bld2(q.T, p.c, q.c_b);
    } else if constexpr (F == 1) {
      r.u_am = bld2(q.U, p.u, q.u_am);
      r.u_b = bld2(q.U, p.u, q.u_b);
      r.p_a = bld2(q.P, p.c, q.c_a);
      r.t_a = bld2(q.T, p.c, q.c_a);
    } else {
      r.v_am = bld2(q.V, p.c, q.c_am);
      r.u_am = bld2(q.U, p.u, q.u_am);
      r.p_am = bld2(q.P, p.c, FOLD ? q.p_am : q.c_am);
      r.p_a = bld2(q.P, p.c, q.c_a);
    }
    r.ba = hist_load<F>(q.hr, p, q.h_a);
  } else {
    if constexpr (FOLD) r.s_bp = bld2(q.S, p.c, q.c_bp);
    r.v_bp = bld2(q.V, p.c, q.c_bp);
    if constexpr (F == 0) {
      r.t_bp = bld2(q.T, p.c, q.c_bp);
      r.u_b = bld2(q.U, p.u, q.u_b);
    } else if constexpr (F == 1) {
      r.u_bp = bld2(q.U, p.u, q.u_bp);
      r.p_b = bld2(q.P, p.c, q.c_b);
      r.t_b = bld2(q.T, p.c, q.c_b);
    } else {
      r.u_b = bld2(q.U, p.u, q.u_b);
      r.p_b = bld2(q.P, p.c, q.c_b);
    }
    r.bb = hist_load<F>(q.hr, p, q.h_b);
  }
}

// Stores of a lane's pair of values at byte offset `at` of a row: both in one
// access, or the one that is the block's own (edge: the wave has such lanes;
// wave-uniform).
__device__ __forceinline__ void store_pair(Buf b, const LanePos &p, bool edge, unsigned at,
                                           unsigned row, double2 v) {
  bst2(b, p.out0 && p.out1 ? at : kOff, row, v);
  if (edge) {
    bst(b, p.out0 && !p.out1 ? at : kOff, row, v.x);
    bst(b, p.out1 && !p.out0 ? at + 8u : kOff, row, v.y);
  }
}

// ... of the RK history or increments (h of a low lane is that of its second
// column)
__device__ __forceinline__ void store_hist(Buf b, const LanePos &p, bool edge, unsigned row,
                                           double2 v) {
  bst2(b, p.out0 && p.out1 ? p.h : kOff, row, v);
  if (edge) {
    bst(b, p.out0 && !p.out1 ? p.h : kOff, row, v.x);
    bst(b, p.out1 && !p.out0 ? (p.low ? p.h : p.h + 8u) : kOff, row, v.y);
  }
}

// The previous substage's correction applied to the values raw_load took
// from its ux*, uy* and pressure, with the operations of k_corr (proj_* of
// sns_fast.h; P2 gives the same bits as its divisions).
//
// Faces 2..itot and cells 1..itot are corrected, the rest keep what the
// predictor stored, which is what k_corr leaves there:
//  * faces: psi's wall columns are exact copies of its columns 1 and itot,
//    so psi(i) - psi(i-1) is +0 at the wall faces 1 and itot+1 (and at the
//    clamped lanes past them) and the correction leaves those faces as they
//    are, with no select;
//  * uy: the wall columns 0 and itot+1 are kept by a select in the uy
//    field, the only one whose outputs read them;
//  * p: values outside cells 1..itot feed no output.
// Row ja-2 of the uy field wraps to jtot-1 for ja = 1 (periodic in y), and
// its pressure of row 0 is taken from row jtot: ux*, uy* and psi carry
// periodic copies in their halo rows, the pressure only once k_corr has
// written it.  The uy field stores the corrected pressure of its rows in
// p_out, the stores of k_corr for those cells.
template <int F, bool P2, int IMX, int IMY, int PART>
__device__ __forceinline__ void raw_fold(const PredArgs &a, const RowSrc<F, true> &q,
                                         const LanePos &p, int ja, int jb, bool write_a,
                                         bool edge, double dt, Raw<F> &r) {
  const Geo &g = a.g;
  const Tables &tb = a.tb;
  const int itot = g.itot;
  const double gdt = a.corr_gamma * dt;
  const double fac = -gdt / g.two_Re;
  const double dy = tb.dy, rdy = tb.rdy;
  // Lane shifts run on every lane, never under a divergent condition (a
  // shift there would read the inactive neighbour lanes as 0).
  auto west = [](double2 s) { return make_double2(from_left(s.y), s.x); };
  auto east = [](double2 s) { return make_double2(s.y, from_right(s.x)); };
  auto ux = [&](double2 &u, double2 s, double2 w) {
    u.x = proj_ux(u.x, s.x, w.x, gdt, r.x.rdxc.x);
    u.y = proj_ux(u.y, s.y, w.y, gdt, r.x.rdxc.y);
  };
  auto uy = [&](double2 v, double2 s, double2 south) {
    return make_double2(proj_uy<P2>(v.x, s.x, south.x, gdt, dy, rdy),
                        proj_uy<P2>(v.y, s.y, south.y, gdt, dy, rdy));
  };
  if constexpr (F == 0) {
    if constexpr (PART == 0) {
      ux(r.u_a, r.s_a, west(r.s_a));
      r.v_a = uy(r.v_a, r.s_a, r.s_am);
      r.v_b = uy(r.v_b, r.s_b, r.s_a);
    } else {
      ux(r.u_b, r.s_b, west(r.s_b));
      r.v_bp = uy(r.v_bp, r.s_bp, r.s_b);
    }
    return;
  }
  const double dxc_r = from_right(r.x.dxc.x), rdxc_r = from_right(r.x.rdxc.x);
  const ProjX x0 = {r.x.dxc.x, r.x.rdxc.x, r.x.dxc.y, r.x.rdxc.y, r.x.dxf.x, r.x.rdxf.x};
  const ProjX x1 = {r.x.dxc.y, r.x.rdxc.y, dxc_r, rdxc_r, r.x.dxf.y, r.x.rdxf.y};
  auto pr = [&](double2 &v, double2 s, double2 w, double2 e, double2 south, double2 north) {
    v.x = proj_p<P2>(v.x, s.x, w.x, e.x, south.x, north.x, x0, dy, rdy, fac, IMX, IMY);
    v.y = proj_p<P2>(v.y, s.y, w.y, e.y, south.y, north.y, x1, dy, rdy, fac, IMX, IMY);
  };
  if constexpr (F == 1) {
    if constexpr (PART == 0) {
      ux(r.u_am, r.s_am, west(r.s_am));
      ux(r.u_a, r.s_a, west(r.s_a));
      ux(r.u_b, r.s_b, west(r.s_b));
      r.v_a = uy(r.v_a, r.s_a, r.s_am);
      r.v_b = uy(r.v_b, r.s_b, r.s_a);
      pr(r.p_a, r.s_a, west(r.s_a), east(r.s_a), r.s_am, r.s_b);
    } else {
      ux(r.u_bp, r.s_bp, west(r.s_bp));
      r.v_bp = uy(r.v_bp, r.s_bp, r.s_b);
      pr(r.p_b, r.s_b, west(r.s_b), east(r.s_b), r.s_a, r.s_bp);
    }
  }
  if constexpr (F == 2) {
    // uy cells the correction moves
    const bool c0 = p.i >= 1 && p.i <= itot, c1 = p.i >= 0 && p.i + 1 <= itot;
    auto keep = [&](double2 &v, double2 w) {
      v.x = c0 ? w.x : v.x;
      v.y = c1 ? w.y : v.y;
    };
    // the pressure of row j (byte offset row) is stored, with its wall copies
    // (the blocks that hold cell 1 or itot); `halo` its periodic copy's row
    auto put = [&](double2 v, unsigned row, bool copy, unsigned halo) {
      store_pair(q.pout, p, edge, p.c, row, v);
      if (p.interior && !copy) return;
      // element 0 next to cell 1, element itot+1 next to cell itot
      const unsigned wl = p.out0 && p.i == 1 ? 8u : kOff, we = (unsigned)(itot + 2) * 8u;
      const unsigned w0 = p.out0 && p.i == itot ? we : kOff;
      const unsigned w1 = p.out1 && p.i + 1 == itot ? we : kOff;
      bst(q.pout, wl, row, v.x);
      bst(q.pout, w0, row, v.x);
      bst(q.pout, w1, row, v.y);
      if (copy) {
        store_pair(q.pout, p, edge, p.c, halo, v);
        bst(q.pout, wl, halo, v.x);
        bst(q.pout, w0, halo, v.x);
        bst(q.pout, w1, halo, v.y);
      }
    };
    if constexpr (PART == 0) {
      keep(r.v_am, uy(r.v_am, r.s_am, r.s_amm));
      keep(r.v_a, uy(r.v_a, r.s_a, r.s_am));
      keep(r.v_b, uy(r.v_b, r.s_b, r.s_a));
      ux(r.u_am, r.s_am, west(r.s_am));
      ux(r.u_a, r.s_a, west(r.s_a));
      pr(r.p_am, r.s_am, west(r.s_am), east(r.s_am), r.s_amm, r.s_a);
      pr(r.p_a, r.s_a, west(r.s_a), east(r.s_a), r.s_am, r.s_b);
      if (write_a)
        put(r.p_a, q.c_a, ja == 1, (unsigned)(g.jtot + 1) * (unsigned)g.pc * 8u);
    } else {
      keep(r.v_bp, uy(r.v_bp, r.s_bp, r.s_b));
      ux(r.u_b, r.s_b, west(r.s_b));
      pr(r.p_b, r.s_b, west(r.s_b), east(r.s_b), r.s_a, r.s_bp);
      put(r.p_b, q.c_b, jb == g.jtot, 0u);
    }
  }
}

// Source terms and RK increments of row ja (PART 0) or jb (1) from the loaded
// values; the new RK history is stored.
template <int F, bool P2, int IMX, int IMY, int PART, class Q>
__device__ __forceinline__ void raw_eval(const PredArgs &a, const Q &q, const Raw<F> &r,
                                         const LanePos &p, bool write_a, bool edge, double dt,
                                         double2 &d) {
  const Geo &g = a.g;
  const Tables &tb = a.tb;
  const Weights<IMX, IMY> w{};
  auto incr = [&](double2 A, double2 B, double2 G) {
    return make_double2(rk_incr(a.alpha, a.beta, a.gamma, dt, A.x, B.x, G.x),
                        rk_incr(a.alpha, a.beta, a.gamma, dt, A.y, B.y, G.y));
  };
  const Metric &m = r.x;
  double2 A, G;
  if constexpr (F == 1) {
    // faces: metrics DXC(i) and the weights; gradients over cells
    const FaceX x0 = {m.wm.x, m.wp.x, m.dxc.x, m.rdxc.x};
    const FaceX x1 = {m.wm.y, m.wp.y, m.dxc.y, m.rdxc.y};
    auto row = [&](double2 u_s, double2 u, double2 u_n, double2 v_s,
                   double2 v_n, double vl_s, double vl_n, double2 pc,
                   double2 t) {
      const double ul = from_left(u.y), ur = from_right(u.x);
      const double g0 = dv<P2>(-u.x + u.y, m.dxf.x, m.rdxf.x);
      const double g1 = dv<P2>(-u.y + ur, m.dxf.y, m.rdxf.y);
      const double gl = from_left(g1), pl = from_left(pc.y), tl = from_left(t.y);
      // without buoyancy T reads as 0
      const double tf0 = 0.5 * tl + 0.5 * t.x, tf1 = 0.5 * t.x + 0.5 * t.y;
      const UxPt p0 = {u.x, ul, u.y, u_s.x, u_n.x, vl_s, v_s.x, vl_n, v_n.x, pc.x, pl, tf0};
      const UxPt p1 = {u.y, u.x, ur, u_s.y, u_n.y, v_s.x, v_s.y, v_n.x, v_n.y, pc.y, pc.x, tf1};
      ux_src_g<P2>(g, tb, x0, p0, gl, g0, w, A.x, G.x);
      ux_src_g<P2>(g, tb, x1, p1, g0, g1, w, A.y, G.y);
    };
    if constexpr (PART == 0)
      row(r.u_am, r.u_a, r.u_b, r.v_a, r.v_b, from_left(r.v_a.y), from_left(r.v_b.y), r.p_a,
          r.t_a);
    else
      row(r.u_a, r.u_b, r.u_bp, r.v_b, r.v_bp, from_left(r.v_b.y), from_left(r.v_bp.y), r.p_b,
          r.t_b);
  } else {
    // cells: gradients over faces, DXC(i+1) at the right one
    const double dxc_r = from_right(m.dxc.x), rdxc_r = from_right(m.rdxc.x);
    const CellX x0 = {m.dxc.x, m.rdxc.x, m.dxc.y, m.rdxc.y, m.dxf.x, m.rdxf.x, m.wm.x, m.wp.x};
    const CellX x1 = {m.dxc.y, m.rdxc.y, dxc_r, rdxc_r, m.dxf.y, m.rdxf.y, m.wm.y, m.wp.y};
    if constexpr (F == 0) {
      auto row = [&](double2 t_s, double2 t, double2 t_n, double2 u,
                     double2 v_s, double2 v_n) {
        const double tr = from_right(t.x), ur = from_right(u.x);
        const double g0 = dv<P2>(-t.x + t.y, m.dxc.y, m.rdxc.y);
        const double g1 = dv<P2>(-t.y + tr, dxc_r, rdxc_r);
        const double gl = from_left(g1);
        const TempPt p0 = {t.x, t_s.x, t_n.x, u.x, u.y, v_s.x, v_n.x};
        const TempPt p1 = {t.y, t_s.y, t_n.y, u.y, ur, v_s.y, v_n.y};
        temp_src_g<P2>(g, tb, x0, p0, gl, g0, w, A.x, G.x);
        temp_src_g<P2>(g, tb, x1, p1, g0, g1, w, A.y, G.y);
      };
      if constexpr (PART == 0) row(r.t_am, r.t_a, r.t_b, r.u_a, r.v_a, r.v_b);
      else row(r.t_a, r.t_b, r.t_bp, r.u_b, r.v_b, r.v_bp);
    } else {
      auto row = [&](double2 v_s, double2 v, double2 v_n,
                     double2 u_s, double2 u, double ur_s, double ur,
                     double2 pc, double2 p_s) {
        const double vr = from_right(v.x);
        const double g0 = dv<P2>(-v.x + v.y, m.dxc.y, m.rdxc.y);
        const double g1 = dv<P2>(-v.y + vr, dxc_r, rdxc_r);
        const double gl = from_left(g1);
        const UyPt p0 = {v.x, v_s.x, v_n.x, u_s.x, u.x, u_s.y, u.y, pc.x, p_s.x};
        const UyPt p1 = {v.y, v_s.y, v_n.y, u_s.y, u.y, ur_s, ur, pc.y, p_s.y};
        uy_src_g<P2>(g, tb, x0, p0, gl, g0, w, A.x, G.x);
        uy_src_g<P2>(g, tb, x1, p1, g0, g1, w, A.y, G.y);
      };
      if constexpr (PART == 0)
        row(r.v_am, r.v_a, r.v_b, r.u_am, r.u_a, from_right(r.u_am.x), from_right(r.u_a.x),
            r.p_a, r.p_am);
      else
        row(r.v_a, r.v_b, r.v_bp, r.u_a, r.u_b, from_right(r.u_a.x), from_right(r.u_b.x), r.p_b,
            r.p_a);
    }
  }
  if (PART || write_a) store_hist(q.hw, p, edge, PART ? q.h_b : q.h_a, A);
  d = incr(A, PART ? r.bb : r.ba, G);
}

}  // namespace sns
