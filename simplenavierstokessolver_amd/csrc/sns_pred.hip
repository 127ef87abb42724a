// sns_pred.hip -- implicit-x predictor: shared LU factorisation of the
// Crank-Nicolson x operators and the row kernel (gfx950).
//
// k_pred_rows evaluates, for one field and two adjacent rows per workgroup,
// the source terms and RK increments of src/temperature/update.c:11-122 and
// src/fluid/update_velocity.c:11-229 (sns_rows.h), then solves the
// Crank-Nicolson system in x of both rows (src/temperature/update.c:124-156,
// src/fluid/update_velocity.c:231-270, 381-414) with the shared LU tables.
//
// What bounds it on large grids is neither the HBM bytes (88 B per cell, 98.7
// folded; with what is read twice 4.6 GB and 4.5 TB/s on average at 4096x8192)
// nor the arithmetic, but the way from the L2: the three
// fields' workgroups read 18 rows for each row, and a run of columns that
// does not start on a cache line costs a line more.  Evaluating one block of
// a wave's own contiguous columns after the other, so that the lines at the
// block ends were fetched twice, took 0.96 ms where the waves of a workgroup
// side by side take 0.85; loads issued a block ahead did not help.  With one
// column per lane and unrolled blocks (15900 instructions, 1700 of them moving
// spilled scalars) it took 0.93.  us per launch, before and now: 4096x8192
// 929 and 865, folded 1288 and 1134; 2048x4096 244 and 202; 1537x3000 164 and
// 146, folded 221 and 203; 512x1024 24.1 and 18.5; 225x360 13.9 and 9.0, folded
// 16.9 and 11.4.
#include "sns_launch.h"
#include "sns_fast.h"
#include "sns_fused.h"
#include "sns_lu.h"
#include "sns_rows.h"

namespace sns {

// ------------------------------------------ shared LU factorisation of CN-x

// Coefficients of row r (0-based unknown index) of the CN-x operator of
// field f (0: T, 1: ux, 2: uy): src/temperature/update.c:141-149,
// src/fluid/update_velocity.c:253-261,398-406.
__device__ __forceinline__ void cnx_row(const Geo &g, const Tables &tb, int f, double pf, int r,
                                        double &l, double &c, double &u) {
  const int i = r + (f == 1 ? 2 : 1);
  const double coef_xm = f == 1 ? tb.nU_xm()[i - 1] : tb.nT_xm()[i - 1];
  const double coef_xp = f == 1 ? tb.nU_xp()[i - 1] : tb.nT_xp()[i - 1];
  const double coef_x0 = -coef_xm - coef_xp;
  l = -pf * coef_xm;
  u = -pf * coef_xp;
  c = 1. - pf * coef_x0;
}

__device__ __forceinline__ double cn_pf(const Geo &g, int f, double gdt) {
  return f == 0 ? gdt / g.two_sqrtPr_sqrtRa : (gdt * g.sqrtPr) / g.two_sqrtRa;
}

struct M22 {
  double a, b, c, d;
};
__device__ __forceinline__ M22 mmul(const M22 &x, const M22 &y) {  // x*y
  return {x.a * y.a + x.b * y.c, x.a * y.b + x.b * y.d, x.c * y.a + x.d * y.c,
          x.c * y.b + x.d * y.d};
}
// exact power-of-two rescaling (ratios of entries are unchanged)
__device__ __forceinline__ M22 mnorm(M22 m) {
  const double mx = fmax(fmax(fabs(m.a), fabs(m.b)), fmax(fabs(m.c), fabs(m.d)));
  if (mx == 0. || !isfinite(mx)) return m;
  const int e = ilogb(mx);
  return {ldexp(m.a, -e), ldexp(m.b, -e), ldexp(m.c, -e), ldexp(m.d, -e)};
}
__device__ __forceinline__ M22 mshfl_up(const M22 &m, int off) {
  return {__shfl_up(m.a, off), __shfl_up(m.b, off), __shfl_up(m.c, off), __shfl_up(m.d, off)};
}

// Thomas factorisation of the CN-x operator of field blockIdx.x for the
// substage blockIdx.y, written as the interleaved tables of sns_lu.h.  The
// pivot recurrence u'_i = u_i/(c_i - l_i u'_{i-1}) is the Moebius map of the
// vector v_i = [[0, u_i], [-l_i, c_i]] v_{i-1}, v_0 = (u_0, c_0), with
// u'_i = p_i/q_i and 1/pivot_i = q_{i-1}/q_i; the products of these 2x2
// matrices are scanned across the workgroup.
template <int NT, int M, class S>
__global__ void __launch_bounds__(NT) k_lu_factor(S src) {
  const LuFactorArgs a = src.get();
  constexpr int NW = NT / 64;
  __shared__ double wtot[NW][4];
  const Geo &g = a.g;
  const int f = blockIdx.x, s = blockIdx.y;
  const int n = f == 1 ? g.itot - 1 : g.itot;
  // substage gamma selected without indexing (keeps the argument block in registers)
  const double gam = s == 0 ? a.gamma[0] : s == 1 ? a.gamma[1] : a.gamma[2];
  const double dt = dt_of_step(a.dt, a.dtp, f == 0 && s == 0);
  const double pf = cn_pf(g, f, gam * dt);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  // chunk product of the row matrices (rows >= 1)
  M22 T = {1., 0., 0., 1.};
#pragma unroll
  for (int k = 0; k < M; k++) {
    const int r = t * M + k;
    if (r >= 1 && r < n) {
      double l, c, u;
      cnx_row(g, a.tb, f, pf, r, l, c, u);
      T = mnorm(mmul(M22{0., u, -l, c}, T));
    }
  }
  // inclusive scan within the wave (later chunks multiply from the left)
  M22 X = T;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const M22 o = mshfl_up(X, off);
    if (lane >= off) X = mnorm(mmul(X, o));
  }
  if (lane == 63) {
    wtot[wave][0] = X.a; wtot[wave][1] = X.b; wtot[wave][2] = X.c; wtot[wave][3] = X.d;
  }
  __syncthreads();
  M22 cin = {1., 0., 0., 1.};
  for (int w = 0; w < wave; w++)
    cin = mnorm(mmul(M22{wtot[w][0], wtot[w][1], wtot[w][2], wtot[w][3]}, cin));
  const M22 incl = mnorm(mmul(X, cin));
  M22 excl = mshfl_up(incl, 1);
  if (lane == 0) excl = cin;
  // v before this chunk's first row
  double l0, c0, u0;
  cnx_row(g, a.tb, f, pf, 0, l0, c0, u0);
  double p = excl.a * u0 + excl.b * c0, q = excl.c * u0 + excl.d * c0;
  double rr[M], al[M], be[M];
#pragma unroll
  for (int k = 0; k < M; k++) {
    const int r = t * M + k;
    rr[k] = al[k] = be[k] = 0.;
    if (r >= n) continue;
    double l, c, u;
    cnx_row(g, a.tb, f, pf, r, l, c, u);
    double up;
    if (r == 0) {
      rr[k] = 1. / c;
      up = u / c;
      p = u0;
      q = c0;
    } else {
      const double pn = u * q, qn = -l * p + c * q;
      rr[k] = q / qn;
      up = pn / qn;
      al[k] = -rr[k] * l;
      const double mx = fmax(fabs(pn), fabs(qn));
      const int e = ilogb(mx);
      p = ldexp(pn, -e);
      q = ldexp(qn, -e);
    }
    be[k] = (r == n - 1) ? 0. : -up;
  }
  double *base = a.out + (size_t)((s * 3 + f) * 3) * a.ntm;
#pragma unroll
  for (int k = 0; k < M; k++) {
    base[0 * a.ntm + k * NT + t] = rr[k];
    base[1 * a.ntm + k * NT + t] = al[k];
    base[2 * a.ntm + k * NT + t] = be[k];
  }
  // Header: P = the last row in 1..n-2 whose (r, al, be) differs bit for bit
  // from the row before (0 if none), so that rows P..n-2 all hold the
  // triple of row n-2; on a grid whose interior rows are alike the pivot
  // recurrence reaches that fixed point after a few rows.  Small systems
  // (n < 4) keep every row in the table (P = n).
  __shared__ double wlast[NW][3];
  __shared__ int wmax[NW];
  auto bits = [](double v) { return __double_as_longlong(v); };
  if (lane == 63) {
    wlast[wave][0] = rr[M - 1];
    wlast[wave][1] = al[M - 1];
    wlast[wave][2] = be[M - 1];
  }
  __syncthreads();
  double pr = __shfl_up(rr[M - 1], 1), pa = __shfl_up(al[M - 1], 1), pb = __shfl_up(be[M - 1], 1);
  if (lane == 0 && wave > 0) {
    pr = wlast[wave - 1][0];
    pa = wlast[wave - 1][1];
    pb = wlast[wave - 1][2];
  }
  int pt = 0;
#pragma unroll
  for (int k = 0; k < M; k++) {
    const int r = t * M + k;
    const double qr = k ? rr[k - 1] : pr, qa = k ? al[k - 1] : pa, qb = k ? be[k - 1] : pb;
    if (r >= 1 && r <= n - 2 &&
        (bits(rr[k]) != bits(qr) || bits(al[k]) != bits(qa) || bits(be[k]) != bits(qb)))
      pt = r;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) pt = max(pt, __shfl_xor(pt, off));
  if (lane == 0) wmax[wave] = pt;
  double *hdr = a.out + 27 * (size_t)a.ntm + (s * 3 + f) * kLuHdr;
#pragma unroll
  for (int k = 0; k < M; k++) {
    if (t * M + k == n - 2) {
      hdr[1] = rr[k];
      hdr[2] = al[k];
      hdr[3] = be[k];
    }
  }
  __syncthreads();
  if (t == 0) {
    int P = 0;
    for (int w = 0; w < NW; w++) P = max(P, wmax[w]);
    hdr[0] = (double)(n < 4 ? n : P);
    if (n < 2) hdr[1] = hdr[2] = hdr[3] = 0.;
  }
}

// -------------------------------------------------------- row predictor

template <int NT, int M>
struct PredRowsLds {
  double d[2][NT * (M + 1)];  // padded: chunk t starts at t*(M+1)
  double scr[4 * 2 * (NT / 64)];
};

template <int M>
__device__ __forceinline__ int pad_idx(int r) {
  return r + (int)((unsigned)r / M);
}

// Stencil blocks of kBlockCols adjacent columns.  Block k of wave w is number
// k*NW + w of the row, so the waves of a workgroup work side by side and share
// the cache lines at the block ends while those are in L1.
template <int NW>
__device__ __forceinline__ LanePos block_pos(int k, int i0, int n, int itot) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  return lane_pos(1 + (k * NW + wave) * kBlockCols - 2, i0, n, itot, 0, n, 1, 63);
}

// LDS slots of a lane's two unknowns; unknowns that are not the block's own go
// to the unused slot after the first chunk.
template <int M>
__device__ __forceinline__ void lds_slots(const LanePos &p, int &s0, int &s1) {
  s0 = p.out0 ? pad_idx<M>(p.ii) : M;
  s1 = p.out1 ? pad_idx<M>(p.ii + 1) : M;
}

// Whether a block has lanes with one own column: the first ux block (its
// pairs start at face 1, which is none) and the last block of an odd row end.
template <int F, int NW>
__device__ __forceinline__ bool block_edge(int k, int n) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = k * NW + wave;
  return (F == 1 && b == 0) || (b + 1) * kBlockCols >= n;
}

// The nk stencil blocks of one wave.
template <int F, int NT, int M, bool P2, bool FOLD, int IMY>
__device__ __forceinline__ void pred_stencils(const PredArgs &a, const RowSrc<F, FOLD> &q,
                                              PredRowsLds<NT, M> &L, int ja, int jb,
                                              bool write_a, int n, int i0, double dt,
                                              int nk) {
  const int itot = a.g.itot;
#pragma unroll 1
  for (int k = 0; k < nk; k++) {
    const LanePos p = block_pos<NT / 64>(k, i0, n, itot);
    const bool edge = block_edge<F, NT / 64>(k, n);
    Raw<F> r;
    double2 da, db;
    raw_load<F, P2, FOLD, 0>(a.tb, q, p, r);
    if constexpr (FOLD) raw_fold<F, P2, 1, 0, 0>(a, q, p, ja, jb, write_a, edge, dt, r);
    raw_eval<F, P2, 1, IMY, 0>(a, q, r, p, write_a, edge, dt, da);
    __builtin_amdgcn_sched_barrier(0);
    raw_load<F, P2, FOLD, 1>(a.tb, q, p, r);
    if constexpr (FOLD) raw_fold<F, P2, 1, 0, 1>(a, q, p, ja, jb, write_a, edge, dt, r);
    raw_eval<F, P2, 1, IMY, 1>(a, q, r, p, write_a, edge, dt, db);
    int s0, s1;
    lds_slots<M>(p, s0, s1);
    L.d[0][s0] = da.x;
    L.d[0][s1] = da.y;
    L.d[1][s0] = db.x;
    L.d[1][s1] = db.y;
  }
}

// The substage-start values of the own field in rows ja, jb (corrected as in
// raw_fold when folded), read again: the registers that would hold them (40 a
// thread, and blocks unrolled to index them) cost more.  On wide grids the rows
// are out of the L2 by then (0.8 GB per launch at 4096x8192).
template <int F, bool P2, bool FOLD>
__device__ __forceinline__ void own_load(const PredArgs &a, const RowSrc<F, FOLD> &q,
                                         const LanePos &p, double dt, double2 &oa, double2 &ob) {
  const Buf &f = F == 0 ? q.T : F == 1 ? q.U : q.V;
  oa = F == 1 ? bld2(f, p.u, q.u_a) : bld2(f, p.c, q.c_a);
  ob = F == 1 ? bld2(f, p.u, q.u_b) : bld2(f, p.c, q.c_b);
  if constexpr (FOLD && F != 0) {
    const double gdt = a.corr_gamma * dt;
    const double2 s_a = bld2(q.S, p.c, q.c_a), s_b = bld2(q.S, p.c, q.c_b);
    if constexpr (F == 1) {
      const double2 r = p.interior && a.tb.uniform
                            ? make_double2(a.tb.u_rdxc, a.tb.u_rdxc)
                            : bld2(q.tab, p.t, 3u * q.ts);
      const double wa = from_left(s_a.y), wb = from_left(s_b.y);
      oa = make_double2(proj_ux(oa.x, s_a.x, wa, gdt, r.x), proj_ux(oa.y, s_a.y, s_a.x, gdt, r.y));
      ob = make_double2(proj_ux(ob.x, s_b.x, wb, gdt, r.x), proj_ux(ob.y, s_b.y, s_b.x, gdt, r.y));
    } else {
      const double2 s_am = bld2(q.S, p.c, q.c_am);
      const double dy = a.tb.dy, rdy = a.tb.rdy;
      oa = make_double2(proj_uy<P2>(oa.x, s_a.x, s_am.x, gdt, dy, rdy),
                        proj_uy<P2>(oa.y, s_a.y, s_am.y, gdt, dy, rdy));
      ob = make_double2(proj_uy<P2>(ob.x, s_b.x, s_a.x, gdt, dy, rdy),
                        proj_uy<P2>(ob.y, s_b.y, s_a.y, gdt, dy, rdy));
    }
  }
}

// Final values in the blocks of the stencil phase: own + increment, or the
// increment itself when a y solve follows (IMY).  rowa, rowb: byte offsets of
// the rows in out; halo rows get copies where copy_* is set.
template <int F, int NT, int M, bool P2, bool FOLD, int IMY>
__device__ __forceinline__ void pred_emit(const PredArgs &a, const RowSrc<F, FOLD> &q,
                                          const Buf &out, const PredRowsLds<NT, M> &L,
                                          unsigned rowa, unsigned rowb, bool write_a,
                                          bool copy_a, bool copy_b, unsigned top, int n, int i0,
                                          double dt, int nk) {
#pragma unroll 1
  for (int k = 0; k < nk; k++) {
    const LanePos p = block_pos<NT / 64>(k, i0, n, a.g.itot);
    const bool edge = block_edge<F, NT / 64>(k, n);
    int s0, s1;
    lds_slots<M>(p, s0, s1);
    double2 va = make_double2(L.d[0][s0], L.d[0][s1]);
    double2 vb = make_double2(L.d[1][s0], L.d[1][s1]);
    if constexpr (IMY) {
      if (write_a) store_hist(out, p, edge, rowa, va);
      store_hist(out, p, edge, rowb, vb);
    } else {
      double2 oa, ob;
      own_load<F, P2, FOLD>(a, q, p, dt, oa, ob);
      va = make_double2(oa.x + va.x, oa.y + va.y);
      vb = make_double2(ob.x + vb.x, ob.y + vb.y);
      const unsigned o = F == 1 ? p.u : p.c;
      if (write_a) store_pair(out, p, edge, o, rowa, va);
      store_pair(out, p, edge, o, rowb, vb);
      if (copy_a) store_pair(out, p, edge, o, top, va);
      if (copy_b) store_pair(out, p, edge, o, 0u, vb);
    }
  }
}

// One workgroup's field F for rows ja and jb (write_a: row ja is written):
// stencils into LDS, the CN-x solve of both rows, final values.
template <int F, int NT, int M, bool P2, bool FOLD, int IMY>
__device__ __forceinline__ void pred_rows_body(const PredArgs &a, PredRowsLds<NT, M> &L, int ja,
                                               int jb, bool write_a) {
  const Geo &g = a.g;
  const int itot = g.itot;
  const int n = F == 1 ? itot - 1 : itot;
  const int i0 = F == 1 ? 2 : 1;
  const double dt = *a.dtp;
  // stencil blocks of this wave that hold unknowns
  constexpr int NW = NT / 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nb = (n + i0 - 1 + kBlockCols - 1) / kBlockCols;
  const int nk = wave < nb ? (nb - wave + NW - 1) / NW : 0;

  // ---- stencils and RK increments of both rows into LDS (lane order)
  const RowSrc<F, FOLD> q = row_src<F, FOLD>(a, ja, jb, n);
  pred_stencils<F, NT, M, P2, FOLD, IMY>(a, q, L, ja, jb, write_a, n, i0, dt, nk);
  __syncthreads();

  // ---- Crank-Nicolson in x of both rows (chunk order)
  double dd[2][M];
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int k = 0; k < M; k++) {
      const int r = threadIdx.x * M + k;
      dd[s][k] = r < n ? L.d[s][pad_idx<M>(r)] : 0.;
    }
  const double *b = a.lu + (size_t)(F * 3) * a.ntm;
  const double *h = a.lu_hdr + F * kLuHdr;
  const LuTabC<M> tab = {b, b + a.ntm, b + 2 * a.ntm, (int)h[0], n, h[1], h[2], h[3]};
  lu_solve_shared<NT, M, 2>(dd, tab, L.scr);
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int k = 0; k < M; k++) {
      const int r = threadIdx.x * M + k;
      if (r < n) L.d[s][pad_idx<M>(r)] = dd[s][k];
    }
  __syncthreads();

  // ---- final values with boundary values, or the increments for a y
  // solve, in the lane order of the stencil phase
  const unsigned pitch = (unsigned)(IMY ? n : F == 1 ? g.pu : g.pc) * 8u;
  const unsigned rows = (unsigned)(IMY ? g.jtot : g.jtot + 2);
  double *dst = IMY ? (F == 0 ? a.q_t : F == 1 ? a.q_u : a.q_v)
                    : (F == 0 ? a.out_t : F == 1 ? a.out_u : a.out_v);
  const Buf out = IMY || F == 1 ? buf_of(dst, pitch * rows) : cell_buf(dst, pitch * rows);
  const unsigned rowa = (unsigned)(IMY ? ja - 1 : ja) * pitch, rowb = rowa + pitch;
  const unsigned top = (unsigned)(g.jtot + 1) * pitch;
  const bool copy_a = !IMY && write_a && ja == 1, copy_b = !IMY && jb == g.jtot;
  pred_emit<F, NT, M, P2, FOLD, IMY>(a, q, out, L, rowa, rowb, write_a, copy_a, copy_b, top, n,
                                     i0, dt, nk);
  if constexpr (!IMY) {
    // wall values: both ends of both rows, one thread each
    if (threadIdx.x < 4) {
      const bool right = threadIdx.x & 1, second = threadIdx.x & 2;
      const double wv = F != 0 ? 0. : right ? -0.5 : +0.5;
      const unsigned wo = F == 1 ? (right ? (unsigned)itot * 8u : 0u)
                                 : (right ? (unsigned)(itot + 2) * 8u : 8u);
      if (second || write_a) bst(out, wo, second ? rowb : rowa, wv);
      // halo rows: ux and uy only (T's walls end at rows 1 and jtot)
      if (F != 0 && (second ? copy_b : copy_a)) bst(out, wo, second ? 0u : top, wv);
    }
  }
}

// Workgroup w: field w % nfld (+1 without the temperature equation) of rows
// a = 2q+1 and b = a+1, q = w / nfld.  For odd jtot the last pair is shifted
// down to (jtot-1, jtot) and writes row b only.  Consecutive w share an XCD.
// FOLD: the fields are corrected as they are loaded (raw_fold).  IMY: a y
// solve follows, the increments are the output.
template <int NT, int M, bool P2, bool FOLD, int IMY, class S>
__global__ void __launch_bounds__(NT, (pred_waves<P2, FOLD>())) k_pred_rows(S src, int nfld) {
  const PredArgs a = src.get();
  extern __shared__ double lds_raw[];
  PredRowsLds<NT, M> &L = *reinterpret_cast<PredRowsLds<NT, M> *>(lds_raw);
  const int w = xcd_groups(blockIdx.x, gridDim.x, kPredGroup * nfld);
  const int q = w / nfld;
  const int f = w % nfld + (nfld == 3 ? 0 : 1);
  const int ja = min(2 * q + 1, a.g.jtot - 1), jb = ja + 1;
  const bool write_a = ja == 2 * q + 1;
  if (f == 0) pred_rows_body<0, NT, M, P2, FOLD, IMY>(a, L, ja, jb, write_a);
  else if (f == 1) pred_rows_body<1, NT, M, P2, FOLD, IMY>(a, L, ja, jb, write_a);
  else pred_rows_body<2, NT, M, P2, FOLD, IMY>(a, L, ja, jb, write_a);
}

// ---------------------------------------------------------------- launch

template <int NT, int M, bool P2, bool FOLD, int IMY, class S>
static void pred_rows_launch(hipStream_t s, const PredArgs &shape, S src, int nz) {
  const size_t lds = sizeof(PredRowsLds<NT, M>);
  static std::atomic<unsigned> attr{0};
  lds_limit_once((const void *)k_pred_rows<NT, M, P2, FOLD, IMY, S>, lds, attr);
  const int nfld = shape.with_temp ? 3 : 2;
  const int npair = (shape.g.jtot + 1) / 2;
  hipLaunchKernelGGL((k_pred_rows<NT, M, P2, FOLD, IMY, S>), dim3(npair * nfld, 1, nz), dim3(NT), lds,
                     s, src, nfld);
}

template <int NT, int M, class S>
static void lu_factor_launch(hipStream_t s, S src, int nz) {
  hipLaunchKernelGGL((k_lu_factor<NT, M, S>), dim3(3, 3, nz), dim3(NT), 0, s, src);
}

// Unknowns per thread: few where the rows' waves would leave SIMDs (1024)
// without one or with one only, so that a wave evaluates one or two stencil
// blocks instead of five and the substitutions are short; 8 where there are
// waves enough, since every thread pays the scans.  Measured (us, M = 8, 4, 2):
// 225x360 folded 14.4, 13.8, 11.4; 512x1024 19.9, 18.1, 20.1; 1024x2048 55.8,
// 56.0 (M = 4); batches of three 128x256 11.8, 10.5, 10.2, of four 512x1024
// 56.3, 59.4, 71.4.  It depends on the grid alone, so instances agree bit for
// bit alone and in a batch.
RowShape row_shape(int itot, int jtot) {
  RowShape r{0, 8};
  if (itot > 8192) return r;
  const long rows = 3l * ((jtot + 1) / 2);
  if (itot <= 512 && rows * ((itot + 127) / 128) <= 2048) r.M = 2;
  else if (itot <= 1024 && rows * ((itot + 255) / 256) <= 4096) r.M = 4;
  r.NT = 64;
  while (r.NT * r.M < itot) r.NT *= 2;
  return r;
}

bool pred_impx_supported(int itot) { return row_shape(itot, 4).NT > 0; }

// With the division sequence the folded kernel needs 148 registers; above 2048
// columns the rows' LDS leaves one workgroup of eight waves a CU beside 128, and
// there the sequence of predictor and correction kernel is the faster one.  us
// per step, folded (128 registers, 19 spilled) and in sequence: 2049x1024 412
// and 399, 3001x512 354 and 327, 4096x512 446 and 403, 4096x2048 1677 and 1641,
// 8192x1024 1711 and 1653; at 2048x1024 342 and 365, at 1100x256 137 and 144.
bool pred_folds(int itot, int jtot, bool p2) {
  return p2 || row_shape(itot, jtot).NT <= kFoldDivThreads;
}

int lu_table_entries(int itot, int jtot) {
  const RowShape r = row_shape(itot, jtot);
  return r.NT * r.M;
}

template <class S>
static void lu_factor_dispatch(hipStream_t s, const Geo &g, S src, int nz) {
#define SNS_CALL(NT_, M_) lu_factor_launch<NT_, M_>(s, src, nz)
  SNS_ROW_DISPATCH(row_shape(g.itot, g.jtot), SNS_CALL);
#undef SNS_CALL
}

void launch_lu_factor(hipStream_t s, const LuFactorArgs &a) {
  lu_factor_dispatch(s, a.g, ArgOne<LuFactorArgs>{a}, 1);
}

void launch_lu_factor_batch(hipStream_t s, const LuFactorArgs &shape, const LuFactorArgs *dev,
                            int nz) {
  lu_factor_dispatch(s, shape.g, arg_batch<LuFactorArgs>(dev), nz);
}

template <bool P2, bool FOLD, int IMY, class S>
static void pred_rows_select(hipStream_t s, const PredArgs &shape, S src, int nz) {
#define SNS_CALL(NT_, M_)                                       \
  if constexpr (!FOLD || P2 || NT_ <= kFoldDivThreads) /* pred_folds */ \
    pred_rows_launch<NT_, M_, P2, FOLD, IMY>(s, shape, src, nz)
  SNS_ROW_DISPATCH(row_shape(shape.g.itot, shape.g.jtot), SNS_CALL);
#undef SNS_CALL
}

// Power-of-two divisors select the kernel that divides by multiplying; a
// psi argument the one that applies the previous substage's correction.
template <class S>
static void pred_rows_dispatch(hipStream_t s, const PredArgs &shape, S src, int nz) {
  const bool p2 = shape.tb.pow2, fold = shape.psi != nullptr;
  const bool imy = shape.tr.implicity;  // excludes fold
  if (p2 && fold) pred_rows_select<true, true, 0>(s, shape, src, nz);
  else if (p2 && imy) pred_rows_select<true, false, 1>(s, shape, src, nz);
  else if (p2) pred_rows_select<true, false, 0>(s, shape, src, nz);
  else if (fold) pred_rows_select<false, true, 0>(s, shape, src, nz);
  else if (imy) pred_rows_select<false, false, 1>(s, shape, src, nz);
  else pred_rows_select<false, false, 0>(s, shape, src, nz);
}

void launch_pred_rows(hipStream_t s, const PredArgs &a) {
  pred_rows_dispatch(s, a, ArgOne<PredArgs>{a}, 1);
}

void launch_pred_rows_batch(hipStream_t s, const PredArgs &shape, const PredArgs *dev, int nz) {
  pred_rows_dispatch(s, shape, arg_batch<PredArgs>(dev), nz);
}

}  // namespace sns
