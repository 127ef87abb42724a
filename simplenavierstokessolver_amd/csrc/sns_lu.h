// sns_lu.h -- Crank-Nicolson line solves with a shared LU factorisation.
//
// The x-direction Crank-Nicolson operators (1 - pf*Dxx) of T, ux and uy
// (src/temperature/update.c:141-154, src/fluid/update_velocity.c:248-267,
// 398-411) depend on the column index and on gamma*dt only, so every row of a
// substage solves the same matrix.  The Thomas factorisation of that matrix
// (the reference's u'_i and 1/pivot, src/linalg.c:9-30) is computed once per
// substage by k_lu_factor; each row then needs only the two first-order
// recurrences
//   forward  y_i = r_i d_i + al_i y_{i-1},     al_i = -r_i l_i
//   backward x_i = y_i + be_i x_{i+1},         be_i = -u'_i
// evaluated in parallel: every thread runs them over its chunk of M rows with
// zero carries, the chunk-end values are combined by an affine scan across
// the workgroup (wave shuffles, then one value per wave), and each element
// is corrected with the running products of al (P) and be (Q) across its
// chunk.  Rounding differs from the sequential sweep at the ulp level.
//
// Tables are stored interleaved, entry (t, k) of row i = t*M + k at
// [k*NT + t], so that the loads of a wave are contiguous.
#pragma once
#include <hip/hip_runtime.h>
#include "sns_fast.h"

namespace sns {

struct LuTab {
  const double *r, *al, *be;  // each NT*M entries, interleaved
  // entry k of this thread's chunk (interleaved index k*NT + t)
  __device__ __forceinline__ double get_r(int k, int nt) const { return r[k * nt + threadIdx.x]; }
  __device__ __forceinline__ double get_al(int k, int nt) const { return al[k * nt + threadIdx.x]; }
  __device__ __forceinline__ double get_be(int k, int nt) const { return be[k * nt + threadIdx.x]; }
};

// LuTab with the repeated rows folded: rows P..n-2 all hold the triple
// (rc, alc, bec) bit for bit (k_lu_factor's header), so only rows below P,
// the last row and the padding rows (zeros) are read from the tables; a
// thread whose chunk lies in P..n-2 reads nothing.
template <int M>
struct LuTabC {
  const double *r, *al, *be;  // each NT*M entries, interleaved
  int P, n;
  double rc, alc, bec;
  __device__ __forceinline__ bool in_table(int k) const {
    const int row = threadIdx.x * M + k;
    return row < P || row >= n - 1;
  }
  __device__ __forceinline__ double get_r(int k, int nt) const {
    return in_table(k) ? r[k * nt + threadIdx.x] : rc;
  }
  __device__ __forceinline__ double get_al(int k, int nt) const {
    return in_table(k) ? al[k * nt + threadIdx.x] : alc;
  }
  __device__ __forceinline__ double get_be(int k, int nt) const {
    return in_table(k) ? be[k * nt + threadIdx.x] : bec;
  }
};

// The same factors when al_i = -(r_i*l_i) and be_i = -(r_i*u_i) hold for
// 0 < i < n-1 with row coefficients l, u that do not depend on the system
// (only r does): l and u are interleaved tables like r.  Row 0 has al = 0 and
// be = -up0 (the first pivot's u'_0 = u_0/c_0), the last row be = 0.
struct LuTabLU {
  const double *r, *l, *u;
  int n, m;    // unknowns; entries per thread
  double up0;  // u'_0 of this system
  __device__ __forceinline__ double get_r(int k, int nt) const { return r[k * nt + threadIdx.x]; }
  __device__ __forceinline__ double get_al(int k, int nt) const {
    const int row = threadIdx.x * m + k;
    return row == 0 ? 0. : -(r[k * nt + threadIdx.x] * l[k * nt + threadIdx.x]);
  }
  __device__ __forceinline__ double get_be(int k, int nt) const {
    const int row = threadIdx.x * m + k;
    return row == n - 1 ? 0.
                        : (row == 0 ? -up0 : -(r[k * nt + threadIdx.x] * u[k * nt + threadIdx.x]));
  }
};

// LuTabLU with this thread's M reciprocal pivots loaded once into registers.
// Rows pfx+1 .. n-2 all have the pivot rinf (the factorisation found every
// pivot from row pfx on equal, bit for bit, up to row n-2), so only rows up
// to pfx and the last row are read from the table: a thread whose chunk
// holds none of them reads nothing.
// With cst set, l of rows 1..n-1 and u of rows 0..n-2 are the constants lc,
// uc (the table entries themselves), so the solve reads no coefficient table.
template <int M>
struct LuTabLUr {
  double rr[M];
  const double *l, *u;
  int n;
  double up0;
  bool cst;
  double lc, uc;
  __device__ __forceinline__ LuTabLUr(const double *r, const double *l_, const double *u_,
                                      int n_, double up0_, int pfx, double rinf, int nt,
                                      bool cst_ = false, double lc_ = 0., double uc_ = 0.)
      : l(l_), u(u_), n(n_), up0(up0_), cst(cst_), lc(lc_), uc(uc_) {
    const int row0 = threadIdx.x * M;
    if (row0 <= pfx || row0 + M - 1 >= n - 1) {
#pragma unroll
      for (int k = 0; k < M; k++) {
        const int row = row0 + k;
        rr[k] = (row <= pfx || row == n - 1) ? r[k * nt + threadIdx.x] : rinf;
      }
    } else {
#pragma unroll
      for (int k = 0; k < M; k++) rr[k] = rinf;
    }
  }
  __device__ __forceinline__ double get_r(int k, int) const { return rr[k]; }
  __device__ __forceinline__ double get_al(int k, int nt) const {
    const int row = threadIdx.x * M + k;
    return row == 0 ? 0. : -(rr[k] * (cst ? lc : l[k * nt + threadIdx.x]));
  }
  __device__ __forceinline__ double get_be(int k, int nt) const {
    const int row = threadIdx.x * M + k;
    return row == n - 1 ? 0.
                        : (row == 0 ? -up0 : -(rr[k] * (cst ? uc : u[k * nt + threadIdx.x])));
  }
};

// Exclusive scan over the threads of a workgroup of the affine maps
// x -> A x + B[f], NF of them with one common A (forward: thread t receives
// the composition of maps 0..t-1 applied to 0; reverse: of maps NT-1..t+1).
// Within a wave the maps are composed across 1, 2, 4 and 8 lanes of each row
// of 16 by DPP, then across the rows; then one map per wave through LDS.  The
// scan is a chain of latencies (a DPP step is a few cycles, a bpermute an LDS
// round trip): with all six steps by bpermute, and A scanned once per f, the
// x solves of the Poisson equation took 5.7 us at 128x192, 9.0 at 512x1024 and
// 131 at 4096x8192, now 4.4, 7.0 and 112.
// scr holds (1 + NF)*(NT/64) doubles; the caller orders any later write of
// scr after the reads here (another scan uses other scratch, and the callers'
// next LDS phase starts behind a barrier of their own).
template <int CTRL, int NF>
__device__ __forceinline__ void affine_step(double &A, double (&B)[NF]) {
  const double Ao = dpp_f64<CTRL>(A, 1.);
#pragma unroll
  for (int f = 0; f < NF; f++) B[f] = __builtin_fma(A, dpp_f64<CTRL>(B[f]), B[f]);
  A *= Ao;
}
template <int CTRL, int ROW_MASK, int NF>
__device__ __forceinline__ void affine_bcast(double &A, double (&B)[NF]) {
  const double Ao = dpp_f64<CTRL, ROW_MASK>(A, 1.);
#pragma unroll
  for (int f = 0; f < NF; f++)
    B[f] = __builtin_fma(A, dpp_f64<CTRL, ROW_MASK>(B[f], 0.), B[f]);
  A *= Ao;
}

template <int NT, int NF, bool REVERSE>
__device__ __forceinline__ void affine_scan_excl(double A, double (&B)[NF], double (&C)[NF],
                                                 double *scr) {
  constexpr int NW = NT / 64;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if constexpr (!REVERSE) {
    affine_step<0x111>(A, B);  // row_shr 1, 2, 4, 8
    affine_step<0x112>(A, B);
    affine_step<0x114>(A, B);
    affine_step<0x118>(A, B);
    affine_bcast<0x142, 0xa>(A, B);  // lane 15 of rows 0, 2 to rows 1, 3
    affine_bcast<0x143, 0xc>(A, B);  // lane 31 to rows 2, 3
  } else {
    affine_step<0x101>(A, B);  // row_shl 1, 2, 4, 8
    affine_step<0x102>(A, B);
    affine_step<0x104>(A, B);
    affine_step<0x108>(A, B);
    // first lane of rows 1, 3 to rows 0, 2, then lane 32 to rows 0, 1
#pragma unroll
    for (int half = 16; half <= 32; half *= 2) {
      const int src = (lane & ~(2 * half - 1)) | half;
      const bool ok = !(lane & half);
      const double Ao = __shfl(A, src);
#pragma unroll
      for (int f = 0; f < NF; f++) {
        const double Bo = __shfl(B[f], src);
        B[f] = ok ? __builtin_fma(A, Bo, B[f]) : B[f];
      }
      A = ok ? A * Ao : A;
    }
  }
  double cin[NF];
#pragma unroll
  for (int f = 0; f < NF; f++) cin[f] = 0.;
  if constexpr (NW > 1) {
    // wave totals
    double *w0 = scr + wave * (1 + NF);
    if (lane == (REVERSE ? 0 : 63)) {
      w0[0] = A;
#pragma unroll
      for (int f = 0; f < NF; f++) w0[1 + f] = B[f];
    }
    __syncthreads();
    for (int k = 0; k < (REVERSE ? NW - 1 - wave : wave); k++) {
      const double *w = scr + (REVERSE ? NW - 1 - k : k) * (1 + NF);
#pragma unroll
      for (int f = 0; f < NF; f++) cin[f] = __builtin_fma(w[0], cin[f], w[1 + f]);
    }
  }
#pragma unroll
  for (int f = 0; f < NF; f++) {
    const double incl = __builtin_fma(A, cin[f], B[f]);  // value after this thread's map
    const double prev = REVERSE ? from_right(incl) : from_left(incl);
    C[f] = lane == (REVERSE ? 63 : 0) ? cin[f] : prev;
  }
}

// Solve NS systems that share one matrix (tab) for this thread's chunk
// d[s][0..M-1] (unknowns t*M .. t*M+M-1).  scr holds 4*NS*(NT/64) doubles
// (the two scans' scratch apart); the caller places a barrier between this
// call and its next write of scr.
template <int NT, int M, int NS, class TAB = LuTab>
__device__ __forceinline__ void lu_solve_shared(double (&d)[NS][M], const TAB &tab,
                                                double *scr) {
  double B[NS], C[NS];
  double P[M];
  {
    double y[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) y[s] = 0.;
    double pr = 1.;
#pragma unroll
    for (int k = 0; k < M; k++) {
      const double r = tab.get_r(k, NT), al = tab.get_al(k, NT);
      pr *= al;
      P[k] = pr;
#pragma unroll
      for (int s = 0; s < NS; s++) {
        y[s] = __builtin_fma(al, y[s], r * d[s][k]);
        d[s][k] = y[s];
      }
    }
#pragma unroll
    for (int s = 0; s < NS; s++) B[s] = y[s];
  }
  affine_scan_excl<NT, NS, false>(P[M - 1], B, C, scr);
  double Q[M];
  {
    double x[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) x[s] = 0.;
    double pr = 1.;
#pragma unroll
    for (int k = M - 1; k >= 0; k--) {
      const double be = tab.get_be(k, NT);
      pr *= be;
      Q[k] = pr;
#pragma unroll
      for (int s = 0; s < NS; s++) {
        x[s] = __builtin_fma(be, x[s], __builtin_fma(P[k], C[s], d[s][k]));
        d[s][k] = x[s];
      }
    }
#pragma unroll
    for (int s = 0; s < NS; s++) B[s] = x[s];
  }
  affine_scan_excl<NT, NS, true>(Q[0], B, C, scr + (1 + NS) * (NT / 64));
#pragma unroll
  for (int s = 0; s < NS; s++)
#pragma unroll
    for (int k = 0; k < M; k++) d[s][k] = __builtin_fma(Q[k], C[s], d[s][k]);
}

}  // namespace sns
