// sns_fused.hip -- fused substage kernels for the time-step hot path (gfx950).
//
// One RK substage (src/main.c:81-98) becomes these kernels:
//   pred : T, ux and uy predictors in one pass over the substage-start fields
//          (buoyancy from T in registers, RK history read/written in place),
//          writing T' (ping-pong buffer), ux*, uy* with their boundary values:
//          explicit x here, with Crank-Nicolson in x solved on chip for a
//          whole row in sns_pred.hip; the increments alone where y is implicit,
//          whose solve follows (sns_ysolve.hip);
//   poisson_fwd / poisson_x / poisson_inv : the potential (sns_poisson.hip, the
//          transforms up to 1024 rows in sns_poisson_one.hip);
//   corr : velocity correction and pressure update in one pass, plus on
//          the last substage the advective time-step bound for the next
//          step (a min-reduction over the corrected velocities).  With
//          explicit y the predictors of substages 2 and 3 apply the one of
//          substages 1 and 2 instead (step_args).
// The explicit and implicit diffusive parts, the RK increments and the
// boundary values follow the reference expression for expression (see
// sns_fast.h for the division scheme); only the line solves round
// differently.
#include "sns_launch.h"
#include "sns_fast.h"
#include "sns_fused.h"
#include "sns_rows.h"

namespace sns {

// ------------------------------------------------------------- predictor

// Explicit diffusion in x: the source terms of one field in one block of
// columns and one pair of rows per wave (sns_rows.h), the final values with
// boundary values, or the increments when a y solve follows (IMY).  FOLD: the
// previous substage's correction is applied to the fields as they are loaded.
//
// Small grids are bound by latency (a launch, a load, a chain of divisions, a
// store), larger ones by the loads: one thread per cell loaded 45 to 60 words
// one at a time, 10 neighbours of each field and the column metrics.  us per
// launch, one thread per cell and now: 700x1000 without T 19.1 and 14.3 (16.3
// with the rows loaded one after the other and two idle waves a workgroup),
// 128x192 5.4 and 5.2, folded 5.9 in place of 5.4 and a correction of 4.2.
// A step of 32x64 takes 79 us instead of 87, twenty of 128x192 1.55 ms
// instead of 1.79: two launches fewer a step.
constexpr int kExpWaves = 4;

template <int F, bool P2, bool FOLD, int IMY>
__device__ __forceinline__ void pred_exp_body(const PredArgs &a, int b, int ja, int jb,
                                              bool write_a, double dt) {
  const Geo &g = a.g;
  const int itot = g.itot;
  const int n = F == 1 ? itot - 1 : itot;
  const int i0 = F == 1 ? 2 : 1;
  const LanePos p = lane_pos(1 + b * kBlockCols - 2, i0, n, itot, 0, n, 1, 63);
  const bool edge = (F == 1 && b == 0) || (b + 1) * kBlockCols >= n;
  const RowSrc<F, FOLD> q = row_src<F, FOLD>(a, ja, jb, n);
  const unsigned pitch = (unsigned)(IMY ? n : F == 1 ? g.pu : g.pc) * 8u;
  const unsigned rows = (unsigned)(IMY ? g.jtot : g.jtot + 2);
  double *dst = IMY ? (F == 0 ? a.q_t : F == 1 ? a.q_u : a.q_v)
                    : (F == 0 ? a.out_t : F == 1 ? a.out_u : a.out_v);
  const Buf out = IMY || F == 1 ? buf_of(dst, pitch * rows) : cell_buf(dst, pitch * rows);
  // result of row j at byte offset `row`; `halo`: its periodic copy's row
  auto emit = [&](double2 d, double2 own, int j, bool copy, unsigned halo) {
    const unsigned row = (unsigned)(IMY ? j - 1 : j) * pitch;
    if constexpr (IMY) {
      store_hist(out, p, edge, row, d);
    } else {
      const double2 v = make_double2(own.x + d.x, own.y + d.y);
      const unsigned o = F == 1 ? p.u : p.c;
      store_pair(out, p, edge, o, row, v);
      if (copy) store_pair(out, p, edge, o, halo, v);
      if (p.interior) return;
      // wall values, by the lanes that hold the first and the last unknown
      // (T's walls end at rows 1 and jtot)
      const bool first = (p.out0 && p.ii == 0) || (p.out1 && p.ii + 1 == 0);
      const bool last = (p.out0 && p.ii == n - 1) || (p.out1 && p.ii + 1 == n - 1);
      const unsigned wl = first ? (F == 1 ? 0u : 8u) : kOff;
      const unsigned wr = last ? (unsigned)(F == 1 ? itot : itot + 2) * 8u : kOff;
      bst(out, wl, row, F == 0 ? +0.5 : 0.);
      bst(out, wr, row, F == 0 ? -0.5 : 0.);
      if (F != 0 && copy) {
        bst(out, wl, halo, 0.);
        bst(out, wr, halo, 0.);
      }
    }
  };
  // both rows' loads first: one wait instead of two
  Raw<F> r;
  double2 da, db;
  raw_load<F, P2, FOLD, 0>(a.tb, q, p, r);
  raw_load<F, P2, FOLD, 1>(a.tb, q, p, r);
  if constexpr (FOLD) {
    raw_fold<F, P2, 0, 0, 0>(a, q, p, ja, jb, write_a, edge, dt, r);
    raw_fold<F, P2, 0, 0, 1>(a, q, p, ja, jb, write_a, edge, dt, r);
  }
  raw_eval<F, P2, 0, IMY, 0>(a, q, r, p, write_a, edge, dt, da);
  raw_eval<F, P2, 0, IMY, 1>(a, q, r, p, write_a, edge, dt, db);
  if (write_a) emit(da, r.own_a(), ja, ja == 1, (unsigned)(g.jtot + 1) * pitch);
  emit(db, r.own_b(), jb, jb == g.jtot, 0u);
}

// Workgroup w: blocks (w % ncg)*waves .. of field (w / ncg) % nfld (+1 without
// the temperature equation), row pair w / ncg / nfld (as k_pred_rows).
template <bool P2, bool FOLD, int IMY, class S>
__global__ void __launch_bounds__(64 * kExpWaves, 3) k_pred_exp(S src, int nfld, int ncg) {
  const PredArgs a = src.get();
  const double dt = dt_of_step(a.dt, a.dtp, blockIdx.x == 0);
  const int w = xcd_groups(blockIdx.x, gridDim.x, kPredGroup * nfld * ncg);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = (w % ncg) * (blockDim.x >> 6) + wave;
  const int r = w / ncg;
  const int q = r / nfld, f = r % nfld + (nfld == 3 ? 0 : 1);
  if (b * kBlockCols >= a.g.itot) return;
  const int ja = min(2 * q + 1, a.g.jtot - 1), jb = ja + 1;
  const bool write_a = ja == 2 * q + 1;
  if (f == 0) pred_exp_body<0, P2, FOLD, IMY>(a, b, ja, jb, write_a, dt);
  else if (f == 1) pred_exp_body<1, P2, FOLD, IMY>(a, b, ja, jb, write_a, dt);
  else pred_exp_body<2, P2, FOLD, IMY>(a, b, ja, jb, write_a, dt);
}

// Power-of-two divisors select the variant that divides by multiplying, a psi
// argument the one that applies the previous substage's correction.
template <class S>
static void pred_exp_launch(hipStream_t s, const PredArgs &shape, S src, int nz) {
  const Geo &g = shape.g;
  const int nb = (g.itot + kBlockCols - 1) / kBlockCols;
  const int ncg = (nb + kExpWaves - 1) / kExpWaves, waves = (nb + ncg - 1) / ncg;
  const int nfld = shape.with_temp ? 3 : 2;
  const dim3 grid((g.jtot + 1) / 2 * nfld * ncg, 1, nz), block(64 * waves);
  const bool p2 = shape.tb.pow2, fold = shape.psi != nullptr;
  const bool imy = shape.tr.implicity;  // excludes fold
#define SNS_CALL(P2, FOLD, IMY) \
  hipLaunchKernelGGL((k_pred_exp<P2, FOLD, IMY, S>), grid, block, 0, s, src, nfld, ncg)
  if (p2 && fold) SNS_CALL(true, true, 0);
  else if (p2 && imy) SNS_CALL(true, false, 1);
  else if (p2) SNS_CALL(true, false, 0);
  else if (fold) SNS_CALL(false, true, 0);
  else if (imy) SNS_CALL(false, false, 1);
  else SNS_CALL(false, false, 0);
#undef SNS_CALL
}

void launch_pred(hipStream_t s, const PredArgs &a, int implicitx) {
  if (implicitx) launch_pred_rows(s, a);
  else pred_exp_launch(s, a, ArgOne<PredArgs>{a}, 1);
}

void launch_pred_batch(hipStream_t s, const PredArgs &shape, int implicitx, const PredArgs *dev,
                       int nz) {
  if (implicitx) launch_pred_rows_batch(s, shape, dev, nz);
  else pred_exp_launch(s, shape, arg_batch<PredArgs>(dev), nz);
}

// ------------------------------------------------- correction + pressure

// rows per workgroup of the correction kernel
constexpr int kCorrRows = 2;
// output columns per wave: lanes 1..62; lanes 0 and 63 hold the neighbours
constexpr int kCorrCols = 62;
constexpr int kCorrThreads = 256;

// src/fluid/correct_velocity.c:6-42 and src/fluid/update_pressure.c:7-60 in
// one pass: reads ux*, uy*, p and psi, writes ux, uy, p with boundary
// values.  psi(i-1) and psi(i+1) come from the adjacent lanes; psi of the
// rows above and below is carried in registers; the column metrics are read
// once per thread.  With red != nullptr it also folds the advective bound of
// src/param/decide_dt.c:25-45 over the corrected velocities: each workgroup
// stores the minimum over its cells in red[workgroup] and k_dt reduces them
// (min is exact, so the result does not depend on the order).
template <class S>
__global__ void __launch_bounds__(kCorrThreads) k_corr(S src) {
  const CorrArgs a = src.get();
  const Geo &g = a.g;
  const Tables &tb = a.tb;
  const int itot = g.itot;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = (blockIdx.x * (kCorrThreads / 64) + wave) * kCorrCols + lane;  // lane 0: i-1 halo
  const bool out = lane >= 1 && lane <= kCorrCols && i <= itot;
  const int ci = clampi(i, 0, itot + 1);
  const int ti = clampi(i - 1, 0, itot + 1);  // table entry of column i
  const int j0 = blockIdx.y * kCorrRows + 1;
  const double dt = *a.dtp;
  const double gdt = a.gamma * dt;
  const double fac = -gdt / g.two_Re;
  const size_t wc = (size_t)g.pc, wu = (size_t)g.pu;
  // column metrics; on a uniform grid a wave whose 64 columns all lie in
  // 2..itot-1 takes them as constants (the table entries themselves)
  const int c0 = i - lane;
  const bool interior = tb.uniform && c0 >= 2 && c0 + 63 <= itot - 1;
  double dxc_i, rdxc_i, dxc_p = 0., rdxc_p = 0., dxf_i = 0., rdxf_i = 0.;
  if (interior) {
    dxc_i = dxc_p = tb.u_dxc;
    rdxc_i = rdxc_p = tb.u_rdxc;
    dxf_i = tb.u_dxf;
    rdxf_i = tb.u_rdxf;
  } else {
    dxc_i = ldr(tb.dxc(), ti);  // DXC(i), 1./DXC(i)
    rdxc_i = ldr(tb.rdxc(), ti);
    if (a.tr.implicitx) {
      dxc_p = from_right(dxc_i);  // DXC(i+1)
      rdxc_p = from_right(rdxc_i);
      dxf_i = ldr(tb.dxf(), ti);
      rdxf_i = ldr(tb.rdxf(), ti);
    }
  }
  double m = 5.e-2;
  double psi_s = ldr(a.psi + (size_t)(j0 - 1) * wc, ci);  // psi(i, j-1)
  double psi_c = ldr(a.psi + (size_t)j0 * wc, ci);
#pragma unroll
  for (int r = 0; r < kCorrRows; r++) {
    const int j = j0 + r;
    if (j > g.jtot) break;
    const double psi_n = ldr(a.psi + (size_t)(j + 1) * wc, ci);  // psi(i, j+1)
    const double psi_w = from_left(psi_c);                        // psi(i-1, j)
    const double psi_e = from_right(psi_c);                       // psi(i+1, j)
    const double us = ldr(a.ux_star + (size_t)j * wu, clampi(i - 1, 0, itot));
    const double vs = ldr(a.uy_star + (size_t)j * wc, ci);
    const double pj = ldr(a.p + (size_t)j * wc, ci);
    if (out) {
      if (i >= 2) {
        const double v = proj_ux(us, psi_c, psi_w, gdt, rdxc_i);
        put_ux(g, a.ux, i, j, v);
        if (a.red) m = fmin(m, dxc_i / fmax(fabs(v), 1.e-8));
      }
      {
        const double v = proj_uy(vs, psi_c, psi_s, gdt, tb.dy, tb.rdy);
        put_c<0>(g, a.uy, i, j, v);
        if (a.red) m = fmin(m, tb.dy / fmax(fabs(v), 1.e-8));
      }
      const ProjX x = {dxc_i, rdxc_i, dxc_p, rdxc_p, dxf_i, rdxf_i};
      const double pv = proj_p(pj, psi_c, psi_w, psi_e, psi_s, psi_n, x, tb.dy, tb.rdy, fac,
                               a.tr.implicitx, a.tr.implicity);
      put_c<1>(g, a.p, i, j, pv);
    }
    psi_s = psi_c;
    psi_c = psi_n;
  }
  if (a.red) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fmin(m, __shfl_xor(m, off));
    __shared__ double wm[kCorrThreads / 64];
    if (lane == 0) wm[wave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
      double r = wm[0];
      for (int w = 1; w < kCorrThreads / 64; w++) r = fmin(r, wm[w]);
      a.red[blockIdx.y * gridDim.x + blockIdx.x] = r;
    }
  }
}

static dim3 corr_grid(const Geo &g) {
  const int cols = (kCorrThreads / 64) * kCorrCols;
  return dim3((g.itot + cols - 1) / cols, (g.jtot + kCorrRows - 1) / kCorrRows);
}

int corr_partials(const Geo &g) {
  const dim3 gr = corr_grid(g);
  return (int)(gr.x * gr.y);
}

void launch_corr(hipStream_t s, const CorrArgs &a) {
  hipLaunchKernelGGL(k_corr<ArgOne<CorrArgs>>, corr_grid(a.g), dim3(kCorrThreads), 0, s,
                     ArgOne<CorrArgs>{a});
}

static dim3 with_z(dim3 d, int nz) { return dim3(d.x, d.y, nz); }

void launch_corr_batch(hipStream_t s, const CorrArgs &shape, const CorrArgs *dev, int nz) {
  hipLaunchKernelGGL(k_corr<ArgBatch<CorrArgs>>, with_z(corr_grid(shape.g), nz),
                     dim3(kCorrThreads), 0, s, arg_batch<CorrArgs>(dev));
}

// The advective bound of src/param/decide_dt.c:25-45 over ux, uy as they
// are, with the tiling and the expressions of the reduction in k_corr: the
// minimum over the cells of workgroup w goes to red[w], so a time-step
// decision from these partials equals one from the partials the previous
// step's last correction stored.
template <class S>
__global__ void __launch_bounds__(kCorrThreads) k_adv_bound(S src) {
  const CorrArgs a = src.get();
  const Geo &g = a.g;
  const Tables &tb = a.tb;
  const int itot = g.itot;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = (blockIdx.x * (kCorrThreads / 64) + wave) * kCorrCols + lane;
  const bool out = lane >= 1 && lane <= kCorrCols && i <= itot;
  const int ci = clampi(i, 0, itot + 1);
  const int ti = clampi(i - 1, 0, itot + 1);
  const int j0 = blockIdx.y * kCorrRows + 1;
  const size_t wc = (size_t)g.pc, wu = (size_t)g.pu;
  const double dxc_i = ldr(tb.dxc(), ti);
  double m = 5.e-2;
#pragma unroll
  for (int r = 0; r < kCorrRows; r++) {
    const int j = j0 + r;
    if (j > g.jtot) break;
    const double u = ldr(a.ux + (size_t)j * wu, clampi(i - 1, 0, itot));
    const double v = ldr(a.uy + (size_t)j * wc, ci);
    if (out) {
      if (i >= 2) m = fmin(m, dxc_i / fmax(fabs(u), 1.e-8));
      m = fmin(m, tb.dy / fmax(fabs(v), 1.e-8));
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmin(m, __shfl_xor(m, off));
  __shared__ double wm[kCorrThreads / 64];
  if (lane == 0) wm[wave] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = wm[0];
    for (int w = 1; w < kCorrThreads / 64; w++) r = fmin(r, wm[w]);
    a.red[blockIdx.y * gridDim.x + blockIdx.x] = r;
  }
}

void launch_adv_bound(hipStream_t s, const CorrArgs &a) {
  hipLaunchKernelGGL(k_adv_bound<ArgOne<CorrArgs>>, corr_grid(a.g), dim3(kCorrThreads), 0, s,
                     ArgOne<CorrArgs>{a});
}

void launch_adv_bound_batch(hipStream_t s, const CorrArgs &shape, const CorrArgs *dev, int nz) {
  hipLaunchKernelGGL(k_adv_bound<ArgBatch<CorrArgs>>, with_z(corr_grid(shape.g), nz),
                     dim3(kCorrThreads), 0, s, arg_batch<CorrArgs>(dev));
}

// ------------------------------------------------ division self-check

__global__ void k_check_div(int n, const double *__restrict__ a, const double *__restrict__ b,
                            const double *__restrict__ r, double *__restrict__ q_cr,
                            double *__restrict__ q_ieee) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  q_cr[t] = div_cr(a[t], b[t], r[t]);
  q_ieee[t] = a[t] / b[t];
}

void launch_check_div(hipStream_t s, int n, const double *a, const double *b, const double *r,
                      double *q_cr, double *q_ieee) {
  hipLaunchKernelGGL(k_check_div, dim3((n + 255) / 256), dim3(256), 0, s, n, a, b, r, q_cr, q_ieee);
}

// ------------------------------------------------------------- time step

// src/param/decide_dt.c:45-97 on the device for a fixed treatment: the
// advective bound (minimum of the n partial minima in part) times 0.7, the
// diffusive bounds (fixed per run, computed on the host) and the treatment's
// dt; the run time advances by dt (src/main.c:34-35).  One workgroup of
// kDtThreads threads.
constexpr int kDtThreads = 1024;

template <class S>
__global__ void __launch_bounds__(kDtThreads) k_dt(S src) {
  const DtArgs a = src.get();
  const double *part = a.part;
  // eight independent loads in flight per thread (the minimum is exact, so
  // the grouping does not change it)
  constexpr int U = 8;
  double mu[U];
#pragma unroll
  for (int u = 0; u < U; u++) mu[u] = part[0];
  int k = threadIdx.x;
  for (; k + (U - 1) * kDtThreads < a.n; k += U * kDtThreads) {
    double v[U];
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = part[k + u * kDtThreads];
#pragma unroll
    for (int u = 0; u < U; u++) mu[u] = fmin(mu[u], v[u]);
  }
  for (; k < a.n; k += kDtThreads) mu[0] = fmin(mu[0], part[k]);
  double m = mu[0];
#pragma unroll
  for (int u = 1; u < U; u++) m = fmin(m, mu[u]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmin(m, __shfl_xor(m, off));
  __shared__ double wm[kDtThreads / 64];
  if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int w = 1; w < kDtThreads / 64; w++) m = fmin(m, wm[w]);
  m = fmin(m, wm[0]);
  const double d = dt_of(a, m);
  *a.dt = d;
  *a.time += d;
}

void launch_dt(hipStream_t s, const DtArgs &a) {
  hipLaunchKernelGGL(k_dt<ArgOne<DtArgs>>, dim3(1), dim3(kDtThreads), 0, s, ArgOne<DtArgs>{a});
}

void launch_dt_batch(hipStream_t s, const DtArgs *dev, int nz) {
  hipLaunchKernelGGL(k_dt<ArgBatch<DtArgs>>, dim3(1, 1, nz), dim3(kDtThreads), 0, s,
                     arg_batch<DtArgs>(dev));
}

}  // namespace sns
