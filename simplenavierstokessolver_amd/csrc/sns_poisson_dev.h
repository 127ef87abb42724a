// sns_poisson_dev.h -- what the y transforms of the Poisson solve share (gfx950):
// the right-hand side as the forward transforms read it, the spectra of column
// pairs, psi as the inverse ones store it, and their launch.
#pragma once
#include <atomic>
#include "sns_launch.h"
#include "sns_fast.h"
#include "sns_fft.h"
#include "sns_poisson.h"

namespace sns {

constexpr int kElems = 2048;  // complex values per workgroup and pass
constexpr int kMaxThreads = 512;
constexpr size_t kMaxLds = 160 * 1024;

// P2: every divisor a power of two (the quotients are products, see dv)
template <bool P2>
__device__ __forceinline__ double poisson_rhs2(const Geo &g, const Tables &tb, const double *ux,
                                               const double *uy, double inv_gdt, int i, int j) {
  // 1./(gamma*dt)*((ux_xp-ux_xm)/DXF(i) + (uy_yp-uy_ym)/dy)
  const double ax = dv<P2>(ux[ux_idx(g, i + 1, j)] - ux[ux_idx(g, i, j)], tb.dxf()[i - 1],
                           tb.rdxf()[i - 1]);
  const double ay = dv<P2>(uy[c_idx(g, i, j + 1)] - uy[c_idx(g, i, j)], tb.dy, tb.rdy);
  return inv_gdt * (+ax + ay);
}

__device__ __forceinline__ void put_psi(const Geo &g, double *f, int i, int j, double v) {
  // Neumann walls and periodic halo rows (src/fluid/boundary_conditions.c:39-55)
  f[c_idx(g, i, j)] = v;
  if (j == 1) f[c_idx(g, i, g.jtot + 1)] = v;
  if (j == g.jtot) f[c_idx(g, i, 0)] = v;
  if (i == 1 || i == g.itot) {
    const int iw = i == 1 ? 0 : g.itot + 1;
    f[c_idx(g, iw, j)] = v;
    if (j == 1) f[c_idx(g, iw, g.jtot + 1)] = v;
    if (j == g.jtot) f[c_idx(g, iw, 0)] = v;
  }
}

// RHS of the column pair (ia, ia+1), ia odd, at 0-based rows j.  AL: the
// padded state layout (ux rows and uy's column 1 on 16-byte boundaries, even
// pitches), in 16-byte loads: ux faces ia, ia+1 (one pair), ia+2; uy of rows
// j+1 and j+2 (one pair each).  Columns past itot give 0.
template <bool P2, bool AL>
struct RhsCol {
  const PoisArgs &a;
  double inv_gdt;
  int ia, ic;  // lanes past the last column read column 1
  double dxa, rdxa, dxb, rdxb;
  __device__ __forceinline__ RhsCol(const PoisArgs &args, double ig, int pair)
      : a(args), inv_gdt(ig), ia(2 * pair + 1) {
    const int itot = a.g.itot;
    ic = ia <= itot ? ia : 1;
    if constexpr (AL) {
      dxa = dxb = a.tb.u_dxf;
      rdxa = rdxb = a.tb.u_rdxf;
      if (!a.tb.uniform) {
        dxa = a.tb.dxf()[ic - 1];
        rdxa = a.tb.rdxf()[ic - 1];
        dxb = a.tb.dxf()[min(ic, itot - 1)];
        rdxb = a.tb.rdxf()[min(ic, itot - 1)];
      }
    }
  }
  __device__ __forceinline__ double2 operator()(int j) const {
    const Geo &g = a.g;
    const Tables &tb = a.tb;
    const int itot = g.itot;
    double2 z;
    if constexpr (AL) {
      const double *urow = a.ux + (size_t)((j + 1) * g.pu);
      const double2 u01 = ldr2(reinterpret_cast<const double2 *>(urow + ic - 1), 0);
      const double u2 = ldr(urow, min(ic + 1, itot));  // face ic+2 (used when ic+1 <= itot)
      const double *vrow = a.uy + (size_t)((j + 1) * g.pc);
      const double2 v0 = ldr2(reinterpret_cast<const double2 *>(vrow + ic), 0);
      const double2 v1 = ldr2(reinterpret_cast<const double2 *>(vrow + g.pc + ic), 0);
      // the expressions of poisson_rhs2, column by column
      const double axa = dv<P2>(u01.y - u01.x, dxa, rdxa);
      const double aya = dv<P2>(v1.x - v0.x, tb.dy, tb.rdy);
      const double axb = dv<P2>(u2 - u01.y, dxb, rdxb);
      const double ayb = dv<P2>(v1.y - v0.y, tb.dy, tb.rdy);
      z.x = ia <= itot ? inv_gdt * (+axa + aya) : 0.;
      z.y = ia + 1 <= itot ? inv_gdt * (+axb + ayb) : 0.;
    } else {
      z.x = ia <= itot ? poisson_rhs2<P2>(g, tb, a.ux, a.uy, inv_gdt, ia, j + 1) : 0.;
      z.y = ia + 1 <= itot ? poisson_rhs2<P2>(g, tb, a.ux, a.uy, inv_gdt, ia + 1, j + 1) : 0.;
    }
    return z;
  }
};

// Spectra of the two real columns of a pair from the packed one:
// X_a = (Z_k + conj Z_{n-k})/2, X_b = (Z_k - conj Z_{n-k})/(2i).
__device__ __forceinline__ void put_spectra(const PoisArgs &a, int k, int pair, double2 zk,
                                            double2 zn) {
  const int ia = 2 * pair + 1;
  double2 xa, xb;
  xa.x = 0.5 * (zk.x + zn.x);
  xa.y = 0.5 * (zk.y - zn.y);
  xb.x = 0.5 * (zk.y + zn.y);
  xb.y = 0.5 * (zn.x - zk.x);
  double2 *row = a.psihat + (size_t)k * a.g.itot;
  if (ia <= a.g.itot) row[ia - 1] = xa;
  if (ia + 1 <= a.g.itot) row[ia] = xb;
}

// ... and the packed spectrum from the two columns' (wavenumber k <= n/2):
// Z_k = X_a + i X_b, zn = Z_{n-k} = conj X_a + i conj X_b
// (src/fluid/compute_potential.c:147-149: c2r input).
__device__ __forceinline__ double2 get_spectra(const PoisArgs &a, int k, int pair, double2 &zn) {
  const int ia = 2 * pair + 1;
  const double2 *row = a.psihat + (size_t)k * a.g.itot;
  double2 xa = make_double2(0., 0.), xb = make_double2(0., 0.);
  if (ia <= a.g.itot) xa = row[ia - 1];
  if (ia + 1 <= a.g.itot) xb = row[ia];
  if (k == 0 || 2 * k == a.pl.n) { xa.y = 0.; xb.y = 0.; }
  zn = make_double2(xa.x + xb.y, -xa.y + xb.x);
  return make_double2(xa.x - xb.y, xa.y + xb.x);
}

// the side of a transform that goes through LDS
struct NoIo {
  __device__ __forceinline__ NoIo operator()(int) const { return *this; }
  __device__ __forceinline__ void operator()(int, double2) const {}
};

// psi = q/jtot at 0-based rows j of a column pair with boundary values: the
// exact division of div_cr, or (jtot a power of two) the product with the
// exact reciprocal; both equal IEEE q/jtot bit for bit.
template <bool AL>
struct PsiCol {
  const PoisArgs &a;
  double njtot, rnj;
  int ia;
  bool jp2, wall;
  __device__ __forceinline__ PsiCol(const PoisArgs &args, int pair)
      : a(args), njtot(1. * args.g.jtot), rnj(1. / njtot), ia(2 * pair + 1),
        jp2((args.g.jtot & (args.g.jtot - 1)) == 0),
        wall(!AL || ia == 1 || ia + 1 >= args.g.itot) {}
  __device__ __forceinline__ void operator()(int j0, double2 z) const {
    const Geo &g = a.g;
    const int j = j0 + 1;
    const double va = jp2 ? z.x * rnj : div_cr(z.x, njtot, rnj);
    const double vb = jp2 ? z.y * rnj : div_cr(z.y, njtot, rnj);
    if (!(wall || j == 1 || j == g.jtot)) {
      // both columns in one 16-byte store (no halo or wall copies here)
      *reinterpret_cast<double2 *>(a.psi + (unsigned)(j * g.pc + ia)) = make_double2(va, vb);
    } else {
      if (ia <= g.itot) put_psi(g, a.psi, ia, j, va);
      if (ia + 1 <= g.itot) put_psi(g, a.psi, ia + 1, j, vb);
    }
  }
};

inline size_t fft_lds_bytes(int S, int L) { return (fft_slots(S * L) + L) * sizeof(double2); }
inline int fft_threads(int S, const FftSched &sc) { return (S * sc.L / sc.rmin + 63) / 64 * 64; }

// Kernel k_<name>: <name> with the schedule type Sc and the template arguments
// `args`.  128 registers, 16 waves per CU.
#define SNS_FFT_KERNEL(name, params, args)                                         \
  template <class Sc, params class S>                                              \
  __global__ void __launch_bounds__(kMaxThreads, 4) k_##name(S src) {              \
    name<Sc args>(src.get());                                                      \
  }
#define SNS_C ,

// Launch kernel K for the transform sc of S_ sequences a workgroup
#define SNS_FFT_LAUNCH(K, S_, sc, grid)                                                     \
  do {                                                                                      \
    static std::atomic<unsigned> attr{0};                                                   \
    const size_t lds = fft_lds_bytes(S_, (sc).L);                                           \
    lds_limit_once((const void *)(K), kMaxLds, attr);                                       \
    hipLaunchKernelGGL((K), dim3((grid).x, (grid).y, nz), dim3(fft_threads(S_, sc)), lds, s, src);      \
  } while (0)

// The one-kernel transforms (sns_poisson_one.hip): the schedule of length n
// (false: none), and the launches.
bool one_pass_sched(int n, FftSched &sc);
template <class S>
void one_pass_forward(hipStream_t s, const Fft2Plan &pl, bool aligned, S src, int nz);
template <class S>
void one_pass_inverse(hipStream_t s, const Fft2Plan &pl, bool aligned, S src, int nz);

}  // namespace sns
