// sns_poisson.hip -- the pressure-potential Poisson solve (gfx950).
//
// Reference: src/fluid/compute_potential.c:15-168: RHS = div(u*)/(gamma dt),
// real FFT along y (FFTW r2c, unnormalised), one tri-diagonal system along x
// per wavenumber, inverse c2r FFT, psi = result / jtot with Neumann walls.
//
// Up to 1024 rows the y transforms take one kernel each (sns_poisson_one.hip).
// Above, they run as four-step FFTs, n = n1*n2, j = n2*j1 + j2, k = k1 + n1*k2:
//   forward  pass A : Y[k1*n2+j2] = W_n^(j2 k1) * DFT_n1 over j1 of x[n2 j1 + j2]
//            pass B : X[k1 + n1 k2] = DFT_n2 over j2 of Y[k1*n2+j2]
//   inverse  pass B': Y[k1*n2+j2] = W_n^(-j2 k1) * IDFT_n2 over k2 of Z[k1 + n1 k2]
//            pass A': x[n2 j1 + j2] = IDFT_n1 over k1 of Y[k1*n2+j2]
// Every pass works on a tile of 16 real columns (8 complex pairs = 128-byte
// row segments), so all global accesses are whole cache lines; two real
// columns are packed as one complex sequence, and the spectra of the pair are
// separated (forward) or combined (inverse) in pass B / B', which therefore
// handles the wavenumber rows k1 and n1-k1 together.
//
// The passes move 3, 2, 2 and 2 words per cell; from 4096x8192 (4.1, 5.0, 4.4
// and 4.6 TB/s) they are bound by memory, whose rate the short strided runs
// keep under that of a copy; smaller grids by a workgroup's chain of latencies.
// us of the four passes with every stage through LDS, and with the first and
// last stage in registers and Y in one run per tile: 1537x3000 130 and 109,
// 1024x2048 50 and 44, 2048x4096 138 and 133, 4096x8192 571 and 543.
#include <float.h>
#include "sns_launch.h"
#include "sns_fast.h"
#include "sns_poisson_dev.h"
#include "sns_lu.h"

namespace sns {

// Intermediate of the two passes: one tile of column pairs after the other, so
// that a workgroup of either pass stays within one run of n*128 bytes.  (Runs
// that start off a multiple of 256 bytes cost a quarter more at 4096x8192.)
__device__ __forceinline__ unsigned y_idx(const Fft2Plan &pl, int k1, int j2, int pair) {
  const int t = pair >> pl.lgt, q = pair - (t << pl.lgt);
  return (((unsigned)(t * pl.n1 + k1) * pl.n2 + j2) << pl.lgt) + q;
}

// ------------------------------------------------------------ forward A

template <class Sc, bool P2, bool AL>
__device__ __forceinline__ void pfwd_a(const PoisArgs &a) {
  extern __shared__ double2 lds_fft[];
  const Fft2Plan &pl = a.pl;
  const FftSched &sc = Sc::get(pl.s1);
  // consecutive tiles of one row group on the same XCD: a tile's last ux
  // face is the first of the next tile's 128-byte line, which then stays in
  // that XCD's L2
  const int nb = gridDim.x * gridDim.y;
  const int w = xcd_remap(blockIdx.y * gridDim.x + blockIdx.x, nb);
  const int tile = w % gridDim.x, j20 = (w / gridDim.x) * pl.G;
  const int lt = pl.lgt, n2 = pl.n2;
  const double inv_gdt = 1. / (a.gamma * (*a.dtp));
  const FftLds l = fft_lds(lds_fft, sc, pl.G << lt, a.tw, pl.n);
  const int pair0 = tile << lt, qm = (1 << lt) - 1;
  fft_run<Sc, -1, true, true, AL>(
      l, sc,
      [&](int s) {
        const RhsCol<P2, AL> rhs(a, inv_gdt, pair0 + (s & qm));
        const int j2 = j20 + (s >> lt);
        return [=](int j1) { return rhs(n2 * j1 + j2); };
      },
      [&](int s) {
        const int j2 = j20 + (s >> lt), pair = pair0 + (s & qm);
        return [=, &a](int k1, double2 z) {
          if (pair >= a.pl.npair) return;
          if (k1 && j2) z = cmul(z, a.tw[j2 * k1]);
          a.Y[y_idx(a.pl, k1, j2, pair)] = z;
        };
      });
}

// ------------------------------------------------------------ forward B

// The wavenumber rows k1a and k1b = n1-k1a of one tile: sequences (h << lgt) + q.
struct PassB {
  int pair0, k1a, k1b, nh, S;
  int lt, qm;
  int c0, cn;  // wavenumbers k <= n/2 of row k1a, of both
  // the i-th of them: wavenumber and element
  __device__ __forceinline__ int k_of(int n1, int i, int &k2, int &h) const {
    h = i >= c0;
    k2 = h ? i - c0 : i;
    return (h ? k1b : k1a) + n1 * k2;
  }
  // element and sequence half of the mirror n-k of k = k1 + n1*k2
  __device__ __forceinline__ void mirror(int n2, int k2, int h, int &k2p, int &hp) const {
    if ((h ? k1b : k1a) == 0) {
      k2p = k2 ? n2 - k2 : 0;
      hp = h;
    } else {
      k2p = n2 - 1 - k2;
      hp = nh == 1 ? h : 1 - h;
    }
  }
};
__device__ __forceinline__ PassB pass_b(const Fft2Plan &pl) {
  PassB b;
  b.lt = pl.lgt;
  b.qm = (1 << pl.lgt) - 1;
  b.pair0 = blockIdx.x << pl.lgt;
  b.k1a = blockIdx.y;
  b.k1b = b.k1a ? pl.n1 - b.k1a : 0;
  b.nh = b.k1a == b.k1b ? 1 : 2;
  b.S = b.nh << pl.lgt;
  b.c0 = (pl.n / 2 - b.k1a) / pl.n1 + 1;
  b.cn = b.c0 + (b.nh == 2 ? (pl.n / 2 - b.k1b) / pl.n1 + 1 : 0);
  return b;
}

template <class Sc>
__device__ __forceinline__ void pfwd_b(const PoisArgs &a) {
  extern __shared__ double2 lds_fft[];
  const Fft2Plan &pl = a.pl;
  const FftSched &sc = Sc::get(pl.s2);
  const PassB B = pass_b(pl);
  const int n1 = pl.n1, n2 = pl.n2, n = pl.n;
  const FftLds l = fft_lds(lds_fft, sc, B.S, a.tw, n);
  fft_run<Sc, -1, true, false>(
      l, sc,
      [&](int s) {
        const int pair = min(B.pair0 + (s & B.qm), pl.npair - 1);
        const int k1 = s >> B.lt ? B.k1b : B.k1a;
        return [=, &a](int j2) { return a.Y[y_idx(a.pl, k1, j2, pair)]; };
      },
      NoIo{});
#pragma unroll 4
  for (int e = threadIdx.x; e < B.cn << B.lt; e += blockDim.x) {
    const int q = e & B.qm;
    int k2, h, k2p, hp;
    const int k = B.k_of(n1, e >> B.lt, k2, h);
    B.mirror(n2, k2, h, k2p, hp);
    put_spectra(a, k, B.pair0 + q, l.buf[fft_pad(k2 * B.S + (h << B.lt) + q)],
                l.buf[fft_pad(k2p * B.S + (hp << B.lt) + q)]);
  }
}

// ------------------------------------------------------------ inverse B'

// Each stored wavenumber m <= n/2 is read once and fills the slots of k = m
// and of its mirror n-m, which this workgroup holds too.
template <class Sc>
__device__ __forceinline__ void pinv_b(const PoisArgs &a) {
  extern __shared__ double2 lds_fft[];
  const Fft2Plan &pl = a.pl;
  const FftSched &sc = Sc::get(pl.s2);
  const PassB B = pass_b(pl);
  const int n1 = pl.n1, n2 = pl.n2, n = pl.n;
  const FftLds l = fft_lds(lds_fft, sc, B.S, a.tw, n);
#pragma unroll 4
  for (int e = threadIdx.x; e < B.cn << B.lt; e += blockDim.x) {
    const int q = e & B.qm;
    int k2, h;
    const int k = B.k_of(n1, e >> B.lt, k2, h);
    double2 zn;
    l.buf[fft_pad(k2 * B.S + (h << B.lt) + q)] = get_spectra(a, k, B.pair0 + q, zn);
    if (k != 0 && 2 * k != n) {
      int k2p, hp;
      B.mirror(n2, k2, h, k2p, hp);
      l.buf[fft_pad(k2p * B.S + (hp << B.lt) + q)] = zn;
    }
  }
  __syncthreads();
  fft_run<Sc, +1, false, true>(l, sc, NoIo{}, [&](int s) {
    const int pair = B.pair0 + (s & B.qm);
    const int k1 = s >> B.lt ? B.k1b : B.k1a;
    return [=, &a](int j2, double2 z) {
      if (pair >= a.pl.npair) return;
      if (k1 && j2) z = cmul(z, cdir<+1>(a.tw[j2 * k1]));
      a.Y[y_idx(a.pl, k1, j2, pair)] = z;
    };
  });
}

// ------------------------------------------------------------ inverse A'

template <class Sc, bool AL>
__device__ __forceinline__ void pinv_a(const PoisArgs &a) {
  extern __shared__ double2 lds_fft[];
  const Fft2Plan &pl = a.pl;
  const FftSched &sc = Sc::get(pl.s1);
  const int lt = pl.lgt, n2 = pl.n2, j20 = blockIdx.y * pl.G;
  const FftLds l = fft_lds(lds_fft, sc, pl.G << lt, a.tw, pl.n);
  const int pair0 = blockIdx.x << lt, qm = (1 << lt) - 1;
  fft_run<Sc, +1, true, true>(
      l, sc,
      [&](int s) {
        const int pair = min(pair0 + (s & qm), pl.npair - 1), j2 = j20 + (s >> lt);
        return [=, &a](int k1) { return a.Y[y_idx(a.pl, k1, j2, pair)]; };
      },
      [&](int s) {
        const PsiCol<AL> psi(a, pair0 + (s & qm));
        const int j2 = j20 + (s >> lt);
        return [=](int j1, double2 z) { psi(n2 * j1 + j2, z); };
      });
}

// --------------------------------------------------- x solve per wavenumber

// Matrix of wavenumber J (src/fluid/compute_potential.c:117-127): l_i =
// 1/(DXC(i)DXF(i)), u_i = 1/(DXC(i+1)DXF(i)), c_i = -l_i - u_i + lambda_J with
// the Neumann walls folded into c_0 and c_{n-1}.  It does not change during
// a run, so its Thomas factorisation (src/linalg.c:32-50: u'_i and the
// reciprocal pivots, in the reference's sequential order) is computed once
// per instance by k_poisson_factor, one thread per wavenumber.  Only the
// reciprocal pivots r_i depend on J; the substitutions need al_i = -(r_i l_i)
// and be_i = -u'_i = -(r_i u_i) for 0 < i < n-1, so the factor table holds r
// (interleaved as in sns_lu.h, ntm entries per J) followed by u'_0 = u_0/c_0
// of every J, then per J the last row pfx <= n-2 whose pivot differs from
// the previous row's and that pivot (rows pfx..n-2 share it: on a grid with
// identical interior rows the recurrence reaches a fixed point, bit for bit,
// after a few rows for all but the lowest J); l, u are shared interleaved
// tables (LuTabLUr reads only rows up to pfx and the last row).
// The J = 0 system is singular; its last equation is replaced by
// psi_hat(itot) = 0 (r = 0 on that row).  Each solve then needs only the two
// substitutions, evaluated by lu_solve_shared for the real and imaginary
// parts together; with the factors exact, the substitutions keep the
// accuracy of the sequential sweep on the nearly singular low-J systems.
__device__ __forceinline__ int lu_slot(int i, int NT, int M) { return (i % M) * NT + i / M; }

__global__ void __launch_bounds__(64)
    k_poisson_factor(Geo g, Tables tb, const double *__restrict__ eigen, int NT, int M, int ntm,
                     double *__restrict__ fac) {
  const int J = blockIdx.x * blockDim.x + threadIdx.x;
  const int nJ = g.jtot / 2 + 1;
  if (J >= nJ) return;
  const int n = g.itot;
  const double lam = eigen[J];
  double *R = fac + (size_t)J * ntm;
  auto coef = [&](int i, double &l, double &c, double &u) {
    l = tb.pl()[i];
    u = tb.pu()[i];
    c = -l - u + lam;
    if (i == 0) c += l;
    if (i == n - 1) c += u;
  };
  double l, c, u;
  coef(0, l, c, u);
  double up = u / c;  // u'_0
  double r = 1. / c;
  R[lu_slot(0, NT, M)] = r;
  fac[(size_t)nJ * ntm + J] = up;
  int pfx = 0;
  double rpfx = r;
  for (int i = 1; i < n; i++) {
    coef(i, l, c, u);
    const double val = c - l * up;
    const double rp = r;
    if (fabs(val) < DBL_EPSILON || (J == 0 && i == n - 1)) {
      up = 0.;
      r = 0.;
    } else {
      r = 1. / val;
      up = r * u;
    }
    R[lu_slot(i, NT, M)] = r;
    if (i <= n - 2 && __double_as_longlong(r) != __double_as_longlong(rp)) {
      pfx = i;
      rpfx = r;
    }
  }
  fac[(size_t)nJ * ntm + nJ + J] = (double)pfx;
  fac[(size_t)nJ * ntm + 2 * nJ + J] = rpfx;
}

template <int NT, int M>
struct PxLds {
  double2 row[NT * (M + 1)];
  double scr[4 * 2 * (NT / 64)];
};

// One workgroup per wavenumber row; the row is staged through LDS (coalesced
// global access, chunk order for the substitutions).
template <int NT, int M>
__device__ __forceinline__ void poisson_x3(const Geo &g, const Tables &tb,
                                           const double *__restrict__ fac,
                                           const double *__restrict__ plu, int ntm,
                                           double2 *__restrict__ psihat) {
  extern __shared__ double lds_raw[];
  PxLds<NT, M> &L = *reinterpret_cast<PxLds<NT, M> *>(lds_raw);
  const int J = xcd_remap(blockIdx.x, gridDim.x);
  const int n = g.itot;
  double2 *row = psihat + (size_t)J * n;
  for (int r = threadIdx.x; r < n; r += NT) L.row[r + r / M] = row[r];
  __syncthreads();
  double d[2][M];
#pragma unroll
  for (int k = 0; k < M; k++) {
    const int r = threadIdx.x * M + k;
    const double2 v = r < n ? L.row[r + r / M] : make_double2(0., 0.);
    d[0][k] = v.x;
    d[1][k] = v.y;
  }
  const int nJ = g.jtot / 2 + 1;
  const double *tail = fac + (size_t)nJ * ntm;
  const LuTabLUr<M> tab(fac + (size_t)J * ntm, plu, plu + ntm, n, tail[J], (int)tail[nJ + J],
                        tail[2 * nJ + J], NT, tb.plu_const != 0, tb.plc, tb.puc);
  lu_solve_shared<NT, M, 2>(d, tab, L.scr);
#pragma unroll
  for (int k = 0; k < M; k++) {
    const int r = threadIdx.x * M + k;
    if (r < n) L.row[r + r / M] = make_double2(d[0][k], d[1][k]);
  }
  __syncthreads();
  for (int r = threadIdx.x; r < n; r += NT) row[r] = L.row[r + r / M];
}

// ---------------------------------------------------------------- kernels
// Argument source S: ArgOne<PoisArgs> (one instance) or ArgBatch<PoisArgs>
// (instance blockIdx.z of a batch).

// Forward: AL on the padded state layout (pair loads), P2 with power-of-two
// divisors; inverse: AL on the padded state layout (psi's column 1 on a
// 16-byte boundary).
SNS_FFT_KERNEL(pfwd_a, bool P2 SNS_C bool AL SNS_C, SNS_C P2 SNS_C AL)
SNS_FFT_KERNEL(pfwd_b, , )
SNS_FFT_KERNEL(pinv_b, , )
SNS_FFT_KERNEL(pinv_a, bool AL SNS_C, SNS_C AL)

template <int NT, int M, class S>
__global__ void __launch_bounds__(NT) k_poisson_x3(S src) {
  const PoisArgs a = src.get();
  poisson_x3<NT, M>(a.g, a.tb, a.fac, a.plu, NT * M, a.psihat);
}

// Threads NT and unknowns per thread M of the x solve for n = itot unknowns
// (NT*M >= n).  One workgroup solves one wavenumber row, so with only
// jtot/2+1 rows the narrower grids take 4 unknowns per thread (twice the
// waves per row) and the wider ones 8.
static void px_shape(int n, int &NT, int &M) {
  M = n <= 1024 ? 4 : 8;
  NT = 64;
  while (NT < 1024 && NT * M < n) NT *= 2;
}

int poisson_factor_entries(int itot) {
  int NT, M;
  px_shape(itot, NT, M);
  return NT * M;
}

size_t poisson_factor_doubles(int itot, int jtot) {
  return (size_t)(jtot / 2 + 1) * (poisson_factor_entries(itot) + 3);
}

void poisson_lu_coefs(int itot, const double *pl, const double *pu, double *plu) {
  int NT, M;
  px_shape(itot, NT, M);
  const int ntm = NT * M;
  for (int k = 0; k < 2 * ntm; k++) plu[k] = 0.;
  for (int i = 0; i < itot; i++) {
    const int slot = (i % M) * NT + i / M;
    plu[slot] = pl[i];
    plu[ntm + slot] = pu[i];
  }
}

void launch_poisson_factor(hipStream_t s, const Geo &g, const Tables &tb, const double *eigen,
                           double *fac) {
  int NT, M;
  px_shape(g.itot, NT, M);
  const int ntm = NT * M;
  const int nJ = g.jtot / 2 + 1;
  hipLaunchKernelGGL(k_poisson_factor, dim3((nJ + 63) / 64), dim3(64), 0, s, g, tb, eigen, NT,
                     M, ntm, fac);
}

template <int NT, int M, class S>
static void px_launch(hipStream_t s, const Geo &g, S src, int nz) {
  const size_t lds = sizeof(PxLds<NT, M>);
  static std::atomic<unsigned> attr{0};
  lds_limit_once((const void *)k_poisson_x3<NT, M, S>, lds, attr);
  hipLaunchKernelGGL((k_poisson_x3<NT, M, S>), dim3(g.jtot / 2 + 1, 1, nz), dim3(NT), lds, s, src);
}

// ------------------------------------------------------------- plan, launch

// Column pairs per workgroup (as its binary logarithm) of the one-kernel
// transforms, -1 where the two-pass ones are taken.  Up to 1024 rows one kernel
// is the faster at every width, with more pairs where there are workgroups to
// spare (longer runs of memory).  us per step, two passes and one: 32x64 72 and
// 55, 128x192 85 and 64, 225x360 122 and 112, 512x1024 210 and 196, 700x1000 244
// and 230, 2048x512 263 and 240 (4 pairs; 244 and 262 with 2 and 1), 4096x1024
// 755 and 720.  With 2048 rows the two are about equal up to 1024 columns, and
// at 2048x2048 one takes 790 where two take 727.
static int one_pass_pairs(int n, int itot) {
  if (n > 1024) return -1;
  return itot >= 1024 ? 2 : itot >= 256 ? 1 : 0;
}

// Powers of two have their schedules compiled in on either layout, other factors
// read theirs (registers of the largest radix, a switch per stage: 512x1024 30 us
// that way, 24 compiled in; passes A and A' on the packed layout, 512x2048 13.3
// and 6.7 read, 12.4 and 6.3 compiled in).
using Any = AnySched<16, 3>;

// the two passes' factors
static bool pass_sched(int m, FftSched &sc) { return fft_sched(m, sc, Any::rmax, Any::npmax); }

bool fft2_plan(int n, int itot, Fft2Plan &pl, int n1) {
  if (n < 4) return false;
  // n1 = the given factor, else the largest divisor of n not above sqrt(n)
  // that the radices cover
  FftSched s1, s2;
  int best = -1;
  if (n1 > 0) {
    if (n % n1 || n1 < 2 || n / n1 < 2 || !pass_sched(n1, s1) || !pass_sched(n / n1, s2))
      return false;
    best = n1;
  } else {
    for (int d = 2; d * d <= n; d++)
      if (n % d == 0 && pass_sched(d, s1) && pass_sched(n / d, s2)) best = d;
  }
  if (best < 2) return false;
  pl = Fft2Plan{};
  pl.n = n;
  pl.n1 = best;
  pl.n2 = n / best;
  pl.npair = (itot + 1) / 2;
  if (pl.n1 > 256 || pl.n2 > 128) return false;  // the workgroups' LDS
  int lgt = n1 > 0 ? -1 : one_pass_pairs(n, itot);
  if (lgt >= 0 && one_pass_sched(n, pl.s1))
    while (lgt >= 0 && (fft_threads(1 << lgt, pl.s1) > kMaxThreads ||
                        fft_lds_bytes(1 << lgt, n) > kMaxLds))
      lgt--;
  else lgt = -1;
  if (lgt >= 0) {
    pl.one = true;
    pl.lgt = lgt;
    return true;
  }
  pass_sched(pl.n1, pl.s1);
  pass_sched(pl.n2, pl.s2);
  // 8 pairs, 128-byte runs: 16 measured the same (564 and 579 us for the four
  // passes of 4096x8192, 145 both at 2048x4096), 4 slower (707 and 158)
  pl.lgt = 3;
  while (fft_threads(1 << pl.lgt, pl.s1) > kMaxThreads ||
         fft_threads(2 << pl.lgt, pl.s2) > kMaxThreads)
    pl.lgt--;
  const int T = 1 << pl.lgt;
  pl.G = 1;
  for (int c = 2; c <= pl.n2; c++)
    if (pl.n2 % c == 0 && c * T * pl.n1 <= kElems && fft_threads(c * T, pl.s1) <= kMaxThreads)
      pl.G = c;
  return true;
}

static dim3 with_z(dim3 d, int nz) { return dim3(d.x, d.y, nz); }

// f(schedule type) for the fixed schedules, else Any.
template <class F>
static void two_pass_sched(const FftSched &sc, F f) {
  if (FixedSched<4, 8>::is(sc)) f(FixedSched<4, 8>{});
  else if (FixedSched<8, 8>::is(sc)) f(FixedSched<8, 8>{});
  else if (FixedSched<8, 16>::is(sc)) f(FixedSched<8, 16>{});
  else f(Any{});
}

// ... of pass B', with the stages its threads are counted by.  Its first stage
// reads LDS, so two stages save it nothing, and a last one of radix 16 leaves
// half of the threads without a butterfly while the others store 16 values each:
// 4096x8192 147 us with radices 8, 16, 136 with 16, 8, 130 with 8, 4, 4; 8, 8 and
// 4, 4, 4: 4096x4096 48.7 and 45.4, 2048x4096 26.4 and 23.6, 512x2048 8.4 and 7.2.
// (More threads beside two stages: 160 us at 4096x8192.)
template <class F>
static void pass_b_inverse_sched(const FftSched &sc, F f) {
  if (FixedSched<8, 8>::is(sc)) f(FixedSched<4, 4, 4>{}, FixedSched<4, 4, 4>::make());
  else if (FixedSched<8, 16>::is(sc)) f(FixedSched<8, 4, 4>{}, FixedSched<8, 4, 4>::make());
  else if (FixedSched<4, 8>::is(sc)) f(FixedSched<4, 8>{}, sc);
  else f(Any{}, sc);
}

template <class S>
static void poisson_forward(hipStream_t s, const Fft2Plan &pl, bool pow2, bool aligned, S src,
                            int nz) {
  if (pl.one) return one_pass_forward(s, pl, aligned, src, nz);
  const int T = 1 << pl.lgt, nt = (pl.npair + T - 1) / T;
  const dim3 ga(nt, pl.n2 / pl.G), gb(nt, pl.n1 / 2 + 1);
  two_pass_sched(pl.s1, [&](auto sc) {
    if (!aligned) SNS_FFT_LAUNCH((k_pfwd_a<decltype(sc), false, false, S>), pl.G * T, pl.s1, ga);
    else if (pow2) SNS_FFT_LAUNCH((k_pfwd_a<decltype(sc), true, true, S>), pl.G * T, pl.s1, ga);
    else SNS_FFT_LAUNCH((k_pfwd_a<decltype(sc), false, true, S>), pl.G * T, pl.s1, ga);
  });
  two_pass_sched(pl.s2, [&](auto sc) {
    SNS_FFT_LAUNCH((k_pfwd_b<decltype(sc), S>), 2 * T, pl.s2, gb);
  });
}

template <class S>
static void poisson_inverse(hipStream_t s, const Fft2Plan &pl, bool aligned, S src, int nz) {
  if (pl.one) return one_pass_inverse(s, pl, aligned, src, nz);
  const int T = 1 << pl.lgt, nt = (pl.npair + T - 1) / T;
  const dim3 ga(nt, pl.n2 / pl.G), gb(nt, pl.n1 / 2 + 1);
  pass_b_inverse_sched(pl.s2, [&](auto sc, const FftSched &st) {
    SNS_FFT_LAUNCH((k_pinv_b<decltype(sc), S>), 2 * T, st, gb);
  });
  two_pass_sched(pl.s1, [&](auto sc) {
    if (!aligned) SNS_FFT_LAUNCH((k_pinv_a<decltype(sc), false, S>), pl.G * T, pl.s1, ga);
    else SNS_FFT_LAUNCH((k_pinv_a<decltype(sc), true, S>), pl.G * T, pl.s1, ga);
  });
}

template <class S>
static void poisson_stage(hipStream_t s, const Geo &g, const Fft2Plan &pl, bool pow2,
                          bool aligned, S src, int nz, int stage) {
  if (stage == 0 || stage < 0) poisson_forward(s, pl, pow2, aligned, src, nz);
  if (stage == 1 || stage < 0) {
    int NT, M;
    px_shape(g.itot, NT, M);
    if (M == 4) {
      switch (NT) {
        case 64: px_launch<64, 4>(s, g, src, nz); break;
        case 128: px_launch<128, 4>(s, g, src, nz); break;
        default: px_launch<256, 4>(s, g, src, nz); break;
      }
    } else {
      switch (NT) {
        case 256: px_launch<256, 8>(s, g, src, nz); break;
        case 512: px_launch<512, 8>(s, g, src, nz); break;
        default: px_launch<1024, 8>(s, g, src, nz); break;
      }
    }
  }
  if (stage == 2 || stage < 0) poisson_inverse(s, pl, aligned, src, nz);
}

// The padded state layout: even row pitches, ux rows and the column 1 of uy
// and psi on 16-byte boundaries (every instance of a batch is allocated
// alike).
static bool pair_layout(const PoisArgs &a) {
  auto al16 = [](const void *p) { return ((uintptr_t)p & 15u) == 0; };
  return a.g.pu % 2 == 0 && a.g.pc % 2 == 0 && al16(a.ux) && al16(a.uy + 1) && al16(a.psi + 1);
}

void launch_poisson(hipStream_t s, const PoisArgs &a, int stage) {
  poisson_stage(s, a.g, a.pl, a.tb.pow2, pair_layout(a), ArgOne<PoisArgs>{a}, 1, stage);
}

void launch_poisson_batch(hipStream_t s, const PoisArgs &shape, const PoisArgs *dev, int nz,
                          int stage) {
  poisson_stage(s, shape.g, shape.pl, shape.tb.pow2, pair_layout(shape),
                arg_batch<PoisArgs>(dev), nz, stage);
}

}  // namespace sns
