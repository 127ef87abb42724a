// sns_fft.h -- batched complex FFT of short lengths, exchanged through LDS (gfx950).
//
// Stockham auto-sort stages (no bit reversal): the stage with radix R and
// running sub-transform length Ns reads x_r = buf[j + r*L/R], applies the
// twiddles w^(r*k), k = j mod Ns, w = exp(sign*2*pi*i/(Ns*R)), performs an
// R-point DFT and writes buf[(j-k)*R + k + r*Ns].  One butterfly per thread and
// stage.  The first stage may take its inputs in registers and the last one
// leave its outputs there: two stages between global memory and global memory
// (passes A and A' of the two-pass transforms, lengths with two factors up to 16)
// cost one LDS exchange and one barrier where staging each in LDS cost four and
// six.  Every further stage is an exchange more, with two barriers: three stages
// where a length has no two such factors, three or four in the transforms of
// whole columns, whose radices are kept small; and the side of a transform where
// spectra are separated or combined goes through LDS.
//
// Twiddles come from a table tw[m] = exp(-2*pi*i*m/n) evaluated on the host
// (those of the length L in LDS); the inverse transform uses their
// conjugates.  Forward: sign = -1, unnormalised, i.e. the FFTW r2c/c2r
// convention of the reference (src/fluid/compute_potential.c:53-67).
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>

namespace sns {

__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ double2 cscale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
// multiply by sign*i
template <int SIGN>
__device__ __forceinline__ double2 cmul_si(double2 a) {
  return SIGN < 0 ? make_double2(a.y, -a.x) : make_double2(-a.y, a.x);
}
// w for the forward transform, its conjugate for the inverse
template <int SIGN>
__device__ __forceinline__ double2 cdir(double2 w) {
  return SIGN < 0 ? w : make_double2(w.x, -w.y);
}

// Quotients of small non-negative integers by a divisor fixed for a loop:
// for 0 <= x < 2^16 and 1 <= d < 2^16, floor(x * ceil(2^32/d) / 2^32) =
// floor(x/d) (the error term x*(ceil(2^32/d) - 2^32/d)/2^32 stays below
// 2^-16, less than the distance 1/d of x/d to the next integer).
struct FastDiv {
  unsigned m;
  int d;
  FastDiv() = default;
  __host__ __device__ explicit FastDiv(int dv)
      : m(dv == 1 ? 0u : (unsigned)(0xFFFFFFFFull / (unsigned)dv + 1)), d(dv) {}
  __device__ __forceinline__ int div(int x) const {
    return d == 1 ? x : (int)__umulhi((unsigned)x, m);
  }
};

// ------------------------------------------------------------- codelets

template <int R, int SIGN>
struct Dft;

template <int SIGN>
struct Dft<2, SIGN> {
  __device__ __forceinline__ static void run(double2 *x) {
    const double2 a = x[0], b = x[1];
    x[0] = cadd(a, b);
    x[1] = csub(a, b);
  }
};

template <int SIGN>
struct Dft<4, SIGN> {
  __device__ __forceinline__ static void run(double2 *x) {
    const double2 t0 = cadd(x[0], x[2]), t1 = csub(x[0], x[2]);
    const double2 t2 = cadd(x[1], x[3]), t3 = cmul_si<SIGN>(csub(x[1], x[3]));
    x[0] = cadd(t0, t2);
    x[2] = csub(t0, t2);
    x[1] = cadd(t1, t3);
    x[3] = csub(t1, t3);
  }
};

template <int SIGN>
struct Dft<8, SIGN> {
  __device__ __forceinline__ static void run(double2 *x) {
    constexpr double c = 0.70710678118654752440;  // sqrt(2)/2
    double2 e[4] = {x[0], x[2], x[4], x[6]};
    double2 o[4] = {x[1], x[3], x[5], x[7]};
    Dft<4, SIGN>::run(e);
    Dft<4, SIGN>::run(o);
    // o_k *= exp(sign*2*pi*i*k/8)
    const double2 o1 = make_double2(c * (o[1].x - SIGN * o[1].y), c * (o[1].y + SIGN * o[1].x));
    const double2 o2 = cmul_si<SIGN>(o[2]);
    const double2 o3 = make_double2(-c * (o[3].x + SIGN * o[3].y), c * (SIGN * o[3].x - o[3].y));
    x[0] = cadd(e[0], o[0]);
    x[4] = csub(e[0], o[0]);
    x[1] = cadd(e[1], o1);
    x[5] = csub(e[1], o1);
    x[2] = cadd(e[2], o2);
    x[6] = csub(e[2], o2);
    x[3] = cadd(e[3], o3);
    x[7] = csub(e[3], o3);
  }
};

template <int SIGN>
struct Dft<3, SIGN> {
  __device__ __forceinline__ static void run(double2 *x) {
    constexpr double h = 0.86602540378443864676;  // sqrt(3)/2
    const double2 t1 = cadd(x[1], x[2]);
    const double2 t2 = csub(x[0], cscale(t1, 0.5));
    const double2 t3 = cscale(cmul_si<SIGN>(csub(x[1], x[2])), h);
    x[0] = cadd(x[0], t1);
    x[1] = cadd(t2, t3);
    x[2] = csub(t2, t3);
  }
};

template <int SIGN>
struct Dft<5, SIGN> {
  __device__ __forceinline__ static void run(double2 *x) {
    constexpr double c1 = 0.30901699437494742410;   // cos(2 pi/5)
    constexpr double c2 = -0.80901699437494742410;  // cos(4 pi/5)
    constexpr double s1 = 0.95105651629515357212;   // sin(2 pi/5)
    constexpr double s2 = 0.58778525229247312917;   // sin(4 pi/5)
    const double2 t1 = cadd(x[1], x[4]), t2 = cadd(x[2], x[3]);
    const double2 t3 = csub(x[1], x[4]), t4 = csub(x[2], x[3]);
    const double2 a1 = cadd(x[0], cadd(cscale(t1, c1), cscale(t2, c2)));
    const double2 a2 = cadd(x[0], cadd(cscale(t1, c2), cscale(t2, c1)));
    const double2 b1 = cmul_si<SIGN>(cadd(cscale(t3, s1), cscale(t4, s2)));
    const double2 b2 = cmul_si<SIGN>(csub(cscale(t3, s2), cscale(t4, s1)));
    x[0] = cadd(x[0], cadd(t1, t2));
    x[1] = cadd(a1, b1);
    x[4] = csub(a1, b1);
    x[2] = cadd(a2, b2);
    x[3] = csub(a2, b2);
  }
};

// R = A*B with A, B coprime, without twiddles (Good's prime-factor map):
// inputs n = (B*a + A*b) mod R, outputs the k with k = ka mod A, k = kb mod B.
template <int A, int B, int SIGN>
struct DftCoprime {
  static constexpr int R = A * B;
  static constexpr int out(int ka, int kb) {
    int k = ka;
    while (k % B != kb) k += A;
    return k;
  }
  __device__ __forceinline__ static void run(double2 *x) {
    double2 y[A][B];
#pragma unroll
    for (int a = 0; a < A; a++) {
#pragma unroll
      for (int b = 0; b < B; b++) y[a][b] = x[(B * a + A * b) % R];
      Dft<B, SIGN>::run(y[a]);
    }
#pragma unroll
    for (int b = 0; b < B; b++) {
      double2 z[A];
#pragma unroll
      for (int a = 0; a < A; a++) z[a] = y[a][b];
      Dft<A, SIGN>::run(z);
#pragma unroll
      for (int a = 0; a < A; a++) x[out(a, b)] = z[a];
    }
  }
};
template <int SIGN>
struct Dft<6, SIGN> : DftCoprime<2, 3, SIGN> {};
template <int SIGN>
struct Dft<10, SIGN> : DftCoprime<2, 5, SIGN> {};
template <int SIGN>
struct Dft<12, SIGN> : DftCoprime<4, 3, SIGN> {};
template <int SIGN>
struct Dft<15, SIGN> : DftCoprime<3, 5, SIGN> {};

// R = Q*Q: DFTs of the Q residues, twiddles w_R^(n2*k1), DFTs across.
template <int Q, int SIGN, class W>
struct DftSquare {
  __device__ __forceinline__ static void run(double2 *x) {
    double2 y[Q][Q];
#pragma unroll
    for (int b = 0; b < Q; b++) {
#pragma unroll
      for (int a = 0; a < Q; a++) y[b][a] = x[Q * a + b];
      Dft<Q, SIGN>::run(y[b]);
    }
#pragma unroll
    for (int k = 0; k < Q; k++) {
      double2 z[Q];
#pragma unroll
      for (int b = 0; b < Q; b++) {
        const int m = b * k;
        if (m == 0) z[b] = y[b][k];
        else if (4 * m == Q * Q) z[b] = cmul_si<SIGN>(y[b][k]);
        else z[b] = cmul(y[b][k], make_double2(W::c(m), SIGN * W::s(m)));
      }
      Dft<Q, SIGN>::run(z);
#pragma unroll
      for (int b = 0; b < Q; b++) x[k + Q * b] = z[b];
    }
  }
};
struct W9 {  // cos, sin of 2 pi m/9, m = 1, 2, 4
  static constexpr double c(int m) {
    return m == 1 ? 0.76604444311897803520 : m == 2 ? 0.17364817766693034885
                                                    : -0.93969262078590838405;
  }
  static constexpr double s(int m) {
    return m == 1 ? 0.64278760968653932632 : m == 2 ? 0.98480775301220805937
                                                    : 0.34202014332566873304;
  }
};
struct W16 {  // cos, sin of 2 pi m/16, m = 1, 2, 3, 6, 9
  static constexpr double k1 = 0.92387953251128675613;  // cos(pi/8)
  static constexpr double k2 = 0.70710678118654752440;  // cos(pi/4)
  static constexpr double k3 = 0.38268343236508977173;  // cos(3 pi/8)
  static constexpr double c(int m) {
    return m == 1 ? k1 : m == 2 ? k2 : m == 3 ? k3 : m == 6 ? -k2 : -k1;
  }
  static constexpr double s(int m) {
    return m == 1 ? k3 : m == 2 ? k2 : m == 3 ? k1 : m == 6 ? k2 : -k3;
  }
};
template <int SIGN>
struct Dft<9, SIGN> : DftSquare<3, SIGN, W9> {};
template <int SIGN>
struct Dft<16, SIGN> : DftSquare<4, SIGN, W16> {};

// -------------------------------------------------------------- schedule

// Stages of a transform of length L: radices in order, sub-transform lengths.
constexpr int kFftStages = 4;
struct FftSched {
  int L, np;
  int r[kFftStages];
  FastDiv ns[kFftStages];
  int rmin;  // threads = sequences * L / rmin
};

constexpr int kRadix[] = {2, 3, 4, 5, 6, 8, 9, 10, 12, 15, 16};

// Ascending radices up to rmax, up to npmax stages: the smallest number of stages (two at least),
// then the largest smallest radix.  False when L has no such product.
inline bool fft_sched(int L, FftSched &sc, int rmax, int npmax) {
  sc = FftSched{};
  sc.L = L;
  int r[kFftStages];
  // choose np radices >= r[p-1] with product `rest`
  auto pick = [&](auto &&self, int p, int np, int rest) -> bool {
    if (p == np) return rest == 1;
    for (int k = (int)(sizeof kRadix / sizeof kRadix[0]) - 1; k >= 0; k--) {
      const int a = kRadix[k];
      if (a > rmax || rest % a || (p && a < r[p - 1])) continue;
      r[p] = a;
      if (self(self, p + 1, np, rest / a)) return true;
    }
    return false;
  };
  for (int np = 2; np <= npmax && !sc.np; np++)
    if (pick(pick, 0, np, L)) sc.np = np;
  if (!sc.np) {  // a prime length: one stage
    for (int a : kRadix)
      if (a == L && a <= rmax) sc.np = 2;
    if (!sc.np) return false;
    r[0] = 1;
    r[1] = L;
  }
  int ns = 1;
  sc.rmin = r[0];
  for (int p = 0; p < sc.np; p++) {
    sc.r[p] = r[p];
    sc.ns[p] = FastDiv(ns);
    ns *= r[p];
  }
  return true;
}

// Schedules known to the kernel: every index is a constant's multiple and only
// the radices it takes are compiled in.
template <int... R>
struct FixedSched {
  static constexpr int rmax = 16, npmax = kFftStages;
  __device__ __forceinline__ static FftSched get(const FftSched &) {
    constexpr int r[] = {R...};
    FftSched sc{};
    sc.np = (int)sizeof...(R);
    int ns = 1;
    for (int p = 0; p < sc.np; p++) {
      sc.r[p] = r[p];
      sc.ns[p] = FastDiv(ns);
      ns *= r[p];
    }
    sc.L = ns;
    return sc;
  }
  static FftSched make() {
    constexpr int r[] = {R...};
    FftSched sc{};
    sc.np = (int)sizeof...(R);
    sc.L = 1;
    sc.rmin = r[0];
    for (int p = 0; p < sc.np; p++) {
      if (r[p] < sc.rmin) sc.rmin = r[p];
      sc.r[p] = r[p];
      sc.ns[p] = FastDiv(sc.L);
      sc.L *= r[p];
    }
    return sc;
  }
  static bool is(const FftSched &sc) {
    constexpr int r[] = {R...};
    bool same = sc.np == (int)sizeof...(R);
    for (int p = 0; same && p < sc.np; p++) same = sc.r[p] == r[p];
    return same;
  }
};
// Any schedule of up to NP stages with radices up to RMAX.
template <int RMAX, int NP>
struct AnySched {
  static constexpr int rmax = RMAX, npmax = NP;
  __device__ __forceinline__ static const FftSched &get(const FftSched &sc) { return sc; }
};

// ---------------------------------------------------------------- stages

// LDS slot of element e: one unused slot in nine spreads the strided stores
// of few sequences over the banks.
__device__ __forceinline__ int fft_pad(int e) { return e + (e >> 3); }
constexpr size_t fft_slots(int elems) { return (size_t)elems + elems / 8; }

// Element idx of sequence s lives at buf[fft_pad(idx*S + s)], so consecutive
// threads touch consecutive LDS words.
struct FftLds {
  double2 *buf;  // fft_slots(S*L)
  double2 *tw;   // L twiddles exp(-2 pi i m/L)
  int S;
  FastDiv fs;
};

__device__ __forceinline__ FftLds fft_lds(double2 *lds, const FftSched &sc, int S,
                                          const double2 *__restrict__ tw, int n) {
  FftLds l = {lds, lds + fft_slots(S * sc.L), S, FastDiv(S)};
  const int step = n / sc.L;
  for (int m = threadIdx.x; m < sc.L; m += blockDim.x) l.tw[m] = tw[m * step];
  return l;
}

// First stage: inputs from load(s)(idx).
template <int R, int SIGN, bool BATCH, class Ld>
__device__ __forceinline__ void fft_first(const FftLds &l, const FftSched &sc, Ld load) {
  const int nb = sc.L / R;
  if ((int)threadIdx.x < l.S * nb) {
    const int j = l.fs.div(threadIdx.x), s = threadIdx.x - j * l.S;
    double2 x[R];
    auto in = load(s);
#pragma unroll
    for (int r = 0; r < R; r++) {
      x[r] = in(j + r * nb);
      // inputs that take several loads: 4 at a time (registers)
      if (BATCH && r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (R > 1) Dft<R, SIGN>::run(x);
#pragma unroll
    for (int r = 0; r < R; r++) l.buf[fft_pad((j * R + r) * l.S + s)] = x[r];
  }
}

// Stage p from LDS, back into LDS (in place: the barrier after the reads) or,
// OUT, to store(s)(idx, value).
template <int R, int SIGN, bool OUT, class St>
__device__ __forceinline__ void fft_stage(const FftLds &l, const FftSched &sc, FastDiv ns,
                                          St store) {
  const int nb = sc.L / R;
  const bool on = (int)threadIdx.x < l.S * nb;
  const int j = l.fs.div(threadIdx.x), s = threadIdx.x - j * l.S;
  const int kk = j - ns.div(j) * ns.d;
  double2 x[R];
  if (on) {
#pragma unroll
    for (int r = 0; r < R; r++) x[r] = l.buf[fft_pad((j + r * nb) * l.S + s)];
    // w_(Ns R)^(r kk) = w_L^(r kk L/(Ns R))
    if (ns.d > 1) {
      const int step = kk * (sc.L / (ns.d * R));
#pragma unroll
      for (int r = 1; r < R; r++) x[r] = cmul(x[r], cdir<SIGN>(l.tw[r * step]));
    }
    if constexpr (R > 1) Dft<R, SIGN>::run(x);
  }
  const int base = (j - kk) * R + kk;
  if constexpr (OUT) {
    if (on) {
      auto out = store(s);
#pragma unroll
      for (int r = 0; r < R; r++) {
        out(base + r * ns.d, x[r]);
        if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
    }
  } else {
    __syncthreads();
    if (on) {
#pragma unroll
      for (int r = 0; r < R; r++) l.buf[fft_pad((base + r * ns.d) * l.S + s)] = x[r];
    }
  }
}

// f(radix) with the radix as a constant
template <int RMAX, class F>
__device__ __forceinline__ void fft_radix(int r, F f) {
  switch (r) {
    case 2: f(std::integral_constant<int, 2>()); break;
    case 3: f(std::integral_constant<int, 3>()); break;
    case 4: f(std::integral_constant<int, 4>()); break;
    case 5: f(std::integral_constant<int, 5>()); break;
    case 6: f(std::integral_constant<int, 6>()); break;
    case 8: f(std::integral_constant<int, 8>()); break;
    case 9: f(std::integral_constant<int, 9>()); break;
    case 10: f(std::integral_constant<int, 10>()); break;
    default:
      if constexpr (RMAX > 10) {
        if (r == 12) f(std::integral_constant<int, 12>());
        else if (r == 15) f(std::integral_constant<int, 15>());
        else f(std::integral_constant<int, 16>());
      }
  }
}

// The whole transform.  IN: from load(s)(idx), else from LDS (complete before
// the call).  OUT: to store(s)(idx, value), else into LDS (complete after).
// load and store are given the sequence once per butterfly, so what depends on
// it alone (column metrics, addresses) is formed once.  Sc: the schedule's type.
template <class Sc, int SIGN, bool IN, bool OUT, bool BATCH = false, class Ld, class St>
__device__ __forceinline__ void fft_run(const FftLds &l, const FftSched &sc, Ld load, St store) {
  auto mid = [&](int r, FastDiv ns) {
    fft_radix<Sc::rmax>(r, [&](auto R) { fft_stage<R(), SIGN, false>(l, sc, ns, store); });
    __syncthreads();
  };
  if constexpr (IN) {
    if (sc.r[0] == 1) fft_first<1, SIGN, BATCH>(l, sc, load);
    else fft_radix<Sc::rmax>(sc.r[0], [&](auto R) { fft_first<R(), SIGN, BATCH>(l, sc, load); });
    __syncthreads();
  } else if (sc.r[0] != 1) {
    mid(sc.r[0], sc.ns[0]);
  }
  int rl = sc.r[1];
  FastDiv nl = sc.ns[1];
  if (sc.np > 2) {
    mid(rl, nl);
    rl = sc.r[2];
    nl = sc.ns[2];
  }
  if constexpr (Sc::npmax > 3) {
    if (sc.np > 3) {
      mid(rl, nl);
      rl = sc.r[3];
      nl = sc.ns[3];
    }
  }
  fft_radix<Sc::rmax>(rl, [&](auto R) { fft_stage<R(), SIGN, OUT>(l, sc, nl, store); });
  if constexpr (!OUT) __syncthreads();
}

}  // namespace sns
