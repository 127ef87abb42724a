// sns_poisson_one.hip -- y transforms of whole columns in one kernel (gfx950).
//
// The transforms of src/fluid/compute_potential.c:53-67, 147-168 for grids small
// enough that launches and latency count (rule: one_pass_pairs): a workgroup
// holds all rows of a few column pairs in LDS, so the forward transform (with
// the right-hand side) and the inverse one (with psi's boundary values) take
// one kernel each instead of two.  What bounds them is latency: the loads of the
// right-hand side, one thread's chain of butterflies, the barriers.  us, forward
// and inverse, two passes and one kernel: 32x64 16.0 and 9.2, 128x192 19.9 and
// 10.7, 225x360 24.5 and 17.6, 512x1024 24.4 and 19.1.
#include "sns_poisson_dev.h"

namespace sns {

// Small grids: the whole transform of 2^lgt column pairs in one workgroup.
template <class Sc, bool AL>
__device__ __forceinline__ void pfwd_one(const PoisArgs &a) {
  extern __shared__ double2 lds_fft[];
  const Fft2Plan &pl = a.pl;
  const FftSched &sc = Sc::get(pl.s1);
  const int T = 1 << pl.lgt, n = pl.n;
  const int pair0 = xcd_remap(blockIdx.x, gridDim.x) << pl.lgt;
  const double inv_gdt = 1. / (a.gamma * (*a.dtp));
  const FftLds l = fft_lds(lds_fft, sc, T, a.tw, n);
  fft_run<Sc, -1, true, false, AL>(
      l, sc,
      [&](int s) { return RhsCol<false, AL>(a, inv_gdt, pair0 + s); },
      NoIo{});
#pragma unroll 4
  for (int e = threadIdx.x; e < (n / 2 + 1) << pl.lgt; e += blockDim.x) {
    const int k = e >> pl.lgt, q = e & (T - 1);
    put_spectra(a, k, pair0 + q, l.buf[fft_pad(e)], l.buf[fft_pad(((k ? n - k : 0) << pl.lgt) + q)]);
  }
}

template <class Sc, bool AL>
__device__ __forceinline__ void pinv_one(const PoisArgs &a) {
  extern __shared__ double2 lds_fft[];
  const Fft2Plan &pl = a.pl;
  const FftSched &sc = Sc::get(pl.s1);
  const int T = 1 << pl.lgt, n = pl.n;
  const int pair0 = xcd_remap(blockIdx.x, gridDim.x) << pl.lgt;
  const FftLds l = fft_lds(lds_fft, sc, T, a.tw, n);
#pragma unroll 4
  for (int e = threadIdx.x; e < (n / 2 + 1) << pl.lgt; e += blockDim.x) {
    const int k = e >> pl.lgt, q = e & (T - 1);
    double2 zn;
    l.buf[fft_pad(e)] = get_spectra(a, k, pair0 + q, zn);
    if (k != 0 && 2 * k != n) l.buf[fft_pad(((n - k) << pl.lgt) + q)] = zn;
  }
  __syncthreads();
  fft_run<Sc, +1, false, true>(l, sc, NoIo{}, [&](int s) { return PsiCol<AL>(a, pair0 + s); });
}

SNS_FFT_KERNEL(pfwd_one, bool AL SNS_C, SNS_C AL)
SNS_FFT_KERNEL(pinv_one, bool AL SNS_C, SNS_C AL)

// Schedules compiled in for 2^k, 3*2^k and 5*2^k rows, other lengths read
// theirs.  Radix 4 first: what bounds these kernels is one thread's chain of
// instructions, and a butterfly of radix 4 is half of one of radix 8.
template <class F>
static bool fixed_sched(F f) {
#define SNS_TRY(...) if (f(FixedSched<__VA_ARGS__>{})) return true;
  SNS_TRY(4, 4) SNS_TRY(4, 8) SNS_TRY(4, 4, 4) SNS_TRY(4, 4, 8) SNS_TRY(4, 4, 4, 4)
  SNS_TRY(4, 4, 4, 8) SNS_TRY(4, 4, 8, 8)
  SNS_TRY(3, 4, 4) SNS_TRY(4, 4, 6) SNS_TRY(3, 4, 4, 4) SNS_TRY(4, 4, 4, 6) SNS_TRY(4, 4, 6, 8)
  SNS_TRY(4, 4, 5) SNS_TRY(4, 5, 8) SNS_TRY(4, 4, 4, 5) SNS_TRY(4, 4, 5, 8)
#undef SNS_TRY
  return false;
}
using Any = AnySched<10, 4>;

bool one_pass_sched(int n, FftSched &sc) {
  if (fixed_sched([&](auto f) {
        sc = f.make();
        return sc.L == n;
      }))
    return true;
  return fft_sched(n, sc, Any::rmax, Any::npmax);
}

// f(schedule type) for the schedule sc; the unaligned layout always reads it.
template <class F>
static void with_sched(const FftSched &sc, F f) {
  if (!fixed_sched([&](auto t) {
        if (!t.is(sc)) return false;
        f(t);
        return true;
      }))
    f(Any{});
}

template <class S>
void one_pass_forward(hipStream_t s, const Fft2Plan &pl, bool aligned, S src, int nz) {
  const int T = 1 << pl.lgt;
  const dim3 grid((pl.npair + T - 1) / T);
  if (!aligned) SNS_FFT_LAUNCH((k_pfwd_one<Any, false, S>), T, pl.s1, grid);
  else
    with_sched(pl.s1, [&](auto sc) {
      SNS_FFT_LAUNCH((k_pfwd_one<decltype(sc), true, S>), T, pl.s1, grid);
    });
}

template <class S>
void one_pass_inverse(hipStream_t s, const Fft2Plan &pl, bool aligned, S src, int nz) {
  const int T = 1 << pl.lgt;
  const dim3 grid((pl.npair + T - 1) / T);
  if (!aligned) SNS_FFT_LAUNCH((k_pinv_one<Any, false, S>), T, pl.s1, grid);
  else
    with_sched(pl.s1, [&](auto sc) {
      SNS_FFT_LAUNCH((k_pinv_one<decltype(sc), true, S>), T, pl.s1, grid);
    });
}

template void one_pass_forward(hipStream_t, const Fft2Plan &, bool, ArgOne<PoisArgs>, int);
template void one_pass_forward(hipStream_t, const Fft2Plan &, bool, ArgBatch<PoisArgs>, int);
template void one_pass_inverse(hipStream_t, const Fft2Plan &, bool, ArgOne<PoisArgs>, int);
template void one_pass_inverse(hipStream_t, const Fft2Plan &, bool, ArgBatch<PoisArgs>, int);

}  // namespace sns
