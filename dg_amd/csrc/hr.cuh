// Hierarchical-reconstruction helpers in the Taylor basis x^n/n! on [-1,1]
// (limiting_kernels.cu:1470-1486 minmod, 1534-1583 limit_monomial,
// 1748-1790 integrals and average_monomial).  Every body is compiled without
// FMA contraction so that the limiter rounds like the CPU path whichever
// translation unit includes this header.
#pragma once

namespace dgx {

// minmod (limiting_kernels.cu:1470-1486): the argument of smaller magnitude
// where both have the same sign, else +0.  In the reference's terms (sa, sb
// the signs, 0 for a zero or a NaN) a NaN gives 0 unless both signs are 0,
// then 0*|b|: kept.  Signs and magnitudes are taken from the bits, and every
// value is formed before it is selected: a branch here cuts the unrolled
// limiters into blocks (half the instructions of integer signs and their
// products).
__device__ inline double minmod_d(double a, double b) {
#pragma clang fp contract(off)
  const double m = fmin(fabs(a), fabs(b)), limited = copysign(m, a);
  const bool same = (__builtin_bit_cast(long, a) ^ __builtin_bit_cast(long, b)) >= 0;
  const bool both = same & (m > 0) & !__builtin_isunordered(a, b);
  const bool nan = (b != b) & !(fabs(a) > 0);
  const double r = both ? limited : 0.0;
  return nan ? b : r;
}

// skip_zero_terms: the loops below leave out the products with a zero
// integral (known once the loops are unrolled).  Each left-out product of a
// finite value is +-0, and adding +-0 to a sum that started at +0.0 does not
// change it: a non-zero sum stays as it is, and in round-to-nearest the sum
// is never -0 (x + (-x) = +0 and +0 + (-0) = +0).  The results are therefore
// the bits of the full sums the reference forms.
__host__ __device__ constexpr int ifact(int n) { return n <= 1 ? 1 : n * ifact(n - 1); }
__host__ __device__ constexpr long ipow(long b, int n) { return n == 0 ? 1 : b * ipow(b, n - 1); }

// integral over [-1,1] of the k-th derivative of x^n/n! (limiting_kernels.cu:1748-1760)
__device__ inline double integ_deriv(int k, int n) {
#pragma clang fp contract(off)
  int num = n - k + 1;
  if (num % 2) return 2.0 / (double)ifact(num);
  return 0.0;
}
// over [a,b] with integer a,b (limiting_kernels.cu:1762-1775); powers are exact
__device__ inline double integ_deriv_bounds(int k, int n, int a, int b) {
#pragma clang fp contract(off)
  int num = n - k + 1;
  return ((double)ipow(b, num) - (double)ipow(a, num)) / (double)ifact(num);
}

// avg[m-1], m = 1..N: the integral over [-1,1] of the (m-1)-th derivative of a
// slice, all that limit_monomial takes from it
template <int N>
__device__ inline void derivative_averages(const double* A, double* avg) {
#pragma clang fp contract(off)
#pragma unroll
  for (int m = 1; m <= N; m++) {
    double s = 0;
#pragma unroll
    for (int n = m - 1; n <= N; n++) {
      // the zero integrals (n - m even) are left out: see skip_zero_terms
      const double integral = integ_deriv(m - 1, n);
      if (integral != 0.0) s += A[n] * integral;
    }
    avg[m - 1] = s;
  }
}

// limit_monomial from the averages of the left, own and right slices
template <int N>
__device__ inline void limit_averages(const double* L, const double* C, const double* R, double* Alim) {
#pragma clang fp contract(off)
  double avgLC = 0;
#pragma unroll
  for (int n = 0; n <= N; n++) Alim[n] = 0;
#pragma unroll
  for (int m = N; m > 0; m--) {
    double avgRL = 0, avgRC = 0, avgRR = 0;
#pragma unroll
    for (int n = m + 1; n <= N; n++) {
      const double alim = Alim[n], integral = integ_deriv(m - 1, n);
      avgRL += alim * integ_deriv_bounds(m - 1, n, -3, -1);
      if (integral != 0.0) avgRC += alim * integral;
      avgRR += alim * integ_deriv_bounds(m - 1, n, 1, 3);
    }
    double avgLL = 0.5 * (L[m - 1] - avgRL);
    avgLC = 0.5 * (C[m - 1] - avgRC);
    double avgLR = 0.5 * (R[m - 1] - avgRR);
    double c1 = 0.5 * (avgLC - avgLL);
    double c2 = 0.5 * (avgLR - avgLC);
    Alim[m] = minmod_d(c1, c2);
  }
  Alim[0] = avgLC;
}

template <int N>
__device__ inline void limit_monomial_d(const double* AL, const double* AC, const double* AR, double* Alim) {
  double L[N], C[N], R[N];
  derivative_averages<N>(AL, L);
  derivative_averages<N>(AC, C);
  derivative_averages<N>(AR, R);
  limit_averages<N>(L, C, R, Alim);
}

template <int N>
__device__ inline void average_monomial_d(const double* A, double* Alim) {
#pragma clang fp contract(off)
  double avg = 0;
#pragma unroll
  for (int n = 0; n <= N; n++) {
    if (integ_deriv(0, n) != 0.0) avg += A[n] * integ_deriv(0, n);
    Alim[n] = 0;
  }
  Alim[0] = 0.5 * avg;
}

}  // namespace dgx
