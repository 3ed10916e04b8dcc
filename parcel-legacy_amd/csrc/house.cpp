// house.cpp -- Householder R factor of the stacked first-level TSQR factors
// (House_local_Ronly_omp, TSQR.f90:114-261), the host half of tsqr_r.
//
// The same operations in the same order as dense.hpp's house_r: every column's
// sums run down the rows.  The sums of one reflector are independent chains,
// so the rows are held contiguously and all columns advance together, and the
// update by one reflector and the sums of the next share one pass over the
// rows.  8192 x 8 (1024 factors): 1.49 ms as house_r's column loops, whose
// fma() calls the C library, 0.22 ms here (one core); a CA-GMRES(8, 4) restart runs
// it four times.
#include <cmath>
#include <vector>

#include "house.hpp"

namespace parcel {

#if defined(__x86_64__)
namespace {

// Rows of S: element (j, k) at S[j * N + k].
template <int N>
__attribute__((target("avx2,fma"))) void house_rows(int m, double* S, double* R) {
  double d[N];  // d[k] = sum over rows j > i of S(j, i) S(j, k), in row order, from d0[k]
  // column i's own sum starts from 0, the others from y1 * S(i, k), which is
  // known only after the own sum: two passes for the first reflector
  double own = 0.0;
  for (int j = 1; j < m; ++j) own = __builtin_fma(S[(long)j * N], S[(long)j * N], own);
  for (int i = 0; i < N; ++i) {
    double* si = S + (long)i * N;
    const double aii = si[i];
    const double tmp3 = std::sqrt(__builtin_fma(aii, aii, own));
    const double y1 = aii > 0.0 ? aii + tmp3 : aii - tmp3;
    const double tmp = __builtin_fma(y1, aii, own);
    double den = __builtin_fma(y1, y1, own);
    if (den == 0.0) den = 1.0 - 300;
    const double t1 = 2.0 / den;
    si[i] = __builtin_fma(-(t1 * y1), tmp, aii);
    if (i + 1 == N) break;
    for (int k = 0; k < N; ++k) d[k] = y1 * si[k];
    for (int j = i + 1; j < m; ++j) {
      const double* s = S + (long)j * N;
      const double x = s[i];
#pragma clang loop vectorize(enable)
      for (int k = 0; k < N; ++k) d[k] = __builtin_fma(x, s[k], d[k]);
    }
    for (int k = 0; k < N; ++k) d[k] = t1 * d[k];
    // update columns k > i of the rows below i (column i is not read again),
    // and the next column's own sum over the rows below i + 1
    double next = 0.0;
    for (int j = i + 1; j < m; ++j) {
      double* s = S + (long)j * N;
      const double x = s[i];
#pragma clang loop vectorize(enable)
      for (int k = 0; k < N; ++k) s[k] = __builtin_fma(-x, d[k], s[k]);
      if (j > i + 1) next = __builtin_fma(s[i + 1], s[i + 1], next);
    }
    for (int k = i + 1; k < N; ++k) si[k] = __builtin_fma(-y1, d[k], si[k]);
    own = next;
  }
  for (int j = 0; j < N; ++j)
    for (int i = 0; i < N; ++i) R[i + (long)j * N] = i <= j ? S[(long)i * N + j] : 0.0;
}

}  // namespace

bool house_r_rows(int m, int n, double* S, double* R) {
  static const bool ok = __builtin_cpu_supports("fma") && __builtin_cpu_supports("avx2");
  if (!ok || m < n) return false;
  switch (n) {
#define PARCEL_H(N) \
  case N: house_rows<N>(m, S, R); return true;
    PARCEL_H(1) PARCEL_H(2) PARCEL_H(3) PARCEL_H(4) PARCEL_H(5) PARCEL_H(6) PARCEL_H(7) PARCEL_H(8)
    PARCEL_H(9) PARCEL_H(10) PARCEL_H(11) PARCEL_H(12) PARCEL_H(13) PARCEL_H(14) PARCEL_H(15) PARCEL_H(16)
#undef PARCEL_H
    default: return false;
  }
}
#else  // the caller's column loops
bool house_r_rows(int, int, double*, double*) { return false; }
#endif

}  // namespace parcel
