// erfcx for the Ewald direct sum (plain C++17, shared by the HIP kernel and a
// host-side check).
#pragma once

#include <cmath>
#include <utility>
#include <vector>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define EW_HD __host__ __device__ __forceinline__
#else
#define EW_HD inline
#endif

namespace gse {

// erfc(x) = exp(-x^2) erfcx(x), and the pair term needs that exponential
// anyway: erfcx is a polynomial of degree 11 about the centre of x's
// interval (width 1/4 below 8, 1 up to 27, where erfc underflows), fitted at
// Chebyshev nodes in extended precision; its error is below one unit in the
// last place (2.1e-16), at 12 multiply-adds where the library's erfc takes
// about 150 FP64 instructions.
constexpr int kErfcxRows = 51, kErfcxDeg = 11, kErfcxPitch = 14;  // doubles a row, 16-byte rows

inline std::vector<double> make_erfcx_table() {
  typedef long double L;
  const L pi = 3.14159265358979323846264338327950288L;
  constexpr int n = kErfcxDeg + 1;
  std::vector<double> out(kErfcxRows * kErfcxPitch, 0.0);
  for (int row = 0; row < kErfcxRows; row++) {
    const L c = row < 32 ? (row + 0.5L) * 0.25L : row - 24 + 0.5L, h = row < 32 ? 0.125L : 0.5L;
    L f[n], mono[n] = {}, t0[n] = {}, t1[n] = {};
    for (int k = 0; k < n; k++) {
      const L x = c + h * cosl(pi * (k + 0.5L) / n);
      f[k] = erfcl(x) * expl(x * x);
    }
    // sum of the Chebyshev polynomials as powers of u = (x - c) / h
    t0[0] = 1.0L;
    t1[1] = 1.0L;
    for (int j = 0; j < n; j++) {
      L a = 0.0L;
      for (int k = 0; k < n; k++) a += f[k] * cosl(pi * j * (k + 0.5L) / n);
      a *= (j == 0 ? 1.0L : 2.0L) / n;
      for (int k = 0; k < n; k++) mono[k] += a * t0[k];
      for (int k = n - 1; k >= 0; k--) {  // (T_j, T_j+1) -> (T_j+1, T_j+2)
        const L next = (k > 0 ? 2.0L * t1[k - 1] : 0.0L) - t0[k];
        t0[k] = next;
      }
      for (int k = 0; k < n; k++) std::swap(t0[k], t1[k]);
    }
    L p = 1.0L;
    for (int k = 0; k < n; k++, p *= h) out[row * kErfcxPitch + k] = (double)(mono[k] / p);
  }
  return out;
}

EW_HD double ew_erfcx(const double* tab, double x) {
  x = x < 27.0 ? x : 27.0;  // the product is below the normal range from there on
  const bool fine = x < 8.0;
  const int cell = (int)(fine ? 4.0 * x : x);
  const int at = fine ? cell : cell + 24, row = at < kErfcxRows ? at : kErfcxRows - 1;
  const double mid = (double)cell + 0.5, d = x - (fine ? 0.25 * mid : mid);
  const double* t = tab + row * kErfcxPitch;
  double v = t[kErfcxDeg];
#ifdef __HIPCC__
#pragma unroll
#endif
  for (int k = kErfcxDeg - 1; k >= 0; k--) v = __builtin_fma(v, d, t[k]);
  return v;
}

}  // namespace gse
