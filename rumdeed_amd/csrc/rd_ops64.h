// FP64 square roots, reciprocals and quotients, correctly rounded, without the
// range handling of the general IEEE sequences.  The compiler's general
// sequences spend 93 and 69 cycles a wave on a square root and a division
// (measured, gfx950), about half on scaling operands that might overflow or be
// subnormal and on special values; the same Goldschmidt / Newton sequences
// without the scaling take 52 and 40 cycles.  Both forms are correctly
// rounded, so they agree bit for bit wherever the operands are ordinary.
#pragma once

#include <hip/hip_runtime.h>

namespace rd {

// Zero, or a magnitude in [2^-100, 2^101): differences of such coordinates
// are zero or at least 2^-153, so the squares, cubes and products of the pair
// terms and their quotients stay far inside the normal range.
__device__ __forceinline__ bool f64_ordinary(double v) {
  const unsigned e = ((unsigned)__double2hiint(v) >> 20) & 0x7ffu;
  return v == 0.0 || e - (1023u - 100u) <= 200u;
}

// The general IEEE operations.
struct Ieee64 {
  static __device__ __forceinline__ double lift(double v) { return v; }
  static __device__ __forceinline__ double sqrt(double x) { return __builtin_sqrt(x); }
  static __device__ __forceinline__ double rcp(double x) { return 1.0 / x; }
  struct Div {
    double b;
    __device__ __forceinline__ explicit Div(double den) : b(den) {}
    __device__ __forceinline__ double operator()(double a) const { return a / b; }
  };
};

// The same results for ordinary operands.  v_rsq_f64 and v_rcp_f64 are
// accurate to 2^-24; one Goldschmidt step and two residual corrections give
// the correctly rounded root, two Newton steps and one residual correction
// the correctly rounded quotient (Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", 1990).  The residuals
// r = x - g g and r = a - b q are exact in one fma.  Compared with the general
// operations on 1e9 operands: no difference.
struct Fast64 {
  // Added to dx^2 + dy^2 of a pair: turns an exact zero distance, whose
  // reciprocal root is infinite, into one of 2^-500 that the softening (1e-18
  // added to the root) absorbs exactly; the sums of squares, zero or above 2^-306, are
  // unchanged.
  static __device__ __forceinline__ double lift(double v) { return v + 0x1p-1000; }
  static __device__ __forceinline__ double sqrt(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    double d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    d = __builtin_fma(-g, g, x);
    return __builtin_fma(d, h, g);
  }
  static __device__ __forceinline__ double recip(double b) {
    double y = __builtin_amdgcn_rcp(b);
    double e = __builtin_fma(-b, y, 1.0);
    y = __builtin_fma(y, e, y);
    e = __builtin_fma(-b, y, 1.0);
    return __builtin_fma(y, e, y);
  }
  static __device__ __forceinline__ double rcp(double b) {
    const double y = recip(b);
    return __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
  }
  // Quotients by one denominator share its reciprocal.
  struct Div {
    double b, y;
    __device__ __forceinline__ explicit Div(double den) : b(den), y(recip(den)) {}
    __device__ __forceinline__ double operator()(double a) const {
      const double q = a * y;
      return __builtin_fma(__builtin_fma(-b, q, a), y, q);
    }
  };
};

}  // namespace rd
