// FP64 exponential and power for the column kernels.
//
// The device library's pow takes 252 instructions (215 of them vector ones) and its exp 60: their polynomials' constants
// are moved into registers one 32-bit half at a time, and every case of their arguments is handled by selects.  FP64
// sweeps run at one or two waves per SIMD, where each instruction of any kind takes an issue slot, and they spend most
// of them here.  These take their constants from a table by scalar loads (up to 8 numbers each).
//
// exp(x) = 2^n e^r, n = round(x / ln 2), |r| <= ln 2 / 2 with r = x - n ln 2 in two parts, e^r = 1 + r + r^2 P(r).
// log(x) = k ln 2 + 2 atanh(s), s = (z - 1) / (z + 1), x = 2^k z, sqrt(1/2) <= z < sqrt(2), in two parts:
// 2 s + s^3 Q(s^2) with s in two parts.  P and Q interpolate at Chebyshev nodes (truncation 2e-19 and 6e-20 of the
// result).  Largest errors measured against long double over 4 million arguments each of 7 ranges.
#pragma once
#include <hip/hip_runtime.h>

namespace fp64 {

struct Table {
  double x[12];  // P, highest power first, and log2(e)
  double l[8];   // Q, highest power first
  double ln2, ln2_lo;     // rounded to double, rest
  double ln2_42, ln2_42_lo;  // 42 bits, so that k ln2_42 is exact, rest
};
static __constant__ const Table table = {
    {0x1.1f7350a074034p-29, 0x1.af4e70dd7207dp-26, 0x1.27e4db3f36203p-22, 0x1.71de01f07539bp-19,
     0x1.a01a01a6e448ep-16, 0x1.a01a01abfc8ddp-13, 0x1.6c16c16c162bfp-10, 0x1.11111111100b6p-7,
     0x1.5555555555556p-5, 0x1.5555555555557p-3, 0x1.0000000000000p-1, 0x1.71547652b82fep+0},
    {0x1.0c0aff044a970p-3, 0x1.0fbde0f4ad17bp-3, 0x1.3b1c3c1c81c8fp-3, 0x1.745cf8e4bba1bp-3,
     0x1.c71c7201a55d7p-3, 0x1.2492492476a1ap-2, 0x1.9999999999a39p-2, 0x1.5555555555555p-1},
    0x1.62e42fefa39efp-1,
    0x1.abc9e3b39803fp-56,
    0x1.62e42fefa2000p-1,
    0x1.9ef35793c7673p-41};

typedef const __attribute__((address_space(4))) Table* TablePtr;
// The table's address, opaque to the compiler, which would else put the numbers into the code again.  (As a volatile
// statement, which keeps every function's loads to itself, the sweep of 65,536 columns takes 1.56 instead of 1.52 ms.)
__device__ __forceinline__ TablePtr constants() {
  TablePtr t = (TablePtr)&table;
  asm("" : "+s"(t));
  return t;
}

__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }

// a b + c with c in scalar registers.  (The compiler prefers the two-operand form, which first copies c.)
__device__ __forceinline__ double fma_s(double a, double b, double c) {
  double d;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
  return d;
}

// 2^n e^(r + l), |r| <= ln 2 / 2, |l| << 1.
__device__ __forceinline__ double exp_reduced(TablePtr c, double n, double r, double l) {
  const double rr = r + l, r2 = rr * rr;
  // even and odd powers apart: two chains of half the length
  double e = fma_s(c->x[0], r2, c->x[2]), o = fma_s(c->x[1], r2, c->x[3]);
  e = fma_s(e, r2, c->x[4]), o = fma_s(o, r2, c->x[5]);
  e = fma_s(e, r2, c->x[6]), o = fma_s(o, r2, c->x[7]);
  e = fma_s(e, r2, c->x[8]), o = fma_s(o, r2, c->x[9]);
  e = fma_s(e, r2, c->x[10]);
  const double p = fma_(o, rr, e);
  const double h = 1.0 + r;
  const double t = fma_(r2, p, (r - (h - 1.0)) + l);
  return __builtin_amdgcn_ldexp(h + t, (int)n);
}

// Exponents beyond +-800 give inf and 0.
__device__ __forceinline__ double clamp_exponent(double x) {
  return __builtin_fmin(__builtin_fmax(x, -800.0), 800.0);
}

__device__ __forceinline__ double exp(double x) {
  const TablePtr c = constants();
  const double a = clamp_exponent(x), n = __builtin_rint(a * c->x[11]);
  const double r = fma_(-n, c->ln2, a), l = -(n * c->ln2_lo);
  const double v = exp_reduced(c, n, r, l);
  return x == x ? v : x;
}

// log|x| = hi + lo, and x, by whose sign, zero or infinity powers differ.
struct Log {
  double hi, lo, x;
};

__device__ __forceinline__ Log log(double x) {
  const TablePtr c = constants();
  const double ax = __builtin_fabs(x);
  const double m = __builtin_amdgcn_frexp_mant(ax);
  const bool low = m < 0x1.6a09e667f3bcdp-1;
  const double z = low ? m + m : m;
  const double k = (double)(__builtin_amdgcn_frexp_exp(ax) - (low ? 1 : 0));
  // s = a / (h + g), h + g = z + 1 exactly
  const double a = z - 1.0, h = z + 1.0, g = z - (h - 1.0);
  double w = __builtin_amdgcn_rcp(h);
  w = fma_(fma_(-h, w, 1.0), w, w);
  w = fma_(fma_(-h, w, 1.0), w, w);
  const double s = a * w;
  const double sl = fma_(-s, g, fma_(-s, h, a)) * w;
  const double u = s * s, u2 = u * u;
  double e = fma_s(c->l[0], u2, c->l[2]), o = fma_s(c->l[1], u2, c->l[3]);
  e = fma_s(e, u2, c->l[4]), o = fma_s(o, u2, c->l[5]);
  e = fma_s(e, u2, c->l[6]), o = fma_s(o, u2, c->l[7]);
  const double q = fma_(e, u, o);
  const double b = s + s, kb = k * c->ln2_42;
  const double hi = kb + b;
  return Log{hi, (b - (hi - kb)) + fma_(s * u, q, fma_(k, c->ln2_42_lo, sl + sl)), x};
}

// x^y where x is 0, infinite, negative or NaN; v = |x|^y for a finite negative x.  x^0 is 1 for each of them: exponents
// are parameters of the scheme, and the sweep takes powers of 0 wherever there is no rain.
__device__ __forceinline__ double pow_special(double x, double y, double v) {
  if (y == 0.0) return 1.0;
  const double ax = __builtin_fabs(x), inf = __builtin_inf();
  const bool whole = __builtin_rint(y) == y;
  const bool odd = whole && __builtin_rint(0.5 * y) != 0.5 * y;
  if (ax == 0.0) v = y > 0.0 ? 0.0 : inf;
  if (ax == inf) v = y > 0.0 ? inf : 0.0;
  if (odd) v = __builtin_copysign(v, x);
  if (x < 0.0 && ax < inf && ax > 0.0 && !whole) v = __builtin_nan("");
  return x == x ? v : x;
}
__device__ __forceinline__ bool ordinary(double x) { return x > 0.0 && x < __builtin_inf(); }

// x^y from log(x), for a finite y.  Largest error 0.69 ulp (the library's pow 1.33), exp 0.69 (0.87).
__device__ __forceinline__ double pow(const Log& b, double y) {
  const TablePtr c = constants();
  const double p = y * b.hi, pl = fma_(y, b.lo, fma_(y, b.hi, -p));
  const double pc = clamp_exponent(p), d = pc == p ? pl : 0.0;
  const double n = __builtin_rint((pc + d) * c->x[11]);
  double v = exp_reduced(c, n, fma_(-n, c->ln2, pc), fma_(-n, c->ln2_lo, d));
  if (!ordinary(b.x)) v = pow_special(b.x, y, v);
  return v;
}

// log(x^y) from log(x): what log(pow(log(x), y)) gives, without the rounding of the power.
__device__ __forceinline__ Log log_of_pow(const Log& b, double y) {
  const double p = y * b.hi;
  Log r{p, fma_(y, b.lo, fma_(y, b.hi, -p)), b.x};
  if (!ordinary(b.x)) {
    r.x = pow_special(b.x, y, 1.0);
    if (y == 0.0) r.hi = r.lo = 0.0;  // log of infinity or NaN is no number
  }
  return r;
}

}  // namespace fp64
