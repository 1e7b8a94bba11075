// Device helpers shared by the CLOUDSC and CLOUD_SATADJ kernels: FP32/FP64 math on the gfx950 instructions,
// the Tetens saturation functions, CLOUD_SUPERSATCHECK for one point, and 32-bit-offset loads and stores.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include "fp64_math.h"

namespace cloudsc_gpu {

// CLOUDSC_FAST_TRANSCENDENTALS selects all three hardware forms below (exp/pow/log, division, square root);
// CLOUDSC_FAST_EXP, CLOUDSC_FAST_DIV and CLOUDSC_FAST_SQRT select them one by one.
#ifdef CLOUDSC_FAST_TRANSCENDENTALS
#define CLOUDSC_FAST_EXP
#define CLOUDSC_FAST_DIV
#define CLOUDSC_FAST_SQRT
#endif
#ifdef CLOUDSC_FAST_EXP
// FP32 exp and pow on the hardware base-2 instructions (v_exp_f32, v_log_f32):
// exp(x) = 2^(x log2 e), pow(x,y) = 2^(y log2 x).  Relative error ~ (1 + |y log2 x|) ulp.
__device__ __forceinline__ float m_exp(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }
__device__ __forceinline__ float m_pow(float x, float y) { return __builtin_amdgcn_exp2f(y * __builtin_amdgcn_logf(x)); }
__device__ __forceinline__ float m_log(float x) { return __builtin_amdgcn_logf(x) * 0.6931471805599453f; }
#else
__device__ __forceinline__ float m_exp(float x) { return expf(x); }
__device__ __forceinline__ float m_pow(float x, float y) { return powf(x, y); }
__device__ __forceinline__ float m_log(float x) { return logf(x); }
#endif
__device__ __forceinline__ double m_exp(double x) { return exp(x); }
__device__ __forceinline__ double m_pow(double x, double y) { return pow(x, y); }
__device__ __forceinline__ double m_log(double x) { return log(x); }
// The CLOUDSC sweep's exponentials and powers: FP32 as above, FP64 by the table functions, which suit a kernel that runs
// one or two waves to a SIMD (the point kernels, with 3 and more waves, are 2 to 4 % slower with them).
// s_pow(s_base(x), y) = x^y, and s_base_pow(b, y) is the base x^y: in FP64 the logarithm, two thirds of a power, is taken
// once for several powers of a base, and a power that only serves as a base not at all; FP32's is two instructions,
// which the compiler shares by itself.
struct Base32 {
  float x;
};
__device__ __forceinline__ float s_exp(float x) { return m_exp(x); }
__device__ __forceinline__ Base32 s_base(float x) { return Base32{x}; }
__device__ __forceinline__ float s_pow(Base32 b, float y) { return m_pow(b.x, y); }
__device__ __forceinline__ Base32 s_base_pow(Base32 b, float y) { return Base32{m_pow(b.x, y)}; }
__device__ __forceinline__ float s_pow15(float x) { return m_pow(x, 1.5f); }
__device__ __forceinline__ double s_exp(double x) { return fp64::exp(x); }
__device__ __forceinline__ fp64::Log s_base(double x) { return fp64::log(x); }
__device__ __forceinline__ double s_pow(const fp64::Log& b, double y) { return fp64::pow(b, y); }
__device__ __forceinline__ fp64::Log s_base_pow(const fp64::Log& b, double y) { return fp64::log_of_pow(b, y); }
__device__ __forceinline__ double s_pow15(double x) { return x * sqrt(x); }
template <typename R>
__device__ __forceinline__ R s_pow(R x, R y) { return s_pow(s_base(x), y); }
#ifdef CLOUDSC_FAST_DIV
// FP32 division as reciprocal (v_rcp_f32, 1 ulp) times numerator instead of the ~10-instruction
// IEEE sequence.  Measured against the FP64 oracle on 8192 L137 columns, the FP32 kernel's
// relative RMS error per output field stays within 7% of the IEEE build's (both are dominated
// by FP32 threshold flips, not by the last bit of a quotient).  FP64 keeps IEEE division.
__device__ __forceinline__ float m_div(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
#else
__device__ __forceinline__ float m_div(float a, float b) { return a / b; }
#endif
__device__ __forceinline__ double m_div(double a, double b) { return a / b; }
// Quotients that are exactly 1, or exactly the numerator's factor, when the denominator is the numerator's own
// sum or factor (the liquid share of the condensate, the rain share of the precipitation, the precipitation
// cover's overlap factor when the cloud cover does not grow): IEEE division.  a * rcp(a) can be 1 - 2^-24
// instead, which leaves a share of ~6e-8 to the other phase and switches on its processes.
template <typename T>
__device__ __forceinline__ T m_share(T a, T b) { return a / b; }
#ifdef CLOUDSC_FAST_SQRT
// square roots occur only inside rate expressions: v_sqrt_f32 (1 ulp)
__device__ __forceinline__ float m_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
#else
__device__ __forceinline__ float m_sqrt(float x) { return sqrtf(x); }
#endif
__device__ __forceinline__ double m_sqrt(double x) { return sqrt(x); }
// MAX/MIN on v_max/v_min (identical to the Fortran intrinsics for non-NaN arguments)
__device__ __forceinline__ float m_max(float a, float b) { return __builtin_fmaxf(a, b); }
__device__ __forceinline__ float m_min(float a, float b) { return __builtin_fminf(a, b); }
__device__ __forceinline__ double m_max(double a, double b) { return __builtin_fmax(a, b); }
__device__ __forceinline__ double m_min(double a, double b) { return __builtin_fmin(a, b); }
template <typename T>
__device__ __forceinline__ T m_abs(T a) { return a < T(0) ? -a : a; }

// Tetens saturation vapour pressures (fcttre.func.h:84-93,165-166).
template <typename T>
struct Sat {
  T alfa, el, ei;  // FOEALFA, EXP(R3LES*(T-RTT)/(T-R4LES)), EXP(R3IES*(T-RTT)/(T-R4IES))
};
template <typename T, typename KCT, bool SWEEP = false>
__device__ __forceinline__ Sat<T> saturation(const KCT& c, T t) {
  Sat<T> s;
  T x = (m_max(c.rtice, m_min(c.rtwat, t)) - c.rtice) * c.rtwat_rtice_r;
  s.alfa = m_min(T(1), x * x);
  const T xl = m_div(c.r3les * (t - c.rtt), t - c.r4les), xi = m_div(c.r3ies * (t - c.rtt), t - c.r4ies);
  s.el = SWEEP ? s_exp(xl) : m_exp(xl);
  s.ei = SWEEP ? s_exp(xi) : m_exp(xi);
  return s;
}

// CLOUD_SUPERSATCHECK for one point, KFTLIQICE = 1 (cloud_supersatcheck.F90:111-226).  SHARE (FP64 inside an FP32
// point, whose result is rounded to FP32): the quotients by the two temperature differences and by the two saturation
// denominators from one division each.
template <typename T, typename KCT, bool SWEEP = false, bool SHARE = false>
__device__ __forceinline__ void supersatcheck(const KCT& c, T pt, T pq, T pa, T pp, T& t_adj, T& q_adj,
                                              T& a_adj, T& l_adj, T& i_adj) {
  const T zepsec = T(1.e-14);
  T zda = T(0);
  T zt = m_max(pt, T(160));
  T za = m_max(m_min(pa, T(1)), T(0));
  const T zp_r = m_div(T(1), pp);
  const T dl = zt - c.r4les, di = zt - c.r4ies;
  Sat<T> s;
  T fl, fi;  // 1 / dl^2, 1 / di^2
  if constexpr (SHARE) {
    const T w = m_div(T(1), dl * di), rl = w * di, ri = w * dl;
    const T x = (m_max(c.rtice, m_min(c.rtwat, zt)) - c.rtice) * c.rtwat_rtice_r;
    s.alfa = m_min(T(1), x * x);
    s.el = m_exp(c.r3les * (zt - c.rtt) * rl);
    s.ei = m_exp(c.r3ies * (zt - c.rtt) * ri);
    fl = rl * rl, fi = ri * ri;
  } else {
    s = saturation<T, KCT, SWEEP>(c, zt);
    fl = m_div(T(1), dl * dl), fi = m_div(T(1), di * di);
  }
  const T foeeliq = c.r2es * s.el;
  const T zfoeeliq = m_min(foeeliq * zp_r, T(0.5));
  // FOEEW: water above RTT, ice below (FOEDELTA = MAX(0,SIGN(1,T-RTT)))
  const T foeew = (zt - c.rtt >= T(0)) ? c.r2es * s.el : c.r2es * s.ei;
  const T zfoeeice = m_min(foeew * zp_r, T(0.5));
  const T zfokoop = m_min(zfoeeice * (c.rkoop1 - c.rkoop2 * zt), zfoeeliq);
  const T zfoeemix = m_min(c.r2es * (s.alfa * s.el + (T(1) - s.alfa) * s.ei) * zp_r, T(0.5));
  const T dk = T(1) - c.retv * zfokoop, dm = T(1) - c.retv * zfoeemix;
  T zqsliqk, zcor;
  if constexpr (SHARE) {
    const T w = m_div(T(1), dk * dm);
    zqsliqk = zfokoop * (w * dm);
    zcor = w * dk;
  } else {
    zqsliqk = m_div(zfokoop, dk);
    zcor = m_div(T(1), dm);
  }
  const T zqsmix = zfoeemix * zcor;
  const T foedem = s.alfa * c.r5alvcp * fl + (T(1) - s.alfa) * c.r5alscp * fi;
  const T zcorqsmix = T(1) + zqsmix * zcor * foedem;
  zqsliqk = T(0.5) * (zqsliqk + zqsmix);
  T zqslim = za * zqsmix + (T(1) - za) * zqsliqk;
  T zcond = m_max(pq - zqslim, T(0));
  if (zcond > zepsec) {
    const T zfaci = s.alfa + (T(1) - s.alfa) * c.rssicefactor;
    zda = (T(1) - za) * zfaci;
    const T za_upd = za + zda;
    zqslim = za_upd * zqsmix + (T(1) - za_upd) * zqsliqk;
    zcond = m_div(pq - zqslim, zcorqsmix);
  }
  const T foeldcpm = s.alfa * c.ralvdcp + (T(1) - s.alfa) * c.ralsdcp;
  t_adj = foeldcpm * zcond;
  q_adj = -zcond;
  a_adj = zda;
  l_adj = zcond * s.alfa;
  i_adj = zcond * (T(1) - s.alfa);
}

// Loads and stores at 32-bit byte offsets from an array base: the form the hardware
// addresses directly (64-bit base in SGPRs, 32-bit offset in one VGPR).  The launcher
// splits the grid so that every array of one launch spans less than 4 GiB.
// u: byte offset common to the wave (block and level); v: the lane's byte offset within the level.  The sum is
// formed in 32 bits, so every array access is one vector offset on a scalar base; with wave-uniform blocks
// (NPROMA a multiple of 64) u is a scalar and the block-dependent offsets cost no vector registers.
// The casts to the global address space (1) keep the scalar-base form also for bases the compiler cannot trace to a
// kernel argument.
template <typename T>
__device__ __forceinline__ T LD(const T* base, uint32_t u, uint32_t v) {
  typedef const __attribute__((address_space(1))) char gchar;
  typedef const __attribute__((address_space(1))) T gT;
  return *(gT*)((gchar*)base + (u + v));
}
template <typename T>
__device__ __forceinline__ void ST(T* base, uint32_t u, uint32_t v, T x) {
  typedef __attribute__((address_space(1))) char gchar;
  typedef __attribute__((address_space(1))) T gT;
  *(gT*)((gchar*)base + (u + v)) = x;
}

// The same with the non-temporal hint where NT: fields that a sweep reads or writes once, in whole lines.  Rows that share
// a line with the next wave's (NPROMA no multiple of 64) keep the plain form: there the hint drops lines that are
// needed again (FP32 40,007 x L91 in blocks of 100: 375 us without, 398 us with it, 131,072 x L137 1.47 and 1.72 ms; mixed
// 655,360 x L137 in blocks of 128: 3.82 ms without, 3.76 ms with it).  Blocks of 32 have whole lines in FP32, but gain
// nothing from it (66,000 to 200,000 columns within 2.5 % either way).
template <bool NT, typename T>
__device__ __forceinline__ T LDN(const T* base, uint32_t u, uint32_t v) {
  typedef const __attribute__((address_space(1))) char gchar;
  typedef const __attribute__((address_space(1))) T gT;
  if constexpr (NT) return __builtin_nontemporal_load((gT*)((gchar*)base + (u + v)));
  return *(gT*)((gchar*)base + (u + v));
}
template <bool NT, typename T>
__device__ __forceinline__ void STN(T* base, uint32_t u, uint32_t v, T x) {
  typedef __attribute__((address_space(1))) char gchar;
  typedef __attribute__((address_space(1))) T gT;
  if constexpr (NT)
    __builtin_nontemporal_store(x, (gT*)((gchar*)base + (u + v)));
  else
    *(gT*)((gchar*)base + (u + v)) = x;
}

// Work-group number -> position in the grid.  The dispatcher deals consecutive work-groups to the 8 XCDs in turn; here
// each XCD takes one contiguous eighth of the columns, so the groups that run together on it share the pages (and, in
// ragged blocks, the lines) of the ~50 field arrays.  A bijection for every grid size; the first XCDs have a group more
// where the number is no multiple of 8, so a grid had better hold no group without work (the sweep's launcher sees to it).
__host__ __device__ __forceinline__ uint32_t xcd_group(uint32_t id, uint32_t n) {
  const uint32_t x = id & 7u, r = n & 7u;
  return x * (n >> 3) + (x < r ? x : r) + (id >> 3);
}

}  // namespace cloudsc_gpu
