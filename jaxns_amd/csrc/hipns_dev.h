// hipns_dev.h -- device helpers shared by the gfx950 kernels of libhipns.
//
// Wavefront-64 idioms, the Philox4x32-10 counter PRNG, the inverse normal
// CDF used by the prior transform, FP64 numbers of any magnitude and the
// composition algebra of the evidence recurrence.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hipns.h"

#define HIPNS_WAVE 64

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

namespace hipns {

__device__ __forceinline__ int lane_id() { return (int)__lane_id(); }

// ---------------------------------------------------------------------------
// cross-lane reductions among the LPC lanes that share one chain.  Lane l
// serves chain (l % CW) with part h = l / CW, CW = 64 / LPC, so partners are
// at xor distances CW, 2 CW, ...
// ---------------------------------------------------------------------------
// gfx950 lane swaps: permlane16_swap exchanges the odd 16-lane rows of its
// first operand with the even rows of its second, permlane32_swap the upper
// half of the first with the lower half of the second.  Called with the same
// value twice, the two results hold the two partners of every lane, so
// r[0] (op) r[1] is the reduction over lanes l and l^16 (resp. l^32), with the
// operands in the same order on both partners.
__device__ __forceinline__ void swap16(float v, float& a, float& b) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap32(float v, float& a, float& b) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}

// the value of lane l ^ 8 (LPC = 8: the partner 8 lanes away, inside the same 16-lane row): a DPP
// row rotation by 8
__device__ __forceinline__ uint32_t xor8(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xF, 0xF, false);  // row_ror:8
}
__device__ __forceinline__ float xor8f(float v) { return __uint_as_float(xor8(__float_as_uint(v))); }

// value of lane part `part` (wavefront-uniform) of this lane's chain, on every part of the chain:
// r[0] / r[1] of a swap are the values of the lower / upper partner
template <int LPC>
__device__ __forceinline__ uint32_t part_broadcast(uint32_t v, int part) {
  auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  if constexpr (LPC == 8) {
    v = (part & 4) ? r[1] : r[0];
    auto q = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = (part & 2) ? q[1] : q[0];
    // bit 0 of the part is bit 3 of the lane: keep this lane's value where they agree, else the
    // partner's
    const uint32_t x = xor8(v);
    return (((lane_id() >> 3) & 1) == (part & 1)) ? v : x;
  } else if constexpr (LPC == 4) {
    v = (part & 2) ? r[1] : r[0];
    auto q = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return (part & 1) ? q[1] : q[0];
  }
  return part ? r[1] : r[0];
}

// reductions over the LPC lanes of a chain; with a commutative operation the partners compute the
// same value (a + b = b + a in IEEE arithmetic)
template <int LPC>
__device__ __forceinline__ float chain_sum(float v) {
  float a, b;
  if constexpr (LPC == 8) v = v + xor8f(v);
  if constexpr (LPC >= 4) {
    swap16(v, a, b);
    v = a + b;
  }
  swap32(v, a, b);
  return a + b;
}
template <int LPC>
__device__ __forceinline__ float chain_min(float v) {
  float a, b;
  if constexpr (LPC == 8) v = fminf(v, xor8f(v));
  if constexpr (LPC >= 4) {
    swap16(v, a, b);
    v = fminf(a, b);
  }
  swap32(v, a, b);
  return fminf(a, b);
}
template <int LPC>
__device__ __forceinline__ float chain_max(float v) {
  float a, b;
  if constexpr (LPC == 8) v = fmaxf(v, xor8f(v));
  if constexpr (LPC >= 4) {
    swap16(v, a, b);
    v = fmaxf(a, b);
  }
  swap32(v, a, b);
  return fmaxf(a, b);
}

// ---------------------------------------------------------------------------
// a / n rounded to nearest without the operand scaling of the general IEEE division: y = RN(1/n) from
// the hardware reciprocal and one Newton step, then one residual correction of q = a y.  With y the
// correctly rounded reciprocal and q within an ulp of a / n, r = a - n q is exact and RN(q + r y) =
// RN(a / n) (P. Markstein, IBM J. Res. Dev. 34(1), 1990).  y = RN(1/n) holds for every |n| in
// [2^-94, 1] (checked exhaustively on the device); for |a| in [2^-60, 2] nothing under- or overflows,
// so the quotient is bit-identical to a / n.  n = +-0 yields NaN (where a / n is +-inf): both say "no
// bound from this slot".
__device__ __forceinline__ float recip_rn(float n) {
  const float y = __builtin_amdgcn_rcpf(n);
  const float e = fmaf(-n, y, 1.0f);
  return fmaf(e, y, y);
}
__device__ __forceinline__ float quot_rn(float a, float n, float y) {
  const float q = a * y;
  const float r = fmaf(-n, q, a);
  return fmaf(r, y, q);
}

// ---------------------------------------------------------------------------
// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11): 10 rounds of the
// multiply-xor bijection with Weyl key schedule.
// ---------------------------------------------------------------------------
struct u32x4 {
  uint32_t x, y, z, w;
};

__device__ __forceinline__ u32x4 philox4x32(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0,
                                            uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    // one 32x32 -> 64-bit product per multiplier gives both halves of mulhilo
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
    const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
    const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
    uint32_t n0 = hi1 ^ c1 ^ k0;
    uint32_t n2 = hi0 ^ c3 ^ k1;
    c0 = n0;
    c1 = lo1;
    c2 = n2;
    c3 = lo0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return {c0, c1, c2, c3};
}

// uniform in [0,1) with 24 random bits
__device__ __forceinline__ float u01f(uint32_t w) { return (float)(w >> 8) * 5.9604644775390625e-8f; }
// uniform in (0,1]
__device__ __forceinline__ float u01f_open0(uint32_t w) { return (float)((w >> 8) + 1u) * 5.9604644775390625e-8f; }
// uniform in [0,1) with 53 random bits
__device__ __forceinline__ double u01d(uint32_t a, uint32_t b) {
  uint64_t v = (((uint64_t)a << 21) ^ (uint64_t)(b >> 11)) & ((1ull << 53) - 1);
  return (double)v * (1.0 / 9007199254740992.0);
}

// counter-domain tags (word 3 of the Philox counter)
enum : uint32_t {
  RNG_SEED = 0u << 24,
  RNG_DIR = 1u << 24,
  RNG_PICK = 2u << 24,
  RNG_UNIF = 3u << 24,
  RNG_DIR2 = 4u << 24,  // the angle uniforms of the slice directions
};

// ---------------------------------------------------------------------------
// Inverse standard-normal CDF.
//  - binary64: Wichura, Algorithm AS 241 (Applied Statistics 37, 1988), PPND16.
//  - binary32: M. Giles, "Approximating the erfinv function" (GPU Computing
//    Gems Jade, 2011), single-precision polynomials in w = -log(4u(1-u)),
//    evaluated directly in u so that both tails keep relative accuracy;
//    |u - 1/2| > 1/2 - 1e-7 falls back to PPND16.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double ndtri_f64(double p) {
  if (!(p > 0.0 && p < 1.0)) {
    if (p == 0.0) return -__builtin_inf();
    if (p == 1.0) return __builtin_inf();
    return __builtin_nan("");
  }
  double q = p - 0.5;
  if (fabs(q) <= 0.425) {
    double r = 0.180625 - q * q;
    double num = 2.5090809287301226727e+3;
    num = num * r + 3.3430575583588128105e+4;
    num = num * r + 6.7265770927008700853e+4;
    num = num * r + 4.5921953931549871457e+4;
    num = num * r + 1.3731693765509461125e+4;
    num = num * r + 1.9715909503065514427e+3;
    num = num * r + 1.3314166789178437745e+2;
    num = num * r + 3.3871328727963666080e0;
    double den = 5.2264952788528545610e+3;
    den = den * r + 2.8729085735721942674e+4;
    den = den * r + 3.9307895800092710610e+4;
    den = den * r + 2.1213794301586595867e+4;
    den = den * r + 5.3941960214247511077e+3;
    den = den * r + 6.8718700749205790830e+2;
    den = den * r + 4.2313330701600911252e+1;
    den = den * r + 1.0;
    return q * num / den;
  }
  double r = q < 0.0 ? p : 1.0 - p;
  r = sqrt(-log(r));
  double num, den;
  if (r <= 5.0) {
    r -= 1.6;
    num = 7.74545014278341407640e-4;
    num = num * r + 2.27238449892691845833e-2;
    num = num * r + 2.41780725177450611770e-1;
    num = num * r + 1.27045825245236838258e0;
    num = num * r + 3.64784832476320460504e0;
    num = num * r + 5.76949722146069140550e0;
    num = num * r + 4.63033784615654529590e0;
    num = num * r + 1.42343711074968357734e0;
    den = 1.05075007164441684324e-9;
    den = den * r + 5.47593808499534494600e-4;
    den = den * r + 1.51986665636164571966e-2;
    den = den * r + 1.48103976427480074590e-1;
    den = den * r + 6.89767334985100004550e-1;
    den = den * r + 1.67638483018380384940e0;
    den = den * r + 2.05319162663775882187e0;
    den = den * r + 1.0;
  } else {
    r -= 5.0;
    num = 2.01033439929228813265e-7;
    num = num * r + 2.71155556874348757815e-5;
    num = num * r + 1.24266094738807843860e-3;
    num = num * r + 2.65321895265761230930e-2;
    num = num * r + 2.96560571828504891230e-1;
    num = num * r + 1.78482653991729133580e0;
    num = num * r + 5.46378491116411436990e0;
    num = num * r + 6.65790464350110377720e0;
    den = 2.04426310338993978564e-15;
    den = den * r + 1.42151175831644588870e-7;
    den = den * r + 1.84631831751005468180e-5;
    den = den * r + 7.86869131145613259100e-4;
    den = den * r + 1.48753612908506148525e-2;
    den = den * r + 1.36929880922735805310e-1;
    den = den * r + 5.99832206555887937690e-1;
    den = den * r + 1.0;
  }
  double v = num / den;
  return q < 0.0 ? -v : v;
}

__device__ __noinline__ float ndtri_tail_f32(float u) { return (float)ndtri_f64((double)u); }

// Giles' body for u in [1e-7, 1 - 1e-7].  w = -ln(4u(1-u)) comes from the hardware log2 (one
// rounding more than a full-precision log: about 1e-7 relative in w, below the polynomials' own error).
// The w >= 5 polynomial runs only when some lane of the wavefront needs it.
__device__ __forceinline__ float giles_w(float u) {
  return -0.693147180559945309f * __builtin_amdgcn_logf(4.0f * u * (1.0f - u));
}
__device__ __forceinline__ float giles_x(float u) {
  return fmaf(u, 2.82842712474619010f, -1.41421356237309505f);  // sqrt(2) (2u - 1), one rounding
}
// the central polynomial (w < 5)
__device__ __forceinline__ float giles_central(float w) {
  const float z = w - 2.5f;
  float p = 2.81022636e-08f;
  p = fmaf(p, z, 3.43273939e-07f);
  p = fmaf(p, z, -3.5233877e-06f);
  p = fmaf(p, z, -4.39150654e-06f);
  p = fmaf(p, z, 0.00021858087f);
  p = fmaf(p, z, -0.00125372503f);
  p = fmaf(p, z, -0.00417768164f);
  p = fmaf(p, z, 0.246640727f);
  p = fmaf(p, z, 1.50140941f);
  return p;
}
// the tail polynomial (w >= 5)
__device__ __forceinline__ float giles_tail(float w) {
  const float v = __builtin_amdgcn_sqrtf(w) - 3.0f;
  float pt = -0.000200214257f;
  pt = fmaf(pt, v, 0.000100950558f);
  pt = fmaf(pt, v, 0.00134934322f);
  pt = fmaf(pt, v, -0.00367342844f);
  pt = fmaf(pt, v, 0.00573950773f);
  pt = fmaf(pt, v, -0.0076224613f);
  pt = fmaf(pt, v, 0.00943887047f);
  pt = fmaf(pt, v, 1.00167406f);
  pt = fmaf(pt, v, 2.83297682f);
  return pt;
}

__device__ __forceinline__ float ndtri_giles(float u) {
  const float w = giles_w(u);
  const float x = giles_x(u);
  float p = giles_central(w);
  const bool tl = w >= 5.0f;
  if (__any(tl)) p = tl ? giles_tail(w) : p;
  return p * x;
}

// u far in the tails (min(u, 1 - u) < 1e-7) or outside (0, 1): binary64 AS 241
__device__ __forceinline__ bool ndtri_far(float u) { return !(u >= 1e-7f && u <= 0.9999999f); }

__device__ __forceinline__ float ndtri_f32(float u) {
  float z = ndtri_giles(u);
  if (ndtri_far(u)) z = ndtri_tail_f32(u);
  return z;
}

// ---------------------------------------------------------------------------
// Non-negative FP64 numbers of any magnitude: m 2^e, the exponent a whole-valued double.  The evidence
// recurrence multiplies and adds quantities far outside the range of a double (likelihoods of e^-1e10,
// volumes of e^-1000).  Held as logarithms every sum is an exp and a log1p (about 75 FP64 instructions);
// held like this it is two shifts and an add.
// Zero has exponent -inf (so it never sets the scale of a sum); +inf and NaN live in m.
// ---------------------------------------------------------------------------
struct Sc {
  double m, e;
};

__device__ __forceinline__ Sc sc_zero() { return {0.0, -__builtin_inf()}; }

__device__ __forceinline__ Sc sc_mul(const Sc& x, const Sc& y) { return {x.m * y.m, x.e + y.e}; }
__device__ __forceinline__ Sc sc_scale(const Sc& x, double c) { return {x.m * c, x.e}; }

// a difference of exponents as a shift: saturating, NaN to 0.  That is the instruction's own rule; a cast is
// undefined for both, and a compiler that knows the operand may take any value.
__device__ __forceinline__ int sc_shift(double d) {
  int r;
  asm("v_cvt_i32_f64 %0, %1" : "=v"(r) : "v"(d));
  return r;
}

// both mantissas shifted to the larger exponent (a saturated shift gives zero; two zeros have a NaN difference)
__device__ __forceinline__ Sc sc_add(const Sc& x, const Sc& y) {
#pragma clang fp contract(off)
  const double e = fmax(x.e, y.e);
  return {__builtin_amdgcn_ldexp(x.m, sc_shift(x.e - e)) + __builtin_amdgcn_ldexp(y.m, sc_shift(y.e - e)), e};
}

// m in [1/2, 1)
__device__ __forceinline__ Sc sc_norm(const Sc& x) {
  return {__builtin_amdgcn_frexp_mant(x.m), x.e + (double)__builtin_amdgcn_frexp_exp(x.m)};
}

// e^L.  L = k ln 2 + r with k whole and |r| <= ln(2) / 2, e^r by its Taylor series (the first term left out
// is below 2^-53).  Beyond 2^52 a double no longer separates L from its neighbours by less than one, and r
// only has to stay bounded.
__device__ __forceinline__ Sc sc_exp(double L) {
  constexpr double LOG2E = 1.4426950408889634074, LN2_HI = 0.69314718055994530942, LN2_LO = 2.3190468138462996e-17;
  const double k = rint(L * LOG2E);
  double r = fma(-k, LN2_LO, fma(-k, LN2_HI, L));
  r = fmin(fmax(r, -0.35), 0.35);
  double p = 1.0 / 6227020800.0;
  p = fma(p, r, 1.0 / 479001600.0);
  p = fma(p, r, 1.0 / 39916800.0);
  p = fma(p, r, 1.0 / 3628800.0);
  p = fma(p, r, 1.0 / 362880.0);
  p = fma(p, r, 1.0 / 40320.0);
  p = fma(p, r, 1.0 / 5040.0);
  p = fma(p, r, 1.0 / 720.0);
  p = fma(p, r, 1.0 / 120.0);
  p = fma(p, r, 1.0 / 24.0);
  p = fma(p, r, 1.0 / 6.0);
  p = fma(p, r, 0.5);
  p = fma(p, r, 1.0);
  p = fma(p, r, 1.0);
  // -inf, +inf and NaN
  if (!(fabs(L) < __builtin_inf())) return L < 0.0 ? sc_zero() : Sc{L, 0.0};
  return {p, k};
}

// ln(m 2^e) = ln f + k ln 2 with f in [sqrt(1/2), sqrt(2)), ln f = 2 artanh((f - 1) / (f + 1)) by its power
// series (|s| < 0.172: the first term left out is below 2^-54 of the sum).  About two thirds of the
// instructions of the library's log; m is never negative here.
__device__ __forceinline__ double sc_log(const Sc& x) {
  const double f0 = __builtin_amdgcn_frexp_mant(x.m);
  const bool low = f0 < 0.70710678118654752440;
  const double f = low ? f0 + f0 : f0;
  const double k = x.e + (double)(__builtin_amdgcn_frexp_exp(x.m) - (low ? 1 : 0));
  const double num = f - 1.0, den = f + 1.0;
  double y = __builtin_amdgcn_rcp(den);
  y = fma(fma(-den, y, 1.0), y, y);
  y = fma(fma(-den, y, 1.0), y, y);
  double s = num * y;
  s = fma(fma(-den, s, num), y, s);
  const double t = s * s;
  double p = 2.0 / 21.0;
  p = fma(p, t, 2.0 / 19.0);
  p = fma(p, t, 2.0 / 17.0);
  p = fma(p, t, 2.0 / 15.0);
  p = fma(p, t, 2.0 / 13.0);
  p = fma(p, t, 2.0 / 11.0);
  p = fma(p, t, 2.0 / 9.0);
  p = fma(p, t, 2.0 / 7.0);
  p = fma(p, t, 2.0 / 5.0);
  p = fma(p, t, 2.0 / 3.0);
  const double lf = fma(s * t, p, s + s);
  // (zero has k = -inf)
  return x.m == __builtin_inf() ? x.m : fma(k, 0.69314718055994530942, lf);
}

// The same with an unevaluated low part, for the long products of the recurrence: X is a product of up to
// millions of n / (n + 1), and the rounding of a factor that repeats would add up.
struct Scd {
  double m, lo, e;
};

__device__ __forceinline__ Scd scd_zero() { return {0.0, 0.0, -__builtin_inf()}; }
__device__ __forceinline__ Sc sc_of(const Scd& x) { return {x.m, x.e}; }

// x (t + tl), mantissa not renormalised
__device__ __forceinline__ Scd scd_scale(const Scd& x, double t, double tl) {
#pragma clang fp contract(off)
  const double p = x.m * t;
  return {p, fma(x.m, t, -p) + fma(x.m, tl, x.lo * t), x.e};
}
// low part below half an ulp of the high part, m in [1/2, 1)
__device__ __forceinline__ Scd scd_norm(const Scd& x) {
#pragma clang fp contract(off)
  const double s = x.m + x.lo;
  const double lo = x.lo - (s - x.m);
  const int k = __builtin_amdgcn_frexp_exp(s);
  return {__builtin_amdgcn_frexp_mant(s), __builtin_amdgcn_ldexp(lo, -k), x.e + (double)k};
}
__device__ __forceinline__ Scd scd_mul(const Scd& x, const Scd& y) {
  Scd r = scd_scale(x, y.m, y.lo);
  r.e += y.e;
  return scd_norm(r);
}

// ---------------------------------------------------------------------------
// Evidence recurrence as composable maps.
//
// One _update_evidence_calc_op step (internals/shrinkage_statistics.py:43-94)
// acts on (X, X2, Z, ZX, Z2, dZ2) (all >= 0) as
//   X'  = T X                 X2' = T2 X2
//   Z'  = Z  + (t m) X        ZX' = T ZX + (tT m) X2
//   Z2' = Z2 + (2 t m) ZX + (t2 m^2) X2
//   dZ2'= dZ2 + (t2 m^2) X2
// with T=n/(n+1), t=1/(n+1), T2=n/(n+2), t2=2/((n+1)(n+2)), tT=n/((n+1)(n+2)),
// m = (L_prev + L)/2.  With Q = X2 / X and Y = ZX / X, w = t m X (the step's dZ) and
// y = m Q / (n+2) it is
//   X' = T X,  Q' = (n+1)/(n+2) Q,  Z' = Z + w,  Y' = Y + y,  Z2' = Z2 + 2 w Y',  dZ2' = dZ2 + 2 w y:
// two products and four sums, and nothing decays but X and Q.  A sequence of steps is a map
//   X'=aX, Q'=bQ, Z'=Z+gX, Y'=Y+cQ, Z2'=Z2+2gXY+hXQ, dZ2'=dZ2+kXQ,
// closed under composition, so the scan over samples is a prefix scan of 6-coefficient maps.  The
// coefficients of a map are also the state that it takes (1, 1, 0, 0, 0, 0) to, so a sequence of steps
// composes by stepping that state.
// ---------------------------------------------------------------------------
struct EvState {
  Scd X, Q;
  Sc Z, Y, Z2, dZ2;
};
struct EvMap {
  Scd a, b;
  Sc g, c, h, k;
};

__device__ __forceinline__ EvMap evmap_identity() {
  return {{1.0, 0.0, 0.0}, {1.0, 0.0, 0.0}, sc_zero(), sc_zero(), sc_zero(), sc_zero()};
}
__device__ __forceinline__ EvState evstate_initial() {
  return {{1.0, 0.0, 0.0}, {1.0, 0.0, 0.0}, sc_zero(), sc_zero(), sc_zero(), sc_zero()};
}
__device__ __forceinline__ EvState evstate_of(const EvMap& f) { return {f.a, f.b, f.g, f.c, f.h, f.k}; }
// with every mantissa back in [1/2, 1)
__device__ __forceinline__ EvMap evmap_of(const EvState& s) {
  return {scd_norm(s.X), scd_norm(s.Q), sc_norm(s.Z), sc_norm(s.Y), sc_norm(s.Z2), sc_norm(s.dZ2)};
}

// the coefficients of one step that depend on the live-point count n alone.  A count with no logarithm
// gives NaN, as in the reference.
struct EvCoef {
  double n, T, Tl, R, Rl, t, i2;  // T and R = (n+1)/(n+2) with their low parts, t = 1/(n+1), i2 = 1/(n+2)
};
__device__ __forceinline__ EvCoef evcoef(double n) {
  const double n1 = n + 1.0, n2 = n + 2.0;
  const double i1 = 1.0 / n1, i2 = 1.0 / n2;
  const bool whole = n < __builtin_inf();
  EvCoef c;
  c.n = n;
  c.T = n < 0.0 ? __builtin_nan("") : (n < 1.0 ? n * i1 : 1.0 - i1);
  c.Tl = whole ? fma(-c.T, n1, n) * i1 : 0.0;
  c.R = 1.0 - i2;
  c.Rl = whole ? fma(-c.R, n2, n1) * i2 : 0.0;
  c.t = n1 < 0.0 ? __builtin_nan("") : i1;
  c.i2 = n2 < 0.0 ? __builtin_nan("") : i2;
  return c;
}
// the coefficients of n, formed again only when n differs from the cached step's (runs of equal n
// are the rule: a shell's discarded samples all have n = N); the values are those of evcoef(n)
__device__ __forceinline__ const EvCoef& evcoef_cached(EvCoef& c, double n) {
  if (!(c.n == n)) c = evcoef(n);
  return c;
}
__device__ __forceinline__ EvCoef evcoef_empty() {
  EvCoef c;
  c.n = __builtin_nan("");
  c.T = c.Tl = c.R = c.Rl = c.t = c.i2 = 0.0;
  return c;
}

// m = (L_prev + L) / 2 of a step
__device__ __forceinline__ Sc ev_mid(const Sc& Lprev, const Sc& L) { return sc_scale(sc_add(L, Lprev), 0.5); }

// one step of the recurrence; returns dZ = t m X
__device__ __forceinline__ Sc ev_step(EvState& s, const EvCoef& c, const Sc& mid) {
  Sc w = {c.t * mid.m * s.X.m, mid.e + s.X.e};
  Sc y = {c.i2 * mid.m * s.Q.m, mid.e + s.Q.e};
  if (c.t == 0.0) w = y = sc_zero();  // an infinite count
  const Sc w2 = sc_scale(w, 2.0);
  s.Z = sc_add(s.Z, w);
  s.Y = sc_add(s.Y, y);
  s.Z2 = sc_add(s.Z2, sc_mul(w2, s.Y));
  s.dZ2 = sc_add(s.dZ2, sc_mul(w2, y));
  s.X = scd_scale(s.X, c.T, c.Tl);
  s.Q = scd_scale(s.Q, c.R, c.Rl);
  // counts below one shrink X by more than half a step: not left to the end of the caller's run of steps
  if (c.T < 0.5) s.X = c.T == 0.0 ? scd_zero() : scd_norm(s.X);
  return w;
}

// f then g
__device__ __forceinline__ EvMap evmap_then(const EvMap& f, const EvMap& g) {
  EvMap r;
  const Sc fa = sc_of(f.a), fb = sc_of(f.b);
  const Sc ga = sc_mul(g.g, fa), fab = sc_mul(fa, fb);
  r.a = scd_mul(f.a, g.a);
  r.b = scd_mul(f.b, g.b);
  r.g = sc_norm(sc_add(f.g, ga));
  r.c = sc_norm(sc_add(f.c, sc_mul(g.c, fb)));
  r.h = sc_norm(sc_add(sc_add(f.h, sc_scale(sc_mul(ga, f.c), 2.0)), sc_mul(g.h, fab)));
  r.k = sc_norm(sc_add(f.k, sc_mul(g.k, fab)));
  return r;
}

__device__ __forceinline__ EvState evmap_apply(const EvMap& f, const EvState& s) {
  return evstate_of(evmap_then({s.X, s.Q, s.Z, s.Y, s.Z2, s.dZ2}, f));
}

// the fields of EvidenceCalculation that a state stands for
__device__ __forceinline__ Sc ev_X2(const EvState& s) { return sc_mul(sc_of(s.X), sc_of(s.Q)); }
__device__ __forceinline__ Sc ev_ZX(const EvState& s) { return sc_mul(sc_of(s.X), s.Y); }

__device__ __forceinline__ Sc sc_shfl_down(const Sc& x, int o) {
  return {__shfl_down(x.m, o, 64), __shfl_down(x.e, o, 64)};
}
__device__ __forceinline__ Sc sc_shfl_up(const Sc& x, int o) { return {__shfl_up(x.m, o, 64), __shfl_up(x.e, o, 64)}; }
__device__ __forceinline__ Scd sc_shfl_down(const Scd& x, int o) {
  return {__shfl_down(x.m, o, 64), __shfl_down(x.lo, o, 64), __shfl_down(x.e, o, 64)};
}
__device__ __forceinline__ Scd sc_shfl_up(const Scd& x, int o) {
  return {__shfl_up(x.m, o, 64), __shfl_up(x.lo, o, 64), __shfl_up(x.e, o, 64)};
}
__device__ __forceinline__ EvMap shfl_down_map(const EvMap& m, int o) {
  return {sc_shfl_down(m.a, o), sc_shfl_down(m.b, o), sc_shfl_down(m.g, o),
          sc_shfl_down(m.c, o), sc_shfl_down(m.h, o), sc_shfl_down(m.k, o)};
}
__device__ __forceinline__ EvMap shfl_up_map(const EvMap& m, int o) {
  return {sc_shfl_up(m.a, o), sc_shfl_up(m.b, o), sc_shfl_up(m.g, o),
          sc_shfl_up(m.c, o), sc_shfl_up(m.h, o), sc_shfl_up(m.k, o)};
}

// linear_to_log_stats (internals/stats.py:55-74)
__device__ __forceinline__ void linear_to_log_stats(double log_f, double log_f2, double* mu, double* var) {
  double fsq = log_f + log_f;
  *mu = fsq - 0.5 * log_f2;
  double s2 = log_f2 - fsq;
  const double eps = 2.220446049250313e-16;
  *var = __builtin_isnan(s2) ? s2 : fmax(s2, eps);
}

// determine_termination for one TerminationCondition (termination.py:67-147)
__device__ __forceinline__ int determine_termination(const hipns_term_cond_t& c, const hipns_run_state_t& r,
                                                     int64_t* reason) {
  int done = 0;
  int64_t why = 0;
  auto set = [&](bool cond, int bit) {
    if (cond) {
      done = 1;
      why += (int64_t)1 << bit;
    }
  };
  if (c.has_max_samples) set((double)r.num_samples_used >= c.max_samples, 0);
  if (c.has_evidence_uncert) {
    double mu, var;
    linear_to_log_stats(r.evidence_calc_with_remaining[3], r.evidence_calc_with_remaining[5], &mu, &var);
    set(var <= c.evidence_uncert * c.evidence_uncert, 1);
  }
  if (c.has_dlogZ) {
    double mu1, v1, mu0, v0;
    linear_to_log_stats(r.evidence_calc_with_remaining[3], r.evidence_calc_with_remaining[5], &mu1, &v1);
    linear_to_log_stats(r.evidence_calc[3], r.evidence_calc[5], &mu0, &v0);
    set((mu1 - mu0) < c.dlogZ, 2);
  }
  if (c.has_ess) {
    double ess = exp((r.evidence_calc_with_remaining[3] + r.evidence_calc_with_remaining[3]) -
                     r.evidence_calc_with_remaining[7]);
    set(ess >= c.ess, 3);
  }
  if (c.has_max_num_likelihood_evaluations)
    set((double)r.num_likelihood_evaluations >= c.max_num_likelihood_evaluations, 4);
  if (c.has_log_L_contour) set(r.log_L_contour >= c.log_L_contour, 5);
  if (c.has_efficiency_threshold) set(r.efficiency < c.efficiency_threshold, 6);
  set(r.plateau != 0, 7);
  if (c.has_rtol) set(r.relative_spread < c.rtol, 8);
  if (c.has_atol) set(r.absolute_spread < c.atol, 9);
  set(r.no_seed_points != 0, 10);
  if (c.has_peak_XL_frac) {
    double log_XL = r.evidence_calc[1] + r.evidence_calc[0];
    set(log_XL < r.peak_log_XL + log(c.peak_XL_frac), 11);
  }
  *reason = why;
  return done;
}

// First index of `count` entries appended to a sample collection of `size` entries at `next`
// (_add_samples_to_state, sharded_static.py:40-85, through replace_index, internals/maps.py:15-25):
// lax.dynamic_update_slice clamps its start so that the update stays in bounds, so an append that
// would run past the end is shifted back to end at `size` (it overwrites the entries before it) rather
// than wrapped.  `next` itself wraps modulo `size` afterwards.
__host__ __device__ __forceinline__ int64_t append_start(int64_t next, int64_t count, int64_t size) {
  const int64_t last = size - count;
  return next < last ? next : (last > 0 ? last : 0);
}

// key order of a stable FP64 sort: (key, index) lexicographic with NaN last
__device__ __forceinline__ bool key_lt(double ka, int ia, double kb, int ib) {
  bool na = __builtin_isnan(ka), nb = __builtin_isnan(kb);
  if (na || nb) {
    if (na && nb) return ia < ib;
    return nb;  // a < NaN
  }
  return (ka < kb) || (ka == kb && ia < ib);
}
// strict key order ignoring indices (NaN last)
__device__ __forceinline__ bool kless(double a, double b) {
  if (__builtin_isnan(a)) return false;
  if (__builtin_isnan(b)) return true;
  return a < b;
}

}  // namespace hipns
