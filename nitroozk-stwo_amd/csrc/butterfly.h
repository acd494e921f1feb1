// The M31 butterflies of the circle FFT, shared by the transform kernels (fft.hip) and the
// measurement of their issue-rate ceiling (measure.hip), so that both run the same code.
//
// Twiddles are read from doubled trees (every entry 2t, below 2^32): a t (mod P) for a <= P is
// then hi + lo / 2 with a (2t) = hi 2^32 + lo, since a t = hi 2^31 + lo / 2 and 2^31 = 1 (mod P).
// The sum is below 2P, so one conditional subtraction (a minimum) makes it canonical: 5 operations
// against 6 for the product with t itself.
#pragma once
#include "field.h"

namespace sh {

__device__ __forceinline__ uint32_t mul_tw(uint32_t a, uint32_t t2) {
  const uint64_t p = (uint64_t)a * t2;
  const uint32_t s = (uint32_t)(p >> 32) + ((uint32_t)p >> 1);
  const uint32_t r = s - P;
  return r < s ? r : s;
}
// The negation of a doubled twiddle, again doubled: 2P - t2 (0 stays 0).
__device__ __forceinline__ uint32_t neg_tw(uint32_t t2) { return t2 ? 2 * P - t2 : 0u; }

template <bool INV>
__device__ __forceinline__ void bfly(uint32_t& v0, uint32_t& v1, uint32_t t2) {
  const uint32_t a = v0, b = v1;
  if (INV) {  // ibutterfly(v0, v1, t) = (v0 + v1, (v0 - v1) t)
    v0 = m31_add(a, b);
    v1 = mul_tw(m31_sub(a, b), t2);
  } else {  // butterfly(v0, v1, t) = (v0 + v1 t, v0 - v1 t)
    const uint32_t m = mul_tw(b, t2);
    v0 = m31_add(a, m);
    v1 = m31_sub(a, m);
  }
}

// ---- butterflies in double precision ----------------------------------------------------------
// The FP64 unit of gfx950 issues a fused multiply-add at the rate of the 32-bit integer multiply
// (36.9 T lane-instructions per second against 36.6 T for v_mad_u64_u32; 16 workgroups of 256 per CU),
// and a double holds a field element with 22 bits to spare, so that a transform adds and subtracts
// without reducing: a butterfly is 6 instructions (4 for the product, 2 for the sum and the
// difference) against 11, 6.4 T against 3.9 T butterflies per second on register-resident values.
// Every step is exact. With M = 1.5 2^83, whose neighbours are 2^31 apart, fma(b, t, M) - M is b t
// rounded to a multiple Q of 2^31 (while |b t| < 2^82), b t - Q is an integer of at most 31 bits, so
// its fma does not round, and b t = Q + (b t - Q) = Q / 2^31 + (b t - Q) (mod P), an integer of
// magnitude at most |b t| / 2^31 + 2^30. With t < 2^31 a butterfly at most doubles the magnitude (plus
// 2^30): the at most 5 stages between packings keep values below 2^38, products below 2^69.
constexpr double F64_ROUND31 = 0x1.8p83;

__device__ __forceinline__ double mul_f64(double b, double t, double M) {
  const double Q = __builtin_fma(b, t, M) - M;
  const double r = __builtin_fma(b, t, -Q);
  return __builtin_fma(Q, 0x1p-31, r);
}
// NEG: the twiddle is the negation of t, folded into the butterfly's additions.
template <bool INV, bool NEG = false>
__device__ __forceinline__ void bfly_f64(double& v0, double& v1, double t, double M) {
  const double a = v0, b = v1;
  if (INV) {
    v0 = a + b;
    v1 = mul_f64(NEG ? b - a : a - b, t, M);
  } else {
    const double m = mul_f64(b, t, M);
    v0 = NEG ? a - m : a + m;
    v1 = NEG ? a + m : a - m;
  }
}

// A 32-bit word congruent to the integer v, |v| < 2^49. v + K is added to 1.5 2^51, where a double's
// last bit is worth 1/2: the low word is then 2 ((v + K) mod 2^31) and the high word
// F64_HIGH + floor((v + K) / 2^31), and v + K is congruent to the sum of its two 31-bit parts. K is
// minus F64_HIGH (mod P), so the high word needs no correction: 3 instructions.
constexpr uint32_t F64_HIGH = 0x43280000u;
__device__ __forceinline__ uint32_t pack_f64(double v) {
  const uint64_t y = (uint64_t)__double_as_longlong(v + (0x1.8p51 + (double)(P - F64_HIGH)));
  return ((uint32_t)y >> 1) + (uint32_t)(y >> 32);
}
// The canonical word of v, |v| < 2^41. K = 2^12 P makes the high part not negative, and the sum of the
// parts is then below 2P.
__device__ __forceinline__ uint32_t canon_f64(double v) {
  const uint64_t y = (uint64_t)__double_as_longlong(v + (0x1.8p51 + 4096.0 * (double)P));
  const uint32_t s = ((uint32_t)y >> 1) + (uint32_t)(y >> 32);
  const uint32_t x = s - F64_HIGH, r = s - (F64_HIGH + P);
  return x < r ? x : r;
}

}  // namespace sh
