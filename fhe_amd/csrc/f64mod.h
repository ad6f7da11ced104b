// Exact modular arithmetic on integers held in doubles, for primes q < 2^42.
//
// gfx950 issues an FP64 add, multiply, fused multiply-add or rint per wave as
// fast as a 32-bit multiply-add, so a modular product of two integers below
// 2^53 costs six instructions,
//   h = y w, l = fma(y, w, -h)       (h + l = y w exactly)
//   t = rint(h / q)                  (through the rounded reciprocal)
//   r = fma(-t, q, h) + l            (= y w - t q exactly)
// where a Shoup product of 64-bit integers takes about fifteen: register-only
// butterflies measured 4.0 T/s against 1.77 T/s (Shoup) and 0.95 T/s (the
// exact Montgomery form).
//
// Exactness, for |y w| <= 2^50 q: the quotient's error is below
// 1/2 + 3 * 2^-53 * 2^50 < 0.875, so |r| < 0.875 q; h - t q is an integer
// below 2^53 in magnitude (|h - t q| <= |r| + |l| and |l| <= 2^-53 |y w| <
// 2^40), so the fused multiply-add returns it exactly, and so does the last
// sum.  For |y| <= 2^47 the quotient's error is below 0.55.
//
// Transforms (ntt_r16.h) need no reductions in between: forward values, loaded
// below 2^47, grow by less than 0.55 q a stage; inverse sums double, 2^8 in a
// pass, and every inverse pass starts from values centred to q + 2^32 or less
// in magnitude (f64_load_centred, f64_center), so that products see
// |y| <= 2^50 + 2^40.
#pragma once

#include "device.h"

namespace fhe {

// Whether one of 16 integers is negative or at least 2q + 2^32 (at most 4q,
// for q >= 2^31; smaller primes answer yes always).  Decided on the high
// words: half an instruction a value, and lazy residues, below 2q, never pass
// for wider ones.
__device__ __forceinline__ bool beyond_lazy(const int64_t (&v)[16],
                                            uint64_t q) {
  uint32_t top = 0;
#pragma unroll
  for (int i = 0; i < 16; i++)
    top = max(top, uint32_t(uint64_t(v[i]) >> 32));
  return top > uint32_t((2 * q - 1) >> 32) || q < (uint64_t(1) << 31);
}

// Replaces 16 representatives by residues in [0, 2q) where beyond_lazy.  One
// at a time: the rare case takes no registers from the usual one.
__device__ __forceinline__ void load_residues(int64_t (&v)[16], uint64_t q,
                                              uint64_t k, int64_t r2) {
  if (beyond_lazy(v, q)) {
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int64_t y = mont_exit(mont_mult(r2, v[i], q, k), q, k);
      v[i] = y < 0 ? y + int64_t(q) : y;
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

struct F64Mod {
  double q, qi; // the prime and its rounded reciprocal
};

__device__ __forceinline__ double f64_mul(double y, double w,
                                          const F64Mod &m) {
  const double h = y * w;
  const double l = __builtin_fma(y, w, -h);
  const double t = __builtin_rint(h * m.qi);
  return __builtin_fma(-t, m.q, h) + l;
}

// x mod q in [-q/2 - 1, q/2 + 1], |x| <= 2^50 q
__device__ __forceinline__ double f64_center(double x, const F64Mod &m) {
  return __builtin_fma(-__builtin_rint(x * m.qi), m.q, x);
}

// x mod q in [0, q] (q itself only where the rounded quotient of a multiple
// of q falls short), |x| <= 2^50: the quotient's error times q is below 1
__device__ __forceinline__ double f64_floor_mod(double x, const F64Mod &m) {
  return __builtin_fma(-__builtin_floor(x * m.qi), m.q, x);
}

// A product's value (|r| < 0.875 q) as the canonical residue.
__device__ __forceinline__ double f64_canonical(double r, const F64Mod &m) {
  return r < 0 ? r + m.q : r;
}

// Integer in [0, 2^52) to and from a double, through the bits of 2^52 + x.
__device__ __forceinline__ int64_t f64_to_int(double x) {
  const uint64_t b = uint64_t(__double_as_longlong(x + 0x1p52));
  return int64_t(b & ((uint64_t(1) << 52) - 1));
}

// Integer in [-2^51, 2^51) as a double.
__device__ __forceinline__ double f64_from_int(int64_t v) {
  const uint32_t hi = uint32_t(uint64_t(v) >> 32) + 0x43380000u;
  const uint64_t b = (uint64_t(hi) << 32) | uint32_t(v);
  return __longlong_as_double(int64_t(b)) - 0x1.8p52;
}

// Nonzero when some v[m] lies outside [-2^47, 2^47).
__device__ __forceinline__ uint32_t f64_wild(const int64_t (&v)[16]) {
  uint32_t w = 0;
#pragma unroll
  for (int m = 0; m < 16; m++)
    w |= uint32_t(uint64_t(v[m]) >> 32) + 0x8000u;
  return w >> 16;
}

// The residue of any int64 as a double below 2^32 + 0.875 q in magnitude.
__device__ __forceinline__ double f64_from_any(int64_t v, const F64Mod &m) {
  const double c = f64_floor_mod(0x1p32, m); // 2^32 mod q
  return f64_mul(double(int32_t(uint64_t(v) >> 32)), c, m) +
         double(uint32_t(v));
}

// Doubles of 16 integers: exact where all lie in [-2^47, 2^47) (residues
// and sums of residues of primes below 2^42 do), else residues mod q.
__device__ __forceinline__ void f64_load(const int64_t (&v)[16],
                                         double (&x)[16], const F64Mod &m) {
  if (f64_wild(v)) {
#pragma unroll
    for (int i = 0; i < 16; i++)
      x[i] = f64_from_any(v[i], m);
  } else {
#pragma unroll
    for (int i = 0; i < 16; i++)
      x[i] = f64_from_int(v[i]);
  }
}

// Any int64's residue in about [-q/2, q/2].
__device__ __forceinline__ double f64_center_any(int64_t v, const F64Mod &m) {
  return f64_center(f64_from_any(v, m), m);
}

// Doubles of 16 representatives within q + 2^32 of zero: lazy residues less
// q, others centred.
__device__ __forceinline__ void f64_load_centred(const int64_t (&v)[16],
                                                 double (&x)[16], uint64_t q,
                                                 const F64Mod &m) {
  if (beyond_lazy(v, q)) {
#pragma unroll
    for (int i = 0; i < 16; i++)
      x[i] = f64_center_any(v[i], m);
  } else {
#pragma unroll
    for (int i = 0; i < 16; i++)
      x[i] = f64_from_int(v[i]) - m.q;
  }
}

} // namespace fhe
