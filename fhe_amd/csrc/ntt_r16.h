// Register-resident radix-16 rounds of an L-bit NTT pass (L = 6, 7 or 8),
// shared by the standalone NTT kernel and the fused key-switching kernels.
//
// A tile holds 4096 points: 2^(12 - L) sub-transforms of 2^L points;
// sub-transform c is owned by the T = 2^(L - 4) threads with row r = 0..T-1,
// each holding 16 points v[m].  Two ownerships are used:
//   ROWS  j = r + T m    (bits L-1..L-4 of j vary inside a thread)
//   COLS  j = 16 r + m   (bits 3..0 vary inside a thread)
// The forward pass runs its local bits L-1..L-4 in ROWS and the others in
// COLS; the inverse pass runs 0..L-5 in COLS and the last four in ROWS.
// N = 2^13 splits into passes of 7 low and 6 high bits, 2^14 into 7 and 7,
// 2^15 into 8 and 7, 2^16 into 8 and 8 (r16_low_bits).  Twiddle addressing
// is derived in the ntt.hip header comment.
//
// Three arithmetics share the loop structure (template parameter A):
//   kExact      the reference's radix-2 formulas with Montgomery twiddles
//               (src/operation/ntt.cpp:46-134, :177-272), so every lazy
//               representative in [0, 2q) matches the reference;
//   kF64        for q < 2^42: integers in doubles (f64mod.h), standard-form
//               twiddles, no reductions inside a pass.  Between the two
//               passes of a transform the values stay doubles (in the int64
//               buffers); the first pass reads integers and the last one
//               writes integers.
//   kLazyLarge  lazy forms after Harvey for any q < 2^61 on short Shoup
//               products (shoup_short_neg, in [0, 4q)): forward values in
//               [0, 8q), inverse values in [0, 4q), one conditional
//               subtraction of 4q per butterfly.
// The lazy forms give other representatives of the same residues; they serve
// stages whose results are canonicalized before anything representative-
// dependent reads them.
#pragma once

#include <type_traits>

#include "device.h"
#include "f64mod.h"

namespace fhe {

// Low (contiguous) and high (strided) index bits of the two radix-16 passes
// of N = 2^log_n, and the sizes they serve.
__host__ __device__ constexpr bool r16_supported(int log_n) {
  return log_n >= 13 && log_n <= 16;
}
__host__ __device__ constexpr int r16_low_bits(int log_n) {
  return (log_n + 1) / 2;
}
__host__ __device__ constexpr int r16_high_bits(int log_n) {
  return log_n - r16_low_bits(log_n);
}

// Calls f with log2 N (13 .. 16) as a compile-time constant.
template <class F> void with_log_n(int log_n, F &&f) {
  switch (log_n) {
  case 13:
    f(std::integral_constant<int, 13>());
    break;
  case 14:
    f(std::integral_constant<int, 14>());
    break;
  case 15:
    f(std::integral_constant<int, 15>());
    break;
  default:
    f(std::integral_constant<int, 16>());
  }
}

enum NttArith : int { kExact = 0, kF64 = 1, kLazyLarge = 2 };

// Values of a transform in arithmetic A.
template <int A>
using R16Value = std::conditional_t<A == kF64, double, int64_t>;

// Primes below this bound take the kF64 forms.
constexpr uint64_t kF64Bound = uint64_t(1) << 42;

// Host side: whether prime p takes the kF64 forms.
inline bool t_host_q_small(const DeviceTables &t, int p) {
  return t.host_q[p] < kF64Bound;
}

// Exact butterflies with the reference's signed arithmetic.  Operands are
// the reference's representatives: lazy residues in [0, 2q), and at the
// input of a transform possibly negative values (limbs that a larger prime
// rescaled lie in (-q, q)).  The signed product and compares reproduce the
// reference for both; on non-negative operands they equal the unsigned
// forms.  Cooley-Tukey: p = mont(w, y); x' = guard(x + p, 2q);
// y' = guard(x + 2q - p, 2q).  nq2 = -2q, which the guards add in place of
// subtracting 2q (guard_neg); the overloads without it serve callers that
// do not hold it.
__device__ __forceinline__ void ct_butterfly(int64_t &x, int64_t &y, int64_t w,
                                             int64_t q2, int64_t nq2,
                                             uint64_t q, uint64_t k) {
  const int64_t p = mont_mult_cs(w, y, q, k);
  const int64_t x0 = x;
  x = guard_neg(add64(x0, p), q2, nq2);
  y = guard_neg(sub64(add64(x0, q2), p), q2, nq2);
}
__device__ __forceinline__ void ct_butterfly(int64_t &x, int64_t &y, int64_t w,
                                             int64_t q2, uint64_t q,
                                             uint64_t k) {
  ct_butterfly(x, y, w, q2, -q2, q, k);
}

// Gentleman-Sande: x' = guard(x + y, 2q); y' = mont(w, guard(x + 2q - y, 2q))
__device__ __forceinline__ void gs_butterfly(int64_t &x, int64_t &y, int64_t w,
                                             int64_t q2, int64_t nq2,
                                             uint64_t q, uint64_t k) {
  const int64_t x0 = x, y0 = y;
  x = guard_neg(add64(x0, y0), q2, nq2);
  y = mont_mult_cs(w, guard_neg(sub64(add64(x0, q2), y0), q2, nq2), q, k);
}
__device__ __forceinline__ void gs_butterfly(int64_t &x, int64_t &y, int64_t w,
                                             int64_t q2, uint64_t q,
                                             uint64_t k) {
  gs_butterfly(x, y, w, q2, -q2, q, k);
}

// Load-time product with a per-prime constant (mont_enter by R^2 for the
// reference's to_ntt) of a possibly negative input value.  The lazy
// arithmetic takes non-negative operands only: the signed product lies in
// (-q, q), and a negative one is replaced by the residue's representative
// in [0, q).
template <int A>
__device__ __forceinline__ int64_t load_product(int64_t v, int64_t c,
                                                uint64_t q, uint64_t k) {
  int64_t y = mont_mult_cs(c, v, q, k);
  if (A != kExact && y < 0)
    y += int64_t(q);
  return y;
}

// Everything a thread needs to address twiddles in one L-bit pass: the pass
// covers index bits [b, b+L) of a limb of 2^log_n points; hi is the
// sub-transform's index bits above b+L and r the thread's row.
struct R16Pass {
  const int64_t *tw;   // Montgomery twiddles of this prime (kExact)
  const uint64_t *ts;  // {w, w'} pairs of this prime (kLazyLarge)
  const double *tf;    // twiddles of this prime (kF64)
  int64_t n;
  int64_t hi;
  int log_n;
  int b;
  int r;
  int64_t q2;
  int64_t nq2;  // -q2 through opaque_neg, for the exact arithmetic
  uint64_t q, k;
  uint64_t nq;  // 2^64 - q through opaque_neg, for kLazyLarge
  F64Mod f;     // kF64
};

// The fields of a pass that depend on the prime p.
template <int A, bool INV>
__device__ __forceinline__ void r16_prime(R16Pass &s, const DeviceTables &t,
                                          int p) {
  const int64_t at = int64_t(p) << t.log_n;
  s.n = int64_t(1) << t.log_n;
  s.log_n = t.log_n;
  s.q = t.q[p];
  s.k = t.k[p];
  s.q2 = int64_t(t.q2[p]);
  if (A == kExact) {
    s.tw = (INV ? t.root_inverse : t.root) + at;
    s.nq2 = opaque_neg(s.q2);
  } else if (A == kLazyLarge) {
    s.ts = (INV ? t.root_inverse_shoup : t.root_shoup) + at * 2;
    s.nq = uint64_t(opaque_neg(int64_t(s.q)));
  } else {
    s.tf = (INV ? t.root_inverse_f64 : t.root_f64) + at;
    s.f = {t.q_f64[p], t.q_inverse_f64[p]};
  }
}

// One forward butterfly on (x, y) with twiddle entry idx.
template <int A>
__device__ __forceinline__ void fwd_bfly(R16Value<A> &x, R16Value<A> &y,
                                         const R16Pass &s, int64_t idx) {
  if constexpr (A == kExact) {
    ct_butterfly(x, y, s.tw[idx], s.q2, s.nq2, s.q, s.k);
  } else if constexpr (A == kF64) {
    const double p = f64_mul(y, s.tf[idx], s.f);
    y = x - p;
    x = x + p;
  } else {
    const uint64_t w = s.ts[2 * idx], wq = s.ts[2 * idx + 1];
    const int64_t x0 = guard_u(x, 2 * s.q2);
    const int64_t p = int64_t(shoup_short_neg(uint64_t(y), w, wq, s.nq));
    x = add64(x0, p);
    y = sub64(add64(x0, 2 * s.q2), p);
  }
}

// One inverse butterfly.
template <int A>
__device__ __forceinline__ void inv_bfly(R16Value<A> &x, R16Value<A> &y,
                                         const R16Pass &s, int64_t idx) {
  if constexpr (A == kExact) {
    gs_butterfly(x, y, s.tw[idx], s.q2, s.nq2, s.q, s.k);
  } else if constexpr (A == kF64) {
    const double d = x - y;
    x = x + y;
    y = f64_mul(d, s.tf[idx], s.f);
  } else {
    const uint64_t w = s.ts[2 * idx], wq = s.ts[2 * idx + 1];
    const int64_t d = sub64(add64(x, 2 * s.q2), y);
    x = guard_u(add64(x, y), 2 * s.q2);
    y = int64_t(shoup_short_neg(uint64_t(d), w, wq, s.nq));
  }
}

// forward local bits L-1..L-4, ROWS ownership
template <int L, int A>
__device__ __forceinline__ void r16_forward_high(R16Value<A> (&v)[16],
                                                 const R16Pass &s) {
#pragma unroll
  for (int x = 3; x >= 0; x--) {
    const int u = x + L - 4;
    const int stage = s.log_n - 1 - s.b - u;
    const int64_t tb = (int64_t(1) << stage) - 1 + (s.hi << (L - 1 - u));
#pragma unroll
    for (int m = 0; m < 16; m++) {
      if (m & (1 << x))
        continue;
      fwd_bfly<A>(v[m], v[m + (1 << x)], s, tb + (m >> (x + 1)));
    }
  }
}

// forward local bits L-5..0, COLS ownership
template <int L, int A>
__device__ __forceinline__ void r16_forward_low(R16Value<A> (&v)[16],
                                                const R16Pass &s) {
#pragma unroll
  for (int u = L - 5; u >= 0; u--) {
    const int stage = s.log_n - 1 - s.b - u;
    const int64_t tb = (int64_t(1) << stage) - 1 + (s.hi << (L - 1 - u)) +
                       (int64_t(s.r) << (3 - u));
#pragma unroll
    for (int m = 0; m < 16; m++) {
      if (m & (1 << u))
        continue;
      fwd_bfly<A>(v[m], v[m + (1 << u)], s, tb + (m >> (u + 1)));
    }
  }
}

// inverse local bits 0..L-5, COLS ownership
template <int L, int A>
__device__ __forceinline__ void r16_inverse_low(R16Value<A> (&v)[16],
                                                const R16Pass &s) {
#pragma unroll
  for (int u = 0; u <= L - 5; u++) {
    const int64_t tb = s.n - (s.n >> (s.b + u)) + (s.hi << (L - 1 - u)) +
                       (int64_t(s.r) << (3 - u));
#pragma unroll
    for (int m = 0; m < 16; m++) {
      if (m & (1 << u))
        continue;
      inv_bfly<A>(v[m], v[m + (1 << u)], s, tb + (m >> (u + 1)));
    }
  }
}

// inverse local bits L-4..L-1, ROWS ownership
template <int L, int A>
__device__ __forceinline__ void r16_inverse_high(R16Value<A> (&v)[16],
                                                 const R16Pass &s) {
#pragma unroll
  for (int x = 0; x <= 3; x++) {
    const int u = x + L - 4;
    const int64_t tb = s.n - (s.n >> (s.b + u)) + (s.hi << (L - 1 - u));
#pragma unroll
    for (int m = 0; m < 16; m++) {
      if (m & (1 << x))
        continue;
      inv_bfly<A>(v[m], v[m + (1 << x)], s, tb + (m >> (x + 1)));
    }
  }
}

// Bring kLazyLarge forward outputs (below 8q) to [0, 2q).
template <int A>
__device__ __forceinline__ void r16_forward_settle(R16Value<A> (&v)[16],
                                                   const R16Pass &s) {
  if constexpr (A == kLazyLarge) {
#pragma unroll
    for (int m = 0; m < 16; m++)
      v[m] = guard_u(guard_u(v[m], 2 * s.q2), s.q2);
  }
}

// LDS exchange buffer: a tile's sub-transforms in rows of 2^L points, padded
// so that both ownerships and the sub-transforms of a row spread over the
// banks.
template <int L> constexpr int kR16Row = (1 << L) + (1 << (L - 4)) + 1;
template <int L> constexpr int kR16Lds = (4096 >> L) * kR16Row<L>;

template <int L> __device__ __forceinline__ int r16_lds(int c, int j) {
  return c * kR16Row<L> + j + (j >> 4);
}

// Index within its sub-transform of the thread's point m.
template <int L, bool COLS_OWNED>
__device__ __forceinline__ int r16_point(int r, int m) {
  return COLS_OWNED ? 16 * r + m : r + (1 << (L - 4)) * m;
}

// Orders one wavefront's LDS accesses: a wave's LDS instructions execute in
// issue order, so it is enough that the compiler moves no access across.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Re-own the thread's 16 points: ROWS -> COLS (TO_COLS) or COLS -> ROWS.
// Starts with a barrier so the previous use of the buffer has finished.
// WAVE: the threads sharing c are consecutive (c = tid / T, T <= 16), hence
// in one wavefront, and a wavefront barrier replaces the block's.
template <int L, bool TO_COLS, bool WAVE = false, class V>
__device__ __forceinline__ void r16_exchange(V (&v)[16], int64_t *buffer,
                                             int c, int r) {
  V *lds = reinterpret_cast<V *>(buffer);
  if (WAVE)
    wave_lds_sync();
  else
    __syncthreads();
#pragma unroll
  for (int m = 0; m < 16; m++)
    lds[r16_lds<L>(c, r16_point<L, !TO_COLS>(r, m))] = v[m];
  if (WAVE)
    wave_lds_sync();
  else
    __syncthreads();
#pragma unroll
  for (int m = 0; m < 16; m++)
    v[m] = lds[r16_lds<L>(c, r16_point<L, TO_COLS>(r, m))];
}

// r16_exchange through a buffer of 32-bit words, half the LDS of the 64-bit
// exchange (so that twice as many blocks fit on a CU): the low words go
// through first, then the high words, each between two barriers.
template <int L, bool TO_COLS, class V>
__device__ __forceinline__ void r16_exchange_words(V (&x)[16], uint32_t *lds,
                                                   int c, int r) {
  int64_t v[16];
  uint32_t lo[16];
#pragma unroll
  for (int m = 0; m < 16; m++)
    v[m] = __builtin_bit_cast(int64_t, x[m]);
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 16; m++)
    lds[r16_lds<L>(c, r16_point<L, !TO_COLS>(r, m))] = uint32_t(v[m]);
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 16; m++)
    lo[m] = lds[r16_lds<L>(c, r16_point<L, TO_COLS>(r, m))];
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 16; m++)
    lds[r16_lds<L>(c, r16_point<L, !TO_COLS>(r, m))] =
        uint32_t(uint64_t(v[m]) >> 32);
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 16; m++)
    x[m] = __builtin_bit_cast(
        V, (uint64_t(lds[r16_lds<L>(c, r16_point<L, TO_COLS>(r, m))]) << 32) |
               lo[m]);
}

// One register-resident L-bit pass over one 4096-point tile of one limb:
// the sub-transforms of the tile are owned by T threads each (16 points per
// thread) and the L radix-2 stages run as two rounds (four stages and L - 4)
// with one LDS exchange between them.  A second exchange is added where the
// global side of the pass is contiguous and the register ownership is not,
// so that every global access is coalesced.  src / dst point at the limb
// (prime p); the pass covers index bits [b, b + L); COLS is b > 0.  pre
// (forward, per prime) multiplies every loaded value first; post (inverse)
// is the InttPost epilogue; last = the pass completes a forward transform.
// The first pass of a lazy inverse takes any representatives, that of a lazy
// forward transform any with pre or in kF64, else values in [0, 8q).
// zero (lazy inverse): a flag word of the limb, cleared by the first pass and
// set by the last one where a canonical result is zero (repair_zero_kernel).
// more (lazy second inverse pass): this limb of the first of more_count
// buffers, more_stride words apart, that are added to the source.
// OPAQUE: the pass runs inside a persistent loop (opaque_tid).
template <int L, bool INV, bool COLS, int A, bool OPAQUE = false>
__device__ __forceinline__ void r16_limb_pass(const int64_t *src_limb,
                                              int64_t *dst_limb, int p,
                                              int tile, int b,
                                              const int64_t *pre, int post,
                                              bool last, const DeviceTables &t,
                                              int64_t *lds,
                                              uint32_t *zero = nullptr,
                                              const int64_t *more = nullptr,
                                              int64_t more_stride = 0,
                                              int more_count = 0) {
  const int tid = OPAQUE ? opaque_tid() : int(threadIdx.x);
  constexpr int T = 1 << (L - 4), C = 4096 >> L;
  const int c = COLS ? (tid & (C - 1)) : (tid >> (L - 4));
  const int r = COLS ? (tid >> (12 - L)) : (tid & (T - 1));
  const int64_t sp = int64_t(tile) * C + c;
  const int64_t lo = sp & ((int64_t(1) << b) - 1);
  const int64_t hi = sp >> b;
  const int64_t base = (hi << (b + L)) + lo;
  const int64_t *src = src_limb + base;
  int64_t *dst = dst_limb + base;

  R16Pass s;
  r16_prime<A, INV>(s, t, p);
  s.hi = hi;
  s.b = b;
  s.r = r;

  R16Value<A> v[16];
  // load in the ownership of the first round; the contiguous inverse pass
  // loads coalesced ROWS and re-owns through LDS
  constexpr bool cols_load = INV && COLS;
  constexpr bool first_pass = INV != COLS; // of the two in this direction
  int64_t w[16];
#pragma unroll
  for (int m = 0; m < 16; m++)
    w[m] = src[int64_t(r16_point<L, cols_load>(r, m)) << b];
  if constexpr (A == kF64) {
    if (first_pass && INV) {
      f64_load_centred(w, v, s.q, s.f);
    } else if (first_pass) {
      f64_load(w, v, s.f);
      if (pre) {
        // the Montgomery product with pre is one with pre R^-1
        const double c = double(mont_exit(pre[p], s.q, s.k));
#pragma unroll
        for (int m = 0; m < 16; m++)
          v[m] = f64_mul(v[m], c, s.f);
      }
    } else {
#pragma unroll
      for (int m = 0; m < 16; m++) {
        v[m] = __longlong_as_double(w[m]);
      }
      if (INV) {
        for (int g = 0; g < more_count; g++)
#pragma unroll
          for (int m = 0; m < 16; m++)
            v[m] += __longlong_as_double(
                more[g * more_stride + base +
                     (int64_t(r16_point<L, cols_load>(r, m)) << b)]);
#pragma unroll
        for (int m = 0; m < 16; m++)
          v[m] = f64_center(v[m], s.f);
      }
    }
  } else {
    if (A == kLazyLarge && INV && first_pass)
      load_residues(w, s.q, s.k, t.r2[p]);
#pragma unroll
    for (int m = 0; m < 16; m++)
      v[m] = pre ? load_product<A>(w[m], pre[p], s.q, s.k) : w[m];
    if (A == kLazyLarge && INV && !first_pass)
      for (int g = 0; g < more_count; g++)
#pragma unroll
        for (int m = 0; m < 16; m++)
          v[m] = guard_u(
              add64(v[m], more[g * more_stride + base +
                               (int64_t(r16_point<L, cols_load>(r, m))
                                << b)]),
              2 * s.q2);
  }
  if (INV && !COLS)
    r16_exchange<L, true, !COLS>(v, lds, c, r);

  if (!INV) {
    r16_forward_high<L, A>(v, s);
    r16_exchange<L, true, !COLS>(v, lds, c, r);
    r16_forward_low<L, A>(v, s);
    if (last)
      r16_forward_settle<A>(v, s);
    if (!COLS)
      r16_exchange<L, false, !COLS>(v, lds, c, r); // coalesced contiguous store
  } else {
    r16_inverse_low<L, A>(v, s);
    r16_exchange<L, false, !COLS>(v, lds, c, r);
    r16_inverse_high<L, A>(v, s);
    if constexpr (A == kF64) {
      if (post != kInttRaw) {
        // N^-1 and the exit of the Montgomery form in one product; the key
        // products of kInttKeyReduce carry one more R
        int64_t c = mont_exit(mont_exit(t.ninv[p], s.q, s.k), s.q, s.k);
        if (post == kInttKeyReduce)
          c = mont_exit(c, s.q, s.k);
        const double cd = double(c);
#pragma unroll
        for (int m = 0; m < 16; m++)
          v[m] = f64_canonical(f64_mul(v[m], cd, s.f), s.f);
      }
    } else if (post != kInttRaw) {
      const int64_t ninv = t.ninv[p];
      if constexpr (A == kExact) {
        const bool reduce = post != kInttExit;
#pragma unroll
        for (int m = 0; m < 16; m++) {
          // only the exact arithmetic carries negative values
          const int64_t y =
              mont_exit(mont_mult_cs(ninv, v[m], s.q, s.k), s.q, s.k);
          v[m] = reduce ? guard(y, int64_t(s.q)) : y;
        }
      } else {
        // kLazyLarge needs only the residue: one product with N^-1 R^-1
        // (the exit folded into the constant) of v brought below 2q gives it
        // below v q / 2^62 + q < 2q, which the guard makes canonical
        const int64_t ninv_exit = mont_exit(ninv, s.q, s.k);
#pragma unroll
        for (int m = 0; m < 16; m++)
          v[m] = guard_u(
              mont_mult_u(guard_u(v[m], s.q2), ninv_exit, s.q, s.k),
              int64_t(s.q));
      }
    }
  }
  // store: ROWS ownership except the strided forward pass (COLS)
  constexpr bool cols_store = !INV && COLS;
  bool any_zero = false;
#pragma unroll
  for (int m = 0; m < 16; m++) {
    int64_t y;
    if constexpr (A != kF64)
      y = v[m];
    else if (first_pass)
      y = __double_as_longlong(v[m]);
    else
      y = f64_to_int(INV && post != kInttRaw ? v[m]
                                             : f64_floor_mod(v[m], s.f));
    if (INV && A != kExact && !first_pass)
      any_zero = any_zero || y == 0;
    dst[int64_t(r16_point<L, cols_store>(r, m)) << b] = y;
  }
  if (INV && A != kExact && zero) {
    if (first_pass ? (tile == 0 && tid == 0) : any_zero)
      *zero = first_pass ? 0 : 1;
  }
}

} // namespace fhe
