// Work items of the fused key-switching kernels (N = 2^13 .. 2^16), addressed
// through small per-item views so that the batched kernels (one moduli_id
// for the whole batch) and the uneven-level kernels (a moduli_id per
// ciphertext) share one body.
//
// ks_item_tile: the key inner product of one 4096-coefficient tile of one
// extended limb of one ciphertext (src/ckks/core_key_switch.cpp:293-358):
// for every partition in turn, the low-bit forward NTT pass of the extended
// polynomial (the high-bit pass ran before), the products with both key
// halves and their accumulation in registers; then the low-bit pass of the
// inverse NTT on both accumulators before a single write.
//
// ext_item_tile: one extended limb of one partition formed from the Garner
// digits (src/ckks/core_key_switch.cpp:92-108) with the first (high-bit)
// forward NTT pass fused before its only write.
#pragma once

#include "kernels.h"
#include "modup.h"
#include "ntt_r16.h"

namespace fhe {

// Arguments of the batched key inner product (one moduli_id for the batch).
struct KsArgs {
  const int64_t *ext;  // [count][parts][ext_limbs][N], forward pass 1 done
  const int64_t *key;  // [key_polys][key_chain][N]
  int64_t *acc;        // [count][2][ext_limbs][N], inverse pass 1 done
  int count;
  int parts;
  int ext_limbs;
  int moduli_id;
  int key_chain;
  int key_offset;      // first key limb aligned with the ciphertext's limb 0
  int key_partition0;  // key partition index of the ciphertext's partition 0
  int limb0, limbs_here; // extended limbs of the launch
  int swizzle;
  // splits of an item over blocks: `groups` ranges of partitions, group g > 0
  // writing its sums to partials + (g - 1) * [count][2][ext_limbs][N], and
  // with halves = 2 one block per key half
  int groups, halves;
  int64_t *partials;
  // NTT form of the key-switched polynomial, when the caller has it: limb i
  // of ciphertext c at own + c * own_stride + i * N.  The extended limbs of a
  // partition's own primes are that polynomial's limbs, so their transforms
  // are taken from here instead of the extended polynomial (any
  // representative serves: the key products are canonicalized later).
  const int64_t *own;
  int64_t own_stride;
  int start[kMaxFusedParts];
  int size[kMaxFusedParts];
  int lazy_acc;        // large primes: sums below 2q with one guard
};


// The key inner product reaches its data through an addressing policy
// `Addr` (one per kernel family) with the members
//   int parts, ext_limbs, moduli_id, key_chain, lazy_acc;
//   bool is_own(pp, i)          limb i of partition pp is the source's own
//   const int64_t *own(i, off)  that limb's NTT-form tile (thread row 0)
//   const int64_t *ext(pp, i, off)  the extended limb's tile
//   const int64_t *key_tile(pp, i, off)  key half 0 of partition pp (half 1
//                               is key_chain limbs further)
//   int64_t *acc(i, off)        accumulator half 0 (half 1 is ext_limbs
//                               limbs further)
// A partition's own extended limbs are the NTT-form source's limbs, so their
// transforms are taken from there (any representative serves: the key
// products are canonicalized later).

// The (extended limb i, tile) work item of one ciphertext with arithmetic A
// for the two transforms.  The key products of the 64-bit forms are
// Montgomery products of operands whose product stays below q * 2^62,
// accumulated with the reference's guards (lazy_acc: one conditional
// subtraction for kLazyLarge); the kF64 sums need no guards (up to 64 parts
// of less than 0.55 q each).  Every form gives the same residues, and the
// accumulators are canonicalized after the inverse transform.
// LOGN: log2 N.
// OPAQUE: the tile runs inside a persistent loop (opaque_tid).
// p0, p1: the partitions to sum.  BOTH: both key halves, else half `half`.
template <int LOGN, int A, bool BOTH, class Addr, bool OPAQUE = false>
__device__ __forceinline__ void ks_item_tile(const Addr &a,
                                             const DeviceTables &t,
                                             int64_t *lds, int tile, int i,
                                             int p0, int p1, int half) {
  constexpr int L = r16_low_bits(LOGN);
  const int64_t n = int64_t(1) << t.log_n;
  const int p = a.moduli_id + i;
  const int tid = OPAQUE ? opaque_tid() : int(threadIdx.x);
  const int r = tid & ((1 << (L - 4)) - 1);
  const int c = tid >> (L - 4);
  const int64_t sp = int64_t(tile) * (4096 >> L) + c; // sub-transform
  const int64_t off = sp << L;

  R16Pass f;
  r16_prime<A, false>(f, t, p);
  f.hi = sp;
  f.b = 0;
  f.r = r;
  const int64_t qq = int64_t(f.q);

  R16Value<A> acc0[16], acc1[16], v[16];
  for (int pp = p0; pp < p1; pp++) {
    int64_t w[16];
    // block-uniform: every thread of the block has the same (i, pp)
    if (a.is_own(pp, i)) {
      const int64_t *src = a.own(i, off);
#pragma unroll
      for (int m = 0; m < 16; m++)
        w[m] = src[r16_point<L, true>(r, m)];
      if constexpr (A == kF64) {
        f64_load(w, v, f.f);
      } else {
        load_residues(w, f.q, f.k, t.r2[p]);
#pragma unroll
        for (int m = 0; m < 16; m++)
          v[m] = w[m];
      }
    } else {
      const int64_t *src = a.ext(pp, i, off);
#pragma unroll
      for (int m = 0; m < 16; m++)
        v[m] = __builtin_bit_cast(R16Value<A>,
                                  src[r16_point<L, false>(r, m)]);
      r16_forward_high<L, A>(v, f);
      r16_exchange<L, true, true>(v, lds, c, r);
      r16_forward_low<L, A>(v, f);
      r16_forward_settle<A>(v, f);
    }
    // v[m] is now the NTT value at coefficient off + 16 r + m
    const int64_t *k0 = a.key_tile(pp, i, off) + 16 * r +
                        (BOTH ? 0 : int64_t(half) * a.key_chain * n);
    const int64_t *k1 = k0 + int64_t(a.key_chain) * n;
    if constexpr (A == kF64) {
      // plain products: the sums carry the key's Montgomery factor R, which
      // the epilogue of the second inverse pass takes out (kInttKeyReduce)
      auto products = [&](const int64_t *key, double (&acc)[16]) {
        int64_t kw[16];
#pragma unroll
        for (int m = 0; m < 16; m++)
          kw[m] = key[m];
        load_residues(kw, f.q, f.k, t.r2[p]);
#pragma unroll
        for (int m = 0; m < 16; m++) {
          const double x = f64_mul(v[m], f64_from_int(kw[m]), f.f);
          acc[m] = pp == p0 ? x : acc[m] + x;
        }
      };
      products(k0, acc0);
      if constexpr (BOTH)
        products(k1, acc1);
    } else if (pp == p0) {
#pragma unroll
      for (int m = 0; m < 16; m++) {
        acc0[m] = mont_mult_u(v[m], k0[m], f.q, f.k);
        if (BOTH)
          acc1[m] = mont_mult_u(v[m], k1[m], f.q, f.k);
      }
    } else if (A == kLazyLarge && a.lazy_acc) {
      // sums kept below 2q (one conditional subtraction of 2q): the lazy
      // inverse transform that follows takes inputs below 2q
#pragma unroll
      for (int m = 0; m < 16; m++) {
        acc0[m] = guard_u(add64(mont_mult_u(v[m], k0[m], f.q, f.k), acc0[m]),
                          f.q2);
        if (BOTH)
          acc1[m] = guard_u(
              add64(mont_mult_u(v[m], k1[m], f.q, f.k), acc1[m]), f.q2);
      }
    } else {
#pragma unroll
      for (int m = 0; m < 16; m++) {
        acc0[m] = guard_u(
            guard_u(add64(mont_mult_u(v[m], k0[m], f.q, f.k), acc0[m]), f.q2),
            qq);
        if (BOTH)
          acc1[m] = guard_u(
              guard_u(add64(mont_mult_u(v[m], k1[m], f.q, f.k), acc1[m]),
                      f.q2),
              qq);
      }
    }
  }

  R16Pass g = f;
  r16_prime<A, true>(g, t, p);
  int64_t *d0 = a.acc(i, off);
  int64_t *d1 = d0 + int64_t(a.ext_limbs) * n;
  if (!BOTH && half)
    d0 = d1;
  auto inverse = [&](R16Value<A> (&x)[16], int64_t *d) {
    if constexpr (A == kF64) {
#pragma unroll
      for (int m = 0; m < 16; m++)
        x[m] = f64_center(x[m], f.f);
    }
    r16_inverse_low<L, A>(x, g);
    r16_exchange<L, false, true>(x, lds, c, r);
    r16_inverse_high<L, A>(x, g);
#pragma unroll
    for (int m = 0; m < 16; m++)
      d[r16_point<L, false>(r, m)] = __builtin_bit_cast(int64_t, x[m]);
  };
  inverse(acc0, d0);
  if (BOTH)
    inverse(acc1, d1);
}

// Addressing of ciphertext ct of a batch at one moduli_id (KsArgs).
template <int LOGN> struct KsBatchAddr {
  const KsArgs &a;
  int ct;
  int64_t *sums;
  int parts, ext_limbs, moduli_id, key_chain, lazy_acc;
  __device__ KsBatchAddr(const KsArgs &args, int c, int group)
      : a(args), ct(c),
        sums(group == 0
                 ? args.acc
                 : args.partials + ((int64_t(group - 1) * args.count * 2 *
                                     args.ext_limbs)
                                    << LOGN)), parts(args.parts),
        ext_limbs(args.ext_limbs), moduli_id(args.moduli_id),
        key_chain(args.key_chain), lazy_acc(args.lazy_acc) {}
  __device__ bool is_own(int pp, int i) const {
    return a.own != nullptr && i >= a.start[pp] && i < a.start[pp] + a.size[pp];
  }
  __device__ const int64_t *own(int i, int64_t off) const {
    return a.own + int64_t(ct) * a.own_stride + (int64_t(i) << LOGN) + off;
  }
  __device__ const int64_t *ext(int pp, int i, int64_t off) const {
    return a.ext + (((int64_t(ct) * a.parts + pp) * a.ext_limbs + i) << LOGN) +
           off;
  }
  __device__ const int64_t *key_tile(int pp, int i, int64_t off) const {
    const int kp = a.key_partition0 + pp;
    return a.key +
           ((int64_t(2 * kp) * a.key_chain + a.key_offset + i) << LOGN) + off;
  }
  __device__ int64_t *acc(int i, int64_t off) const {
    return sums + ((int64_t(ct) * 2 * a.ext_limbs + i) << LOGN) + off;
  }
};

// Where one (ciphertext, partition)'s digits, constants and extended limbs
// live.
struct ExtItem {
  const int64_t *digits; // this partition's [maxz][N] Garner digits
  const int64_t *cst;    // this partition's ModUp constants
  int64_t *ext;          // this partition's [ext_limbs][N]
  int start, size, ext_limbs, moduli_id, ext_shoup_offset;
};

// lds: kExtendLds<LOGN, A> words.  LOGN, OPAQUE: as for ks_item_tile.
//
// The 64-bit forms exchange through 32-bit words (half the LDS: six waves per
// SIMD); kF64 holds about 100 registers, so that four waves fit either way,
// and takes the 64-bit exchange with half the barriers.
template <int LOGN, int A>
constexpr int kExtendLds =
    kR16Lds<r16_high_bits(LOGN)> * (A == kF64 ? 2 : 1);

template <int LOGN, int A, int MAXZ, bool SIGNED, bool OPAQUE = false>
__device__ __forceinline__ void ext_item_tile(const ExtItem &a,
                                              const DeviceTables &t,
                                              uint32_t *lds, int tile, int i) {
  constexpr int L = r16_high_bits(LOGN), b = LOGN - L;
  const int64_t n = int64_t(1) << t.log_n;
  const int p = a.moduli_id + i;
  const int tid = OPAQUE ? opaque_tid() : int(threadIdx.x);
  const int c = tid & ((4096 >> L) - 1), r = tid >> (12 - L);
  const int64_t sp = int64_t(tile) * (4096 >> L) + c;
  const int size = a.size;
  const int64_t *dg = a.digits + sp;
  R16Pass s;
  r16_prime<A, false>(s, t, p);
  s.hi = 0;
  s.b = b;
  s.r = r;
  R16Value<A> v[16];
  if constexpr (A == kF64 && !SIGNED) {
    // one digit at a time: sum_j d_j c_j, each product below 0.55 q
    const uint64_t *es =
        reinterpret_cast<const uint64_t *>(a.cst + a.ext_shoup_offset) + 2 * i;
#pragma unroll
    for (int j = 0; j < MAXZ; j++) {
      if (j < size) {
        int64_t d[16];
#pragma unroll
        for (int m = 0; m < 16; m++)
          d[m] =
              dg[int64_t(j) * n + (int64_t(r16_point<L, false>(r, m)) << b)];
        const double cj = double(es[2 * int64_t(j) * a.ext_limbs]);
        // the digits of primes below 2^42 are below their prime but for the
        // first, the input itself, which f64_load looks at; those of larger
        // primes are reduced
        double x[16];
        const bool digit_small =
            t.q[a.moduli_id + a.start + j] < kF64Bound; // block-uniform
        if (j == 0) {
          f64_load(d, x, s.f);
        } else {
#pragma unroll
          for (int m = 0; m < 16; m++)
            x[m] = digit_small ? f64_from_int(d[m]) : f64_from_any(d[m], s.f);
        }
#pragma unroll
        for (int m = 0; m < 16; m++) {
          const double y = f64_mul(x[m], cj, s.f);
          v[m] = j == 0 ? y : v[m] + y;
        }
      }
    }
  } else {
#pragma unroll
    for (int m = 0; m < 16; m++) {
      int64_t d[MAXZ];
#pragma unroll
      for (int j = 0; j < MAXZ; j++)
        d[j] = j < size
                   ? dg[int64_t(j) * n +
                        (int64_t(r16_point<L, false>(r, m)) << b)]
                   : 0;
      int64_t y;
      if (A == kExact || SIGNED)
        y = extend_limb<MAXZ, SIGNED>(d, size, i, a.ext_limbs,
                                      a.cst + CkksParams::kKsExtOffset, s.q,
                                      s.k, s.q2);
      else
        y = extend_limb_lazy<MAXZ>(
            d, size, i, a.ext_limbs,
            reinterpret_cast<const uint64_t *>(a.cst + a.ext_shoup_offset),
            s.q, s.nq, false);
      if constexpr (A == kF64)
        v[m] = f64_from_int(y);
      else
        v[m] = y;
    }
  }
  r16_forward_high<L, A>(v, s);
  if constexpr (A == kF64)
    r16_exchange<L, true>(v, reinterpret_cast<int64_t *>(lds), c, r);
  else
    r16_exchange_words<L, true>(v, lds, c, r);
  r16_forward_low<L, A>(v, s);
  int64_t *out = a.ext + int64_t(i) * n + sp;
#pragma unroll
  for (int m = 0; m < 16; m++)
    out[int64_t(r16_point<L, true>(r, m)) << b] =
        __builtin_bit_cast(int64_t, v[m]);
}

} // namespace fhe
