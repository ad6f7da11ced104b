// Fused key-switching core for N = 2^13 .. 2^16 (two radix-16 NTT passes).
//
// The reference (src/ckks/core_key_switch.cpp:293-358, :110-160) runs, per
// partition, a full NTT of the extended polynomial, two Montgomery
// products with the key and an accumulate, and then a full INTT of both
// accumulators.  Here one workgroup owns a 4096-coefficient tile of one
// extended limb of one ciphertext and, for every partition in turn,
// finishes the forward NTT of that tile (the high-bit pass ran before),
// multiplies by both key halves and accumulates in registers; it then runs
// the first (low-bit) pass of the inverse NTT on both accumulators before a
// single write.  With lazy = false each coefficient sees the reference's exact
// sequence of butterflies, products and guards; the lazy forms (ntt_r16.h),
// partial sums and transforms taken from the source's NTT form keep the
// residues only, which is what the canonical accumulators depend on.
#include <algorithm>

#include "kernels.h"
#include "ks_tile.h"

namespace fhe {

namespace {

// Block -> (tile, limb i, ciphertext), ciphertext fastest: the blocks of a
// key tile run together and share its reads through L2; with swizzle each of
// the 8 XCDs (blocks are dealt round-robin to XCDs) gets one contiguous
// range of that order.  The tile runs slowest, so that every XCD has its
// share of the 60-bit limbs, whose items take about three times as long.
template <int LOGN, class F>
__device__ __forceinline__ void ks_block(const KsArgs &a, F &&item) {
  int64_t w = blockIdx.x;
  if (a.swizzle) {
    const int64_t per = int64_t(gridDim.x) >> 3;
    w = int64_t(blockIdx.x & 7) * per + (blockIdx.x >> 3);
  }
  const int ct = int(w % a.count);
  int64_t rest = w / a.count;
  const int sub = int(rest % (a.groups * a.halves));
  rest /= a.groups * a.halves;
  const int group = sub / a.halves;
  // partitions [p0, p1) of the group
  const int p0 = group * a.parts / a.groups;
  const int p1 = (group + 1) * a.parts / a.groups;
  item(KsBatchAddr<LOGN>(a, ct, group), int(rest / a.limbs_here),
       a.limb0 + int(rest % a.limbs_here), p0, p1, sub % a.halves);
}

// One arithmetic per launch, over a run of extended limbs of its class.  Two
// waves per SIMD: with three the kF64 form keeps part of its accumulators in
// scratch memory (32 Gold HMults 8.04 against 7.60 ms).
template <int LOGN, int A>
__global__ __launch_bounds__(kBlock, 2) void ks_inner_product_r16_kernel(
    KsArgs a, DeviceTables t) {
  __shared__ int64_t lds[kR16Lds<r16_low_bits(LOGN)>];
  ks_block<LOGN>(a, [&](const auto &ad, int tile, int i, int p0, int p1,
                        int half) {
    ks_item_tile<LOGN, A, true>(ad, t, lds, tile, i, p0, p1, half);
  });
}

// The lazy arithmetic of each limb's class chosen per block: one launch for
// all limbs.  BOTH: both key halves per block.
template <int LOGN, bool BOTH>
__global__ __launch_bounds__(kBlock, 2) void ks_inner_product_mixed_kernel(
    KsArgs a, DeviceTables t) {
  __shared__ int64_t lds[kR16Lds<r16_low_bits(LOGN)>];
  ks_block<LOGN>(a, [&](const auto &ad, int tile, int i, int p0, int p1,
                        int half) {
    if (t.q[a.moduli_id + i] < kF64Bound)
      ks_item_tile<LOGN, kF64, BOTH>(ad, t, lds, tile, i, p0, p1, half);
    else
      ks_item_tile<LOGN, kLazyLarge, BOTH>(ad, t, lds, tile, i, p0, p1, half);
  });
}

// ---------------------------------------------------------------------------
// ModUp in two stages around HBM: the Garner digits of every partition
// (MAXZ limbs per partition, far fewer than the extended limbs), then one
// kernel that forms each extended limb from the digits and runs the first
// (high-bit) forward NTT pass on it before its only write.  The 4096-
// coefficient digit tile of a block is re-read by the blocks of the other
// extended limbs; the limb index runs fastest in the block order so those
// reads hit the XCD's L2.
struct DigitArgs {
  const int64_t *x;   // source polynomial of ciphertext c at x + c * x_stride
  int64_t x_stride;
  int64_t *digits;    // [count][parts][MAXZ][N]
  const int64_t *cst;
  int cst_stride;
  int count, parts, moduli_id, maxz;
  int start[kMaxFusedParts];
  int size[kMaxFusedParts];
  uint32_t signed_mask;
};

template <int MAXZ>
__global__ __launch_bounds__(kBlock) void modup_digits_kernel(DigitArgs a,
                                                             DeviceTables t) {
  const int64_t n = int64_t(1) << t.log_n;
  const int64_t idx = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (idx >= int64_t(a.count) * a.parts * n)
    return;
  const int64_t coef = idx & (n - 1);
  const int64_t cp = idx >> t.log_n; // ciphertext * parts + partition
  const int part = int(cp % a.parts);
  const int64_t ct = cp / a.parts;
  const int start = a.start[part], size = a.size[part];
  const int64_t *xs = a.x + ct * a.x_stride + coef;
  const int64_t *cst = a.cst + int64_t(part) * a.cst_stride;
  int64_t xv[MAXZ], d[MAXZ];
#pragma unroll
  for (int j = 0; j < MAXZ; j++)
    xv[j] = j < size ? xs[int64_t(start + j) * n] : 0;
  if ((a.signed_mask >> part) & 1)
    garner_digits<MAXZ, true>(xv, d, size, a.moduli_id + start, cst, t);
  else
    garner_digits<MAXZ, false>(xv, d, size, a.moduli_id + start, cst, t);
  int64_t *out = a.digits + cp * MAXZ * n + coef;
#pragma unroll
  for (int j = 0; j < MAXZ; j++)
    if (j < size)
      out[int64_t(j) * n] = d[j];
}

// modup_digits_kernel over kChunk coefficients of one (ciphertext,
// partition) per block (chunked_ok): four independent Garner chains per
// thread.  A partition's limbs past its size are loaded again as its last
// limb and unused, so that every load is unconditional.
template <int MAXZ>
__global__ __launch_bounds__(kBlock) void modup_digits_chunk_kernel(
    DigitArgs a, DeviceTables t) {
  const int64_t n = int64_t(1) << t.log_n;
  const int64_t e0 = int64_t(blockIdx.x) * kChunk;
  const uint32_t cp = uint32_t(e0 >> t.log_n); // ciphertext * parts + part
  const int part = int(cp % uint32_t(a.parts));
  const int64_t ct = cp / uint32_t(a.parts);
  const int64_t coef = (e0 & (n - 1)) + int64_t(threadIdx.x) * kPerThread;
  const int start = a.start[part], size = a.size[part];
  const int64_t *xs = a.x + ct * a.x_stride + coef;
  const int64_t *cst = a.cst + int64_t(part) * a.cst_stride;
  int64_t xv[kPerThread][MAXZ], d[kPerThread][MAXZ];
#pragma unroll
  for (int j = 0; j < MAXZ; j++) {
    int64_t v[kPerThread];
    load4(xs + int64_t(start + min(j, size - 1)) * n, v);
#pragma unroll
    for (int g = 0; g < kPerThread; g++)
      xv[g][j] = j < size ? v[g] : 0;
  }
  if ((a.signed_mask >> part) & 1) {
#pragma unroll
    for (int g = 0; g < kPerThread; g++)
      garner_digits<MAXZ, true>(xv[g], d[g], size, a.moduli_id + start, cst,
                                t);
  } else {
#pragma unroll
    for (int g = 0; g < kPerThread; g++)
      garner_digits<MAXZ, false>(xv[g], d[g], size, a.moduli_id + start, cst,
                                 t);
  }
  int64_t *out = a.digits + int64_t(cp) * MAXZ * n + coef;
#pragma unroll
  for (int j = 0; j < MAXZ; j++)
    if (j < size) {
      int64_t v[kPerThread];
#pragma unroll
      for (int g = 0; g < kPerThread; g++)
        v[g] = d[g][j];
      store4(out + int64_t(j) * n, v);
    }
}

struct ExtendArgs {
  const int64_t *digits; // [count][parts][maxz][N]
  int64_t *ext;          // [count][parts][ext_limbs][N]
  const int64_t *cst;
  int cst_stride, ext_shoup_offset;
  int count, parts, ext_limbs, moduli_id, maxz, swizzle;
  int size[kMaxFusedParts];
  int start[kMaxFusedParts];
  int limb0, limbs_here; // the launch's extended limbs
  int skip_own;          // leave each partition's own limbs unwritten
  uint32_t signed_mask;
};

template <int LOGN, int A, int MAXZ, bool SIGNED>
__device__ __forceinline__ void extend_ntt_tile(const ExtendArgs &a,
                                                const DeviceTables &t,
                                                uint32_t *lds, int64_t cp,
                                                int part, int tile, int i) {
  constexpr int64_t n = int64_t(1) << LOGN;
  ExtItem it;
  it.digits = a.digits + cp * a.maxz * n;
  it.cst = a.cst + int64_t(part) * a.cst_stride;
  it.ext = a.ext + cp * a.ext_limbs * n;
  it.start = a.start[part];
  it.size = a.size[part];
  it.ext_limbs = a.ext_limbs;
  it.moduli_id = a.moduli_id;
  it.ext_shoup_offset = a.ext_shoup_offset;
  ext_item_tile<LOGN, A, MAXZ, SIGNED>(it, t, lds, tile, i);
}

// Block -> (extended limb, tile, ciphertext and partition), the limb
// fastest: the 4096-coefficient digit tile is re-read by the blocks of the
// other limbs through the XCD's L2.
template <int LOGN, class F>
__device__ __forceinline__ void extend_block(const ExtendArgs &a, F &&item) {
  constexpr int tiles = 1 << (LOGN - 12);
  int64_t w = blockIdx.x;
  if (a.swizzle) {
    const int64_t per = int64_t(gridDim.x) >> 3;
    w = int64_t(blockIdx.x & 7) * per + (blockIdx.x >> 3);
  }
  const int i = a.limb0 + int(w % a.limbs_here);
  const int64_t rest = w / a.limbs_here;
  const int tile = int(rest % tiles);
  const int64_t cp = rest / tiles;
  const int part = int(cp % a.parts);
  // the whole block leaves (before any barrier) for a partition's own limb
  if (a.skip_own && i >= a.start[part] && i < a.start[part] + a.size[part])
    return;
  item(cp, part, tile, i);
}

// One lazy arithmetic per launch, over a run of extended limbs of its class
// (no signed partitions).
template <int LOGN, int MAXZ, int A>
__global__ __launch_bounds__(kBlock, A == kF64 || MAXZ > 4 ? 4 : 6)
void extend_ntt_r16_kernel(ExtendArgs a, DeviceTables t) {
  __shared__ __align__(8) uint32_t lds[kExtendLds<LOGN, A>];
  extend_block<LOGN>(a, [&](int64_t cp, int part, int tile, int i) {
    extend_ntt_tile<LOGN, A, MAXZ, false>(a, t, lds, cp, part, tile, i);
  });
}

// The arithmetic chosen per block: signed digits take the exact extension,
// and the transform after it may be lazy all the same.
template <int LOGN, int MAXZ, bool LAZY>
__global__ __launch_bounds__(kBlock) void extend_ntt_mixed_kernel(
    ExtendArgs a, DeviceTables t) {
  __shared__ __align__(8) uint32_t lds[kExtendLds<LOGN, kF64>];
  extend_block<LOGN>(a, [&](int64_t cp, int part, int tile, int i) {
    const bool sgn = (a.signed_mask >> part) & 1;
    const bool small = t.q[a.moduli_id + i] < kF64Bound;
    if (LAZY && small) {
      if (sgn)
        extend_ntt_tile<LOGN, kF64, MAXZ, true>(a, t, lds, cp, part, tile, i);
      else
        extend_ntt_tile<LOGN, kF64, MAXZ, false>(a, t, lds, cp, part, tile, i);
    } else if (sgn) {
      extend_ntt_tile<LOGN, kExact, MAXZ, true>(a, t, lds, cp, part, tile, i);
    } else if (LAZY) {
      extend_ntt_tile<LOGN, kLazyLarge, MAXZ, false>(a, t, lds, cp, part,
                                                     tile, i);
    } else {
      extend_ntt_tile<LOGN, kExact, MAXZ, false>(a, t, lds, cp, part, tile, i);
    }
  });
}

// Calls f(first limb, limbs, small) for each run of extended limbs of one
// prime class.
template <class F>
void for_class_runs(const DeviceTables &t, int moduli_id, int limbs, F &&f) {
  for (int l = 0; l < limbs;) {
    const bool small = t_host_q_small(t, moduli_id + l);
    int e = l + 1;
    while (e < limbs && t_host_q_small(t, moduli_id + e) == small)
      e++;
    f(l, e - l, small);
    l = e;
  }
}

// Launches with fewer blocks than this choose the arithmetic per block (four
// blocks per CU: above it the extra waves of the smaller extension kernel have
// work, and the key product's FP64 blocks do not carry the 64-bit form's code
// and registers).  One launch per class against one mixed launch, both
// kernels together and before the key product's range checks: 8.28 against
// 11.27 ms for 32 Gold HMults (14848 blocks), 1020 against 1183 us for 8 at
// N = 2^15 (1280); below, the second launch would wait for the last blocks of
// the first.
constexpr int64_t kSplitBlocks = 1024;

} // namespace

bool ks_fused_supported(const DeviceTables &t) {
  return r16_supported(t.log_n);
}

bool staged_modup_supported(const DeviceTables &t, int max_partition_size,
                            int parts) {
  return r16_supported(t.log_n) && max_partition_size <= 8 &&
         parts <= kMaxFusedParts;
}

void launch_staged_modup(const DeviceTables &t, const int64_t *x,
                         int64_t x_stride, int64_t *digits, int64_t *ext,
                         int count, int limbs, int moduli_id,
                         const int *starts, const int *sizes,
                         const bool *is_signed, int parts,
                         const int64_t *constants, int constants_stride,
                         int ext_shoup_offset, bool lazy, bool skip_own,
                         hipStream_t stream) {
  int maxz = 1;
  uint32_t mask = 0;
  for (int p = 0; p < parts; p++) {
    while (maxz < sizes[p])
      maxz <<= 1;
    mask |= is_signed[p] ? (uint32_t(1) << p) : 0u;
  }
  DigitArgs d{};
  d.x = x;
  d.x_stride = x_stride;
  d.digits = digits;
  d.cst = constants;
  d.cst_stride = constants_stride;
  d.count = count;
  d.parts = parts;
  d.moduli_id = moduli_id;
  d.maxz = maxz;
  d.signed_mask = mask;
  ExtendArgs e{};
  e.digits = digits;
  e.ext = ext;
  e.cst = constants;
  e.cst_stride = constants_stride;
  e.ext_shoup_offset = ext_shoup_offset;
  e.count = count;
  e.parts = parts;
  e.ext_limbs = limbs + t.alpha;
  e.moduli_id = moduli_id;
  e.maxz = maxz;
  e.signed_mask = mask;
  e.skip_own = skip_own ? 1 : 0;
  for (int p = 0; p < parts; p++) {
    d.start[p] = starts[p];
    d.size[p] = sizes[p];
    e.size[p] = sizes[p];
    e.start[p] = starts[p];
  }
  const int tiles = int((int64_t(1) << t.log_n) >> 12);
  const int64_t per_limb = int64_t(count) * parts * tiles;
  const dim3 dgrid(grid_for((int64_t(count) * parts) << t.log_n));
  const bool chunked = chunked_ok(t.log_n, {x, digits}) && x_stride % 2 == 0;
  // the extensions of the limbs [l, l + n): small per class, or mixed (-1)
  auto extend = [&](auto logn, auto width, int l, int n, int small) {
    constexpr int LOGN = decltype(logn)::value, W = decltype(width)::value;
    e.limb0 = l;
    e.limbs_here = n;
    const int64_t blocks = per_limb * n;
    e.swizzle = blocks % 8 == 0 ? 1 : 0;
    const dim3 grid{unsigned(blocks), 1, 1};
    if (small == 1)
      hipLaunchKernelGGL((extend_ntt_r16_kernel<LOGN, W, kF64>), grid,
                         dim3(kBlock), 0, stream, e, t);
    else if (small == 0)
      hipLaunchKernelGGL((extend_ntt_r16_kernel<LOGN, W, kLazyLarge>), grid,
                         dim3(kBlock), 0, stream, e, t);
    else if (lazy)
      hipLaunchKernelGGL((extend_ntt_mixed_kernel<LOGN, W, true>), grid,
                         dim3(kBlock), 0, stream, e, t);
    else
      hipLaunchKernelGGL((extend_ntt_mixed_kernel<LOGN, W, false>), grid,
                         dim3(kBlock), 0, stream, e, t);
  };
  auto staged = [&](auto logn, auto width) {
    constexpr int W = decltype(width)::value;
    if (chunked)
      hipLaunchKernelGGL(
          modup_digits_chunk_kernel<W>,
          dim3(unsigned(((int64_t(count) * parts) << t.log_n) / kChunk)),
          dim3(kBlock), 0, stream, d, t);
    else
      hipLaunchKernelGGL(modup_digits_kernel<W>, dgrid, dim3(kBlock), 0,
                         stream, d, t);
    if (lazy && mask == 0 && per_limb * e.ext_limbs >= kSplitBlocks)
      for_class_runs(t, moduli_id, e.ext_limbs, [&](int l, int n, bool small) {
        extend(logn, width, l, n, small ? 1 : 0);
      });
    else
      extend(logn, width, 0, e.ext_limbs, -1);
  };
  with_log_n(t.log_n, [&](auto logn) {
    if (maxz == 1)
      staged(logn, std::integral_constant<int, 1>());
    else if (maxz == 2)
      staged(logn, std::integral_constant<int, 2>());
    else if (maxz == 4)
      staged(logn, std::integral_constant<int, 4>());
    else
      staged(logn, std::integral_constant<int, 8>());
  });
}

// A batch whose items fill fewer blocks than there are CUs is split further:
// the partitions into groups until they do, and, where even that leaves most
// of the chip idle, one block per key half.  The line is at one block per CU
// (measured per launch sequence: N = 2^14, 36 blocks, 142 -> 109 us; N = 2^16,
// 464 blocks, 423 -> 468 us with three groups, whose sums then cost more than
// the idle slots did).
constexpr int64_t kSplitTarget = 256;

// The second inverse pass adds the groups' kF64 values as they are, each below
// 2^8 (q / 2 + 2) after eight stages from centred sums: integers below 2^53.
// (kLazyLarge sums are brought below 4q at every step.)
static_assert(uint64_t(kKsMaxGroups) * 256 * (kF64Bound / 2 + 2) <
                  uint64_t(1) << 53,
              "the partial sums must stay exact in doubles");

KsSplit ks_split(const DeviceTables &t, int parts, int count, int ext_limbs,
                 bool lazy) {
  const int64_t blocks = (int64_t(ext_limbs) * count) << (t.log_n - 12);
  KsSplit s;
  if (!lazy || blocks >= kSplitTarget)
    return s;
  s.groups = int(std::min<int64_t>(std::min(parts, kKsMaxGroups),
                                   (kSplitTarget + blocks - 1) / blocks));
  s.halves = blocks * s.groups <= kSplitTarget ? 2 : 1;
  return s;
}

void launch_ks_inner_product_fused(const DeviceTables &t, const int64_t *ext,
                                   const int64_t *key, int key_chain,
                                   int key_offset, int key_partition0,
                                   int parts, int64_t *acc, int count,
                                   int ext_limbs, int moduli_id, bool lazy,
                                   const int64_t *own, int64_t own_stride,
                                   const int *starts, const int *sizes,
                                   bool lazy_accumulate, const KsSplit &split,
                                   int64_t *partials, hipStream_t stream) {
  const int tiles = int((int64_t(1) << t.log_n) >> 12);
  const int64_t blocks = int64_t(ext_limbs) * tiles * count;
  KsArgs a{};
  a.ext = ext;
  a.key = key;
  a.acc = acc;
  a.count = count;
  a.parts = parts;
  a.ext_limbs = ext_limbs;
  a.moduli_id = moduli_id;
  a.key_chain = key_chain;
  a.key_offset = key_offset;
  a.key_partition0 = key_partition0;
  a.own = own;
  a.own_stride = own_stride;
  a.lazy_acc = lazy_accumulate ? 1 : 0;
  a.groups = split.groups;
  a.halves = split.halves;
  a.partials = partials;
  for (int p = 0; p < parts && p < kMaxFusedParts; p++) {
    a.start[p] = own ? starts[p] : 0;
    a.size[p] = own ? sizes[p] : 0;
  }
  with_log_n(t.log_n, [&](auto logn) {
    constexpr int LOGN = decltype(logn)::value;
    auto launch = [&](auto *kernel, int l, int n) {
      a.limb0 = l;
      a.limbs_here = n;
      const int64_t b = blocks / ext_limbs * n * a.groups * a.halves;
      a.swizzle = b % 8 == 0 ? 1 : 0;
      hipLaunchKernelGGL(kernel, dim3(unsigned(b)), dim3(kBlock), 0, stream, a,
                         t);
    };
    if (!lazy)
      launch(ks_inner_product_r16_kernel<LOGN, kExact>, 0, ext_limbs);
    else if (blocks < kSplitBlocks && split.halves == 2)
      launch(ks_inner_product_mixed_kernel<LOGN, false>, 0, ext_limbs);
    else if (blocks < kSplitBlocks)
      launch(ks_inner_product_mixed_kernel<LOGN, true>, 0, ext_limbs);
    else
      for_class_runs(t, moduli_id, ext_limbs, [&](int l, int n, bool small) {
        if (small)
          launch(ks_inner_product_r16_kernel<LOGN, kF64>, l, n);
        else
          launch(ks_inner_product_r16_kernel<LOGN, kLazyLarge>, l, n);
      });
  });
}

} // namespace fhe
