// Batched negacyclic NTT / INTT for gfx950.
//
// Without lazy arithmetic the butterflies are exactly the reference's radix-2
// formulas (src/operation/ntt.cpp:46-134 Cooley-Tukey, :177-272
// Gentleman-Sande), so every lazy representative in [0, 2q) matches; the lazy
// forms (ntt_r16.h) give other representatives of the same residues, and
// where a zero residue's representative matters its limb is recomputed exactly
// (repair_zero_kernel).  The transform of one limb is split into at most two
// passes over HBM: each pass owns a contiguous range of index bits and runs
// all of that range's radix-2 stages on 4096-element tiles of independent
// sub-transforms, in registers for N = 2^13 .. 2^16 and in LDS otherwise.
//
//   forward  stage s flips index bit log_n-1-s; group of element i uses
//            root[2^s - 1 + (i >> (log_n - s))]
//   inverse  stage t flips bit t; group uses
//            root_inverse[N - N/2^t + (i >> (t + 1))]
//
// A pass covering bits [b, b+L) sees sub-transform elements
//   i = (hi << (b+L)) | (j << b) | lo,   j in [0, 2^L)
// and in both directions the twiddle offset is i >> (b + u + 1) for local bit u.
#include <stdexcept>

#include "kernels.h"
#include "ntt_r16.h"

namespace fhe {

namespace {

constexpr int kTile = 4096; // elements per workgroup (32 KiB of LDS)

struct PassArgs {
  const int64_t *src;
  int64_t *dst;
  int64_t total_subs; // sub-transforms over the whole batch
  int limbs;          // limbs per polynomial: limb f uses prime mid + f % limbs
  int moduli_id;
  int low_bit;        // b
  int bits;           // L <= 12
  const int64_t *pre; // forward first pass: multiply by pre[prime] on load
  int post;           // inverse last pass: InttPost
  int last;           // the pass completes the transform
  bool lazy;          // lazy arithmetic (radix-16 passes only)
  uint32_t *zero;     // LazySpec::zero
  int zero_period;
  // radix-16 passes: polynomials from `split` on are read from src2
  const int64_t *src2 = nullptr;
  int64_t split = 0;
  // radix-16 passes: words between the source's polynomials (0: dense)
  int64_t src_stride = 0;
  PartialSums more = {};
};

template <bool INV>
__global__ __launch_bounds__(kBlock) void ntt_pass_kernel(PassArgs a,
                                                          DeviceTables t) {
  __shared__ int64_t lds[kTile];
  const int log_n = t.log_n;
  const int64_t n = int64_t(1) << log_n;
  const int L = a.bits, b = a.low_bit;
  const int sub = 1 << L;
  const int C = kTile >> L;              // sub-transforms per tile
  const int sub_log = log_n - L;         // log2(sub-transforms per limb)
  const int64_t tile0 = int64_t(blockIdx.x) * C;
  const bool columns = b > 0;            // strided sub-transforms
  const int tid = threadIdx.x;

  // sub-transform sp, element j -> limb-local index i, flat limb f
  auto locate = [&](int64_t sp, int j, int64_t &f) -> int64_t {
    f = sp >> sub_log;
    const int64_t r = sp & ((int64_t(1) << sub_log) - 1);
    const int64_t lo = r & ((int64_t(1) << b) - 1);
    const int64_t hi = r >> b;
    return (hi << (b + L)) | (int64_t(j) << b) | lo;
  };

  for (int e = tid; e < kTile; e += kBlock) {
    const int c = columns ? e % C : e / sub;
    const int j = columns ? e / C : e % sub;
    const int64_t sp = tile0 + c;
    int64_t v = 0;
    if (sp < a.total_subs) {
      int64_t f;
      const int64_t i = locate(sp, j, f);
      v = a.src[f * n + i];
      if (a.pre) {
        const int p = a.moduli_id + int(f % a.limbs);
        v = mont_mult_cs(a.pre[p], v, t.q[p], t.k[p]);
      }
    }
    lds[j * C + c] = v;
  }
  __syncthreads();

  for (int step = 0; step < L; step++) {
    const int u = INV ? step : L - 1 - step;
    for (int bf = tid; bf < kTile / 2; bf += kBlock) {
      const int c = bf % C;
      const int kk = bf / C;
      const int64_t sp = tile0 + c;
      if (sp >= a.total_subs)
        continue;
      const int jl = ((kk >> u) << (u + 1)) | (kk & ((1 << u) - 1));
      const int jh = jl | (1 << u);
      int64_t f;
      const int64_t i = locate(sp, jl, f);
      const int p = a.moduli_id + int(f % a.limbs);
      const int64_t q = int64_t(t.q[p]);
      const int64_t q2 = int64_t(t.q2[p]);
      const uint64_t k = t.k[p];
      const int64_t x = lds[jl * C + c];
      const int64_t y = lds[jh * C + c];
      const int64_t off = i >> (b + u + 1);
      if (!INV) {
        const int s = log_n - 1 - (b + u);
        const int64_t w = t.root[int64_t(p) * n + (int64_t(1) << s) - 1 + off];
        int64_t xa = x, ya = y;
        ct_butterfly(xa, ya, w, q2, q, k);
        lds[jl * C + c] = xa;
        lds[jh * C + c] = ya;
      } else {
        const int tt = b + u;
        const int64_t w =
            t.root_inverse[int64_t(p) * n + n - (n >> tt) + off];
        int64_t xa = x, ya = y;
        gs_butterfly(xa, ya, w, q2, q, k);
        lds[jl * C + c] = xa;
        lds[jh * C + c] = ya;
      }
    }
    __syncthreads();
  }

  for (int e = tid; e < kTile; e += kBlock) {
    const int c = columns ? e % C : e / sub;
    const int j = columns ? e / C : e % sub;
    const int64_t sp = tile0 + c;
    if (sp >= a.total_subs)
      continue;
    int64_t f;
    const int64_t i = locate(sp, j, f);
    int64_t v = lds[j * C + c];
    if (INV && a.post != kInttRaw) {
      const int p = a.moduli_id + int(f % a.limbs);
      const uint64_t q = t.q[p], k = t.k[p];
      v = mont_exit(mont_mult_cs(t.ninv[p], v, q, k), q, k);
      if (a.post != kInttExit)
        v = guard(v, int64_t(q));
    }
    a.dst[f * n + i] = v;
  }
}

// A register-resident L-bit pass (r16_limb_pass, ntt_r16.h) over every limb
// of the batch, exact or lazy with the arithmetic of each limb's prime class
// chosen per block: one launch for the batch (the two lazy forms take about
// the same registers, and a launch for the few large primes of a chain alone
// would run its chain of butterflies on a nearly empty chip).
//
// Block -> (tile, limb l, polynomial), polynomial fastest so blocks sharing
// a tile's twiddles run together; with swizzle each of the 8 XCDs (blocks
// are dealt round-robin to XCDs) gets one contiguous range of that order.
// The tile runs slowest, so that every XCD has its share of the 60-bit
// limbs.
template <int L, bool INV, bool COLS, bool LAZY>
__global__ __launch_bounds__(kBlock) void ntt_radix16_kernel(
    PassArgs a, DeviceTables t, int polys, int swizzle) {
  __shared__ int64_t lds[kR16Lds<L>];
  int64_t w = blockIdx.x;
  if (swizzle) {
    const int64_t per = int64_t(gridDim.x) >> 3;
    w = int64_t(blockIdx.x & 7) * per + (blockIdx.x >> 3);
  }
  const int64_t poly = w % polys;
  const int64_t rest = w / polys;
  const int l = int(rest % a.limbs);
  const int tile = int(rest / a.limbs);
  const int64_t limb = (poly * a.limbs + l) << t.log_n;
  const int64_t *src =
      a.src2 && poly >= a.split
          ? a.src2 + (((poly - a.split) * a.limbs + l) << t.log_n)
      : a.src_stride ? a.src + poly * a.src_stride + (int64_t(l) << t.log_n)
                     : a.src + limb;
  int64_t *dst = a.dst + limb;
  const int p = a.moduli_id + l;
  if constexpr (!LAZY) {
    r16_limb_pass<L, INV, COLS, kExact>(src, dst, p, tile, a.low_bit, a.pre,
                                        a.post, a.last != 0, t, lds);
  } else {
    uint32_t *zero =
        a.zero && poly % a.zero_period == a.zero_period - 1
            ? a.zero + (poly / a.zero_period) * a.limbs + l
            : nullptr;
    const int64_t *more = a.more.data + limb;
    if (t.q[p] < kF64Bound)
      r16_limb_pass<L, INV, COLS, kF64>(src, dst, p, tile, a.low_bit, a.pre,
                                        a.post, a.last != 0, t, lds, zero,
                                        more, a.more.stride, a.more.count);
    else
      r16_limb_pass<L, INV, COLS, kLazyLarge>(src, dst, p, tile, a.low_bit,
                                              a.pre, a.post, a.last != 0, t,
                                              lds, zero, more, a.more.stride,
                                              a.more.count);
  }
}

// Split log_n into the bit ranges of at most two passes (each <= 12 bits),
// the first one's bits first: the high bits of a forward transform, the low
// bits of an inverse one.  The radix-16 sizes use the same two ranges in
// both directions (the fused kernels run the low forward pass and the low
// inverse pass on one tile).
void split_bits(int log_n, bool inverse, int &first, int &second) {
  if (r16_supported(log_n)) {
    first = inverse ? r16_low_bits(log_n) : r16_high_bits(log_n);
    second = log_n - first;
  } else if (log_n <= 12) {
    first = log_n;
    second = 0;
  } else {
    first = log_n / 2;
    second = log_n - first;
  }
}

// One radix-16 pass of L bits (low index bits unless COLS).
template <int L, bool INV, bool COLS>
void launch_r16_pass(const PassArgs &a, const DeviceTables &t,
                     hipStream_t stream) {
  const int64_t total_limbs = a.total_subs >> (t.log_n - L);
  const int polys = int(total_limbs / a.limbs);
  const int tiles = int(int64_t(1) << (t.log_n - 12));
  const int64_t blocks = total_limbs * tiles;
  const int swizzle = blocks % 8 == 0 ? 1 : 0;
  // the lazy forms hand doubles or values up to 8q to the other pass, so both
  // have to be lazy: the 8-bit pass of N = 2^17, whose other pass is the
  // generic exact one, stays exact
  if (a.lazy && r16_supported(t.log_n))
    hipLaunchKernelGGL((ntt_radix16_kernel<L, INV, COLS, true>),
                       dim3(unsigned(blocks)), dim3(kBlock), 0, stream, a, t,
                       polys, swizzle);
  else
    hipLaunchKernelGGL((ntt_radix16_kernel<L, INV, COLS, false>),
                       dim3(unsigned(blocks)), dim3(kBlock), 0, stream, a, t,
                       polys, swizzle);
}

template <bool INV>
void launch_pass(const PassArgs &a, const DeviceTables &t,
                 hipStream_t stream) {
  const bool cols = a.low_bit > 0;
  if (t.log_n >= 13 && a.bits == 8) {
    if (cols)
      launch_r16_pass<8, INV, true>(a, t, stream);
    else
      launch_r16_pass<8, INV, false>(a, t, stream);
    return;
  }
  if (t.log_n >= 13 && a.bits == 7) {
    if (cols)
      launch_r16_pass<7, INV, true>(a, t, stream);
    else
      launch_r16_pass<7, INV, false>(a, t, stream);
    return;
  }
  if (t.log_n >= 13 && a.bits == 6 && cols) {
    launch_r16_pass<6, INV, true>(a, t, stream);
    return;
  }
  const int C = kTile >> a.bits;
  const unsigned blocks = unsigned((a.total_subs + C - 1) / C);
  hipLaunchKernelGGL(ntt_pass_kernel<INV>, dim3(blocks), dim3(kBlock), 0,
                     stream, a, t);
}

} // namespace

void ntt_forward(const DeviceTables &t, const int64_t *src, int64_t *dst,
                 int64_t total_limbs, int limbs, int moduli_id,
                 const int64_t *pre, hipStream_t stream, LazySpec lazy) {
  int l1, l2;
  split_bits(t.log_n, false, l1, l2);
  // first pass: the high bits (stages 0 .. l1-1)
  PassArgs a{src,     dst,      total_limbs << (t.log_n - l1),
             limbs,   moduli_id, t.log_n - l1,
             l1,      pre,       kInttRaw,
             l2 == 0, lazy.on, lazy.zero, lazy.zero_period};
  launch_pass<false>(a, t, stream);
  if (l2 > 0) {
    PassArgs b2{dst,   dst,      total_limbs << (t.log_n - l2),
                limbs, moduli_id, 0,
                l2,    nullptr,   kInttRaw,
                1,     lazy.on, lazy.zero, lazy.zero_period};
    launch_pass<false>(b2, t, stream);
  }
}

bool ntt_forward_strided(const DeviceTables &t, const int64_t *src,
                         int64_t src_stride, int64_t *dst, int64_t polys,
                         int limbs, int moduli_id, const int64_t *pre,
                         hipStream_t stream) {
  if (!r16_supported(t.log_n))
    return false;
  int l1, l2;
  split_bits(t.log_n, false, l1, l2);
  PassArgs a{src,     dst,       (polys * limbs) << (t.log_n - l1),
             limbs,   moduli_id, t.log_n - l1,
             l1,      pre,       kInttRaw,
             0,       false,     nullptr,
             1};
  a.src_stride = src_stride;
  launch_pass<false>(a, t, stream);
  ntt_forward_second(t, dst, dst, polys * limbs, limbs, moduli_id, stream);
  return true;
}

void ntt_forward_pair(const DeviceTables &t, const int64_t *x,
                      const int64_t *y, int64_t *dst, int64_t total_limbs,
                      int limbs, int moduli_id, const int64_t *pre,
                      hipStream_t stream, LazySpec lazy) {
  if (!r16_supported(t.log_n)) {
    ntt_forward(t, x, dst, total_limbs, limbs, moduli_id, pre, stream, lazy);
    ntt_forward(t, y, dst + (total_limbs << t.log_n), total_limbs, limbs,
                moduli_id, pre, stream, lazy);
    return;
  }
  int l1, l2;
  split_bits(t.log_n, false, l1, l2);
  PassArgs a{x,       dst,       (2 * total_limbs) << (t.log_n - l1),
             limbs,   moduli_id, t.log_n - l1,
             l1,      pre,       kInttRaw,
             0,       lazy.on,   lazy.zero,
             lazy.zero_period,   y,
             total_limbs / limbs};
  launch_pass<false>(a, t, stream);
  PassArgs b{dst,   dst,       (2 * total_limbs) << (t.log_n - l2),
             limbs, moduli_id, 0,
             l2,    nullptr,   kInttRaw,
             1,     lazy.on,   lazy.zero,
             lazy.zero_period};
  launch_pass<false>(b, t, stream);
}

void ntt_inverse(const DeviceTables &t, const int64_t *src, int64_t *dst,
                 int64_t total_limbs, int limbs, int moduli_id, int post,
                 hipStream_t stream, LazySpec lazy) {
  int l1, l2;
  split_bits(t.log_n, true, l1, l2);
  // first pass: the low bits (stages with span 1 .. 2^(l1-1))
  PassArgs a{src,     dst,      total_limbs << (t.log_n - l1),
             limbs,   moduli_id, 0,
             l1,      nullptr,   l2 > 0 ? int(kInttRaw) : post,
             l2 == 0, lazy.on, lazy.zero, lazy.zero_period};
  launch_pass<true>(a, t, stream);
  if (l2 > 0) {
    PassArgs b2{dst,   dst,      total_limbs << (t.log_n - l2),
                limbs, moduli_id, l1,
                l2,    nullptr,   post,
                1,     lazy.on, lazy.zero, lazy.zero_period};
    launch_pass<true>(b2, t, stream);
  }
}

void ntt_forward_first(const DeviceTables &t, const int64_t *src, int64_t *dst,
                       int64_t total_limbs, int limbs, int moduli_id,
                       const int64_t *pre, hipStream_t stream,
                       LazySpec lazy) {
  int l1, l2;
  split_bits(t.log_n, false, l1, l2);
  PassArgs a{src,     dst,      total_limbs << (t.log_n - l1),
             limbs,   moduli_id, t.log_n - l1,
             l1,      pre,       kInttRaw,
             l2 == 0, lazy.on, lazy.zero, lazy.zero_period};
  launch_pass<false>(a, t, stream);
}

void ntt_forward_second(const DeviceTables &t, const int64_t *src,
                        int64_t *dst, int64_t total_limbs, int limbs,
                        int moduli_id, hipStream_t stream, LazySpec lazy) {
  int l1, l2;
  split_bits(t.log_n, false, l1, l2);
  if (l2 == 0) {
    // single-pass sizes: the first pass was the whole transform
    if (src != dst)
      (void)hipMemcpyAsync(dst, src, size_t(total_limbs << t.log_n) * 8,
                           hipMemcpyDeviceToDevice, stream);
    return;
  }
  PassArgs b2{src,   dst,      total_limbs << (t.log_n - l2),
              limbs, moduli_id, 0,
              l2,    nullptr,   kInttRaw,
              1,     lazy.on, lazy.zero, lazy.zero_period};
  launch_pass<false>(b2, t, stream);
}

void ntt_inverse_second(const DeviceTables &t, const int64_t *src,
                        int64_t *dst, int64_t total_limbs, int limbs,
                        int moduli_id, int post, hipStream_t stream,
                        LazySpec lazy, PartialSums more) {
  int l1, l2;
  split_bits(t.log_n, true, l1, l2);
  PassArgs a{src,   dst,      total_limbs << (t.log_n - l2),
             limbs, moduli_id, l1,
             l2,    nullptr,   post,
             1,     lazy.on, lazy.zero, lazy.zero_period};
  a.more = more;
  launch_pass<true>(a, t, stream);
}

namespace {

// Recomputation of flagged limbs with the reference's exact arithmetic: one
// block per (ciphertext, limb), which leaves at once where the flag is clear
// (the rule: a zero residue comes up once in 2^40 coefficients).  The block
// walks the limb's tiles pass by pass; its own stores of one pass are what
// it reads in the next, behind a block barrier.  bound: latency of the
// launch, 5 us for 800 limbs; a flagged limb takes about 0.2 ms.
struct RepairArgs {
  const uint32_t *zero; // [count][limbs]
  // the NTT-form source polynomial of ciphertext c at z + c * z_stride, or,
  // where a is set, the product of the transforms of a and b (polynomial 1
  // of INTT-form duos, or NTT-form ones), formed in the scratch limbs
  const int64_t *z;
  int64_t z_stride;
  const int64_t *a, *b;
  int a_ntt, b_ntt;
  int64_t *scratch;     // [2][count][limbs][N]
  int64_t *out;         // [limbs][N] of ciphertext c at out + c * out_stride
  int64_t out_stride;
  int count, limbs, moduli_id;
};

template <int LOGN>
__device__ __forceinline__ bool all_zero(const int64_t *x) {
  int any = 0;
  for (int j = threadIdx.x; j < (1 << LOGN); j += kBlock)
    any |= x[j] != 0;
  return !__syncthreads_or(any);
}

template <int LOGN>
__global__ __launch_bounds__(kBlock) void repair_zero_kernel(RepairArgs a,
                                                             DeviceTables t) {
  constexpr int LO = r16_low_bits(LOGN), HI = r16_high_bits(LOGN);
  constexpr int tiles = 1 << (LOGN - 12);
  constexpr int64_t n = int64_t(1) << LOGN;
  __shared__ int64_t
      lds[kR16Lds<LO> > kR16Lds<HI> ? kR16Lds<LO> : kR16Lds<HI>];
  if (a.zero[blockIdx.x] == 0)
    return;
  const int c = int(blockIdx.x) / a.limbs, l = int(blockIdx.x) % a.limbs;
  const int p = a.moduli_id + l;
  int64_t *out = a.out + c * a.out_stride + int64_t(l) * n;
  const int64_t *z;
  if (a.a) {
    const int64_t *x[2];
    bool zero = false;
    int64_t *mine = nullptr;
    for (int k = 0; k < 2; k++) {
      const int64_t *in = (k ? a.b : a.a) +
                          ((int64_t(2) * c + 1) * a.limbs + l) * n;
      zero = zero || all_zero<LOGN>(in);
      x[k] = in;
      mine = a.scratch +
             ((int64_t(k) * a.count + c) * a.limbs + l) * n;
      if (k ? a.b_ntt : a.a_ntt)
        continue;
      x[k] = mine;
      for (int tile = 0; tile < tiles; tile++)
        r16_limb_pass<HI, false, true, kExact>(in, mine, p, tile, LO, t.r2,
                                               kInttRaw, false, t, lds);
      __syncthreads();
      for (int tile = 0; tile < tiles; tile++)
        r16_limb_pass<LO, false, false, kExact>(mine, mine, p, tile, 0,
                                                nullptr, kInttRaw, true, t,
                                                lds);
      __syncthreads();
    }
    // an all-zero factor gives an all-zero product and inverse
    if (zero) {
      for (int j = threadIdx.x; j < n; j += kBlock)
        out[j] = 0;
      return;
    }
    // the exact transforms of signed inputs may hold negative values
    for (int j = threadIdx.x; j < n; j += kBlock)
      mine[j] = mont_mult(x[0][j], x[1][j], t.q[p], t.k[p]);
    __syncthreads();
    z = mine;
  } else {
    z = a.z + c * a.z_stride + int64_t(l) * n;
  }
  for (int tile = 0; tile < tiles; tile++)
    r16_limb_pass<LO, true, false, kExact>(z, out, p, tile, 0, nullptr,
                                           kInttRaw, false, t, lds);
  __syncthreads();
  for (int tile = 0; tile < tiles; tile++)
    r16_limb_pass<HI, true, true, kExact>(out, out, p, tile, LO, nullptr,
                                          kInttExit, true, t, lds);
}

void launch_repair(const DeviceTables &t, const RepairArgs &a,
                   hipStream_t stream) {
  with_log_n(t.log_n, [&](auto logn) {
    hipLaunchKernelGGL(repair_zero_kernel<decltype(logn)::value>,
                       dim3(unsigned(a.count * a.limbs)), dim3(kBlock), 0,
                       stream, a, t);
  });
}

} // namespace

void launch_repair_intt(const DeviceTables &t, const uint32_t *zero,
                        const int64_t *z, int64_t z_stride, int64_t *out,
                        int64_t out_stride, int count, int limbs,
                        int moduli_id, hipStream_t stream) {
  RepairArgs a{};
  a.zero = zero;
  a.z = z;
  a.z_stride = z_stride;
  a.out = out;
  a.out_stride = out_stride;
  a.count = count;
  a.limbs = limbs;
  a.moduli_id = moduli_id;
  launch_repair(t, a, stream);
}

void launch_repair_product(const DeviceTables &t, const uint32_t *zero,
                           const int64_t *x, bool x_ntt, const int64_t *y,
                           bool y_ntt, int64_t *scratch, int64_t *out,
                           int64_t out_stride, int count, int limbs,
                           int moduli_id, hipStream_t stream) {
  RepairArgs a{};
  a.zero = zero;
  a.a = x;
  a.b = y;
  a.a_ntt = x_ntt;
  a.b_ntt = y_ntt;
  a.scratch = scratch;
  a.out = out;
  a.out_stride = out_stride;
  a.count = count;
  a.limbs = limbs;
  a.moduli_id = moduli_id;
  launch_repair(t, a, stream);
}

} // namespace fhe
