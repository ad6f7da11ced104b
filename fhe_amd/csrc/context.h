// fhe_context: device-resident CKKS parameters, tables, workspace and the
// key-switching pipelines shared by the C ABI's source files (context.hip:
// context, memory, transforms and the metric's pipeline; engine.hip: the
// engine-level compositions and the bootstrap; batch.hip: mixed-level
// batches; wire.hip: the wire format).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <complex>
#include <tuple>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

#include "fhe_amd.h"
#include "kernels.h"
#include "params.h"

namespace fhe_host {

// the calling thread's last error message (fhe_last_error)
extern thread_local std::string g_last_error;

struct FheError : std::runtime_error {
  int code;
  FheError(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

inline void hip_check(hipError_t e, const char *what) {
  if (e == hipErrorOutOfMemory)
    throw FheError(FHE_ERR_OUT_OF_MEMORY, std::string(what) + ": out of memory");
  if (e != hipSuccess)
    throw FheError(FHE_ERR_DEVICE,
                   std::string(what) + ": " + hipGetErrorString(e));
}

inline void require(bool ok, const std::string &message) {
  if (!ok)
    throw FheError(FHE_ERR_INVALID, message);
}

// Exponent g of the automorphism X -> X^g for a rotation by delta slots:
// 5^-delta mod 2N, or -1 for conjugation (delta = -1 mod 2N); the
// reference's get_jump (src/ckks/encode.cpp:513-526).
inline uint32_t automorphism_exponent(int log_n, int delta) {
  const int64_t two_n = int64_t(2) << log_n;
  const int64_t shift = ((int64_t(delta) % two_n) + two_n) % two_n;
  if (shift == two_n - 1)
    return uint32_t(shift);
  int64_t g = 1, b = 5;
  for (int64_t e = two_n - shift; e > 0; e >>= 1) {
    if (e & 1)
      g = (g * b) & (two_n - 1);
    b = (b * b) & (two_n - 1);
  }
  return uint32_t(g);
}

template <class F> int guarded(F &&f) {
  try {
    f();
    return FHE_OK;
  } catch (const FheError &e) {
    g_last_error = e.what();
    return e.code;
  } catch (const std::invalid_argument &e) {
    g_last_error = e.what();
    return FHE_ERR_INVALID;
  } catch (const std::exception &e) {
    g_last_error = e.what();
    return FHE_ERR_DEVICE;
  }
}

template <class T> T *upload(const std::vector<T> &v, std::vector<void *> &own) {
  void *p = nullptr;
  hip_check(hipMalloc(&p, std::max<size_t>(1, v.size() * sizeof(T))),
            "table allocation");
  own.push_back(p);
  if (!v.empty())
    hip_check(hipMemcpy(p, v.data(), v.size() * sizeof(T),
                        hipMemcpyHostToDevice),
              "table upload");
  return static_cast<T *>(p);
}

// A C ABI status as an exception (for compositions of entry points).
inline void ok(int rc) {
  if (rc != FHE_OK)
    throw FheError(rc, fhe_last_error());
}

} // namespace fhe_host

using namespace fhe_host;

// Work lists of one uneven-level batch shape (uneven.hip).
struct UnevenPlan;
void uneven_plan_free(UnevenPlan *plan);

struct fhe_context {
  fhe::CkksParams params;
  fhe::DeviceTables tables{};
  hipStream_t stream = nullptr;
  int device = 0;
  std::vector<void *> owned;
  // per-(moduli_id, key_moduli_id) ModUp constants on the device
  std::map<std::pair<int, int>, int64_t *> modup_cache;
  // growable scratch for the fused pipelines
  void *workspace = nullptr;
  size_t workspace_bytes = 0;
  // lazy transforms where results are canonicalized before use
  bool lazy_key_switch = true;
  // ModUp staged through the Garner digits (digits kernel + extension fused
  // with the first NTT pass)
  bool staged_modup = true;
  // each partition's own extended limbs from the NTT-form d2 when at hand
  bool own_limbs = true;
  // large-prime key products kept below 2q with one guard
  bool ks_lazy_accumulate = true;
  // second growable device buffer (Garner digits of the staged ModUp)
  void *aux = nullptr;
  size_t aux_bytes = 0;
  // third growable buffer: intermediates of composite operations whose steps
  // use the other two
  void *stash_buf = nullptr;
  size_t stash_bytes = 0;
  void *partial_buf = nullptr;
  size_t partial_bytes = 0;
  // encoding tables, uploaded on the first encode
  fhe::EncodeDevice encode{};
  bool encode_ready = false;
  // decoding tables, uploaded on the first decode; CRT constants per moduli_id
  fhe::DecodeDevice decode{};
  bool decode_ready = false;
  std::map<int, fhe::DecodeCrtDevice> decode_crt_cache;
  // device buffers of the engine-level compositions, kept by size for
  // reuse by later calls
  std::multimap<size_t, void *> text_pool;
  // prepared (rescaled, NTT-form) plaintexts of every diagonal of one
  // butterfly stage, resident per (direction, stages, stage, level)
  struct StagePlaintexts {
    void *data = nullptr;
    int count = 0, level = 0;
  };
  std::map<std::tuple<bool, int, int, int>, StagePlaintexts> boot_diagonals;
  // bootstrap slot-transform diagonals per (log slots, stages, direction)
  std::map<std::tuple<int, int, bool>,
           std::vector<std::vector<std::vector<std::complex<double>>>>>
      boot_twiddles;
  // uneven-level batches: work lists per (kind, key moduli_id, moduli_ids)
  std::map<std::vector<int>, UnevenPlan *> uneven_plans;
  // launch schedules of the uneven-level kernels chosen by timing the
  // candidates on the first call of each batch shape
  bool uneven_autotune = false;
  // the context's stream is being captured into a HIP graph: no call may
  // synchronize, allocate or upload
  bool capturing = false;

  void *pool_take(size_t bytes) {
    auto it = text_pool.find(bytes);
    if (it != text_pool.end()) {
      void *p = it->second;
      text_pool.erase(it);
      return p;
    }
    require_not_capturing("text allocation");
    void *p = nullptr;
    hip_check(hipMalloc(&p, bytes), "text allocation");
    return p;
  }
  // stage timing: HIP events recorded on `stream` around each stage while
  // enabled, folded into per-stage totals when read
  bool timing = false;
  struct PendingStage {
    const char *name;
    hipEvent_t start, stop;
  };
  std::vector<PendingStage> pending;
  std::vector<std::string> stage_names;
  std::vector<double> stage_ms;
  std::vector<int64_t> stage_launches;

  explicit fhe_context(fhe::CkksParams p) : params(std::move(p)) {
    hip_check(hipGetDevice(&device), "hipGetDevice");
    hip_check(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking),
              "stream creation");
    auto &t = tables;
    t.q = upload(params.q, owned);
    t.k = upload(params.k, owned);
    t.q2 = upload(params.q2, owned);
    t.qh = upload(params.qh, owned);
    t.r2 = upload(params.r2, owned);
    t.ninv = upload(params.ninv, owned);
    t.root = upload(params.root, owned);
    t.root_inverse = upload(params.root_inverse, owned);
    t.root_shoup = upload(params.root_shoup, owned);
    t.root_inverse_shoup = upload(params.root_inverse_shoup, owned);
    {
      // the F64 arithmetic's tables from the Shoup pairs' first words
      const size_t words = size_t(params.prime_count) * params.n;
      std::vector<double> d(words);
      for (auto *table : {&params.root_shoup, &params.root_inverse_shoup}) {
        for (size_t i = 0; i < words; i++)
          d[i] = double((*table)[2 * i]);
        (table == &params.root_shoup ? t.root_f64 : t.root_inverse_f64) =
            upload(d, owned);
      }
      std::vector<double> qd(params.prime_count), qi(params.prime_count);
      for (int i = 0; i < params.prime_count; i++) {
        qd[i] = double(params.q[i]);
        qi[i] = 1.0 / qd[i];
      }
      t.q_f64 = upload(qd, owned);
      t.q_inverse_f64 = upload(qi, owned);
    }
    t.p_inverse = upload(params.p_inverse_mult_r, owned);
    t.p_inverse_shoup = upload(params.p_inverse_shoup, owned);
    t.q_top = upload(params.q_top, owned);
    t.rescale = upload(params.rescale_scale, owned);
    t.host_q = params.q.data();
    t.prime_count = params.prime_count;
    t.log_n = params.log_n;
    t.alpha = params.alpha;
  }

  // teardown: errors are not actionable here, so they are ignored
  ~fhe_context() {
    if (stream)
      (void)hipStreamSynchronize(stream);
    for (auto &st : pending) {
      (void)hipEventDestroy(st.start);
      (void)hipEventDestroy(st.stop);
    }
    for (auto &kv : modup_cache)
      (void)hipFree(kv.second);
    for (void *p : owned)
      (void)hipFree(p);
    for (auto &kv : text_pool)
      (void)hipFree(kv.second);
    for (auto &kv : boot_diagonals)
      (void)hipFree(kv.second.data);
    for (auto &kv : uneven_plans)
      uneven_plan_free(kv.second);
    if (workspace)
      (void)hipFree(workspace);
    if (aux)
      (void)hipFree(aux);
    if (stash_buf)
      (void)hipFree(stash_buf);
    if (partial_buf)
      (void)hipFree(partial_buf);
    if (stream)
      (void)hipStreamDestroy(stream);
  }

  int64_t n() const { return params.n; }

  // Runs f (kernel launches on `stream`), bracketed by events when timing.
  template <class F> void stage(const char *name, F &&f) {
    if (!timing) {
      f();
      return;
    }
    PendingStage st{name, nullptr, nullptr};
    hip_check(hipEventCreate(&st.start), "hipEventCreate");
    hip_check(hipEventCreate(&st.stop), "hipEventCreate");
    pending.push_back(st);
    hip_check(hipEventRecord(st.start, stream), "hipEventRecord");
    f();
    hip_check(hipEventRecord(st.stop, stream), "hipEventRecord");
  }

  void fold_timings() {
    hip_check(hipStreamSynchronize(stream), "timing sync");
    for (auto &st : pending) {
      float ms = 0;
      hip_check(hipEventElapsedTime(&ms, st.start, st.stop),
                "hipEventElapsedTime");
      size_t i = 0;
      while (i < stage_names.size() && stage_names[i] != st.name)
        i++;
      if (i == stage_names.size()) {
        stage_names.push_back(st.name);
        stage_ms.push_back(0);
        stage_launches.push_back(0);
      }
      stage_ms[i] += ms;
      stage_launches[i]++;
      (void)hipEventDestroy(st.start);
      (void)hipEventDestroy(st.stop);
    }
    pending.clear();
  }

  // lazy arithmetic of whole transforms: the radix-16 sizes
  bool lazy_transforms() const {
    return lazy_key_switch && fhe::ks_fused_supported(tables);
  }

  // How key switching of `count` ciphertexts at moduli_id runs: on the fused
  // path with the extended limbs of every partition of `group` ciphertexts at
  // once, group after group, or (group 0) one partition of the whole batch at
  // a time.  ext_words: its extended-limb buffer.
  struct KsPlan {
    int group;
    int64_t ext_words;
  };
  // Chains whose partitions together take more limbs per ciphertext run one
  // partition at a time below N = 2^16.
  static constexpr int kMaxExtLimbs = 1024;
  bool ks_fused(int moduli_id) const {
    return fhe::ks_fused_supported(tables) &&
           (tables.log_n == 16 ||
            params.partition_count(moduli_id) *
                    (params.limbs_at(moduli_id) + params.alpha) <=
                kMaxExtLimbs);
  }
  // A group's extended limbs and digits below N = 2^16: 8 GiB, more than 80
  // ciphertexts of the longest chains, so that larger batches need little
  // more than one partition of each did (N = 2^16 holds the batch).
  static constexpr int64_t kKsGroupWords = int64_t(1) << 30;
  int64_t ext_poly_words(int moduli_id) const {
    return int64_t(params.limbs_at(moduli_id) + params.alpha) * params.n;
  }
  KsPlan ks_one_partition(int count, int moduli_id) const {
    return {0, count * ext_poly_words(moduli_id)};
  }
  KsPlan ks_groups_of(int group, int moduli_id) const {
    return {group, group * int64_t(params.partition_count(moduli_id)) *
                       ext_poly_words(moduli_id)};
  }
  // `others`: words that the caller's workspace holds beside the extended
  // limbs.  Where the workspace may not grow (a graph holds it), the groups
  // are as large as what is there allows.
  KsPlan ks_plan(int count, int moduli_id, int64_t others) const {
    const KsPlan least = ks_one_partition(count, moduli_id);
    if (!ks_fused(moduli_id))
      return least;
    if (tables.log_n == 16)
      return ks_groups_of(count, moduli_id);
    const int64_t one = ks_groups_of(1, moduli_id).ext_words;
    int64_t group = std::max(kKsGroupWords, least.ext_words) /
                    (one + ks_digits_words(1, moduli_id));
    if (!may_grow())
      group = std::min(group,
                       (int64_t(workspace_bytes / 8) - others) / one);
    group = std::min<int64_t>(group, count);
    return group > 0 ? ks_groups_of(int(group), moduli_id) : least;
  }
  // The scratch workspace with `others` words and the plan's extended limbs;
  // below N = 2^16, where the device cannot hold them, smaller groups.
  int64_t *ks_scratch(int count, int moduli_id, int64_t others, KsPlan &plan) {
    plan = ks_plan(count, moduli_id, others);
    while (tables.log_n != 16 && plan.group > 0 &&
           !scratch_fits(size_t(others + plan.ext_words) * 8))
      plan = plan.group > 1 ? ks_groups_of(plan.group / 2, moduli_id)
                            : ks_one_partition(count, moduli_id);
    return scratch(size_t(others + plan.ext_words) * 8);
  }

  // Whether workspaces may be reallocated: not under capture, nor while
  // captured graphs hold their addresses.
  bool may_grow() const { return !capturing && live_graphs == 0; }

  void require_not_capturing(const char *what) const {
    require(!capturing, std::string(what) +
                            ": not allowed while the stream is captured (run "
                            "the call once before capturing it)");
  }
  // captured graphs alive on this context: they hold the addresses of the
  // workspaces, which may then not move
  int live_graphs = 0;
  void require_workspace_fixed(const char *what) const {
    require_not_capturing(what);
    require(live_graphs == 0,
            std::string(what) + ": a captured graph holds the workspace "
                                "(destroy it, or run the larger call before "
                                "capturing)");
  }

  // Grows a buffer to `bytes` if it may and the device has the memory; the
  // old contents are gone either way.
  bool grow(void *&buffer, size_t &have, size_t bytes) {
    if (bytes <= have)
      return true;
    if (!may_grow())
      return false;
    hip_check(hipStreamSynchronize(stream), "workspace sync");
    if (buffer)
      hip_check(hipFree(buffer), "workspace free");
    buffer = nullptr;
    have = 0;
    const hipError_t error = hipMalloc(&buffer, bytes);
    if (error == hipErrorOutOfMemory) {
      (void)hipGetLastError(); // not the next launch check's
      buffer = nullptr;
      return false;
    }
    hip_check(error, "workspace allocation");
    have = bytes;
    return true;
  }
  int64_t *grown(void *&buffer, size_t &have, size_t bytes) {
    if (bytes > have)
      require_workspace_fixed("workspace growth");
    if (!grow(buffer, have, bytes))
      hip_check(hipErrorOutOfMemory, "workspace allocation");
    return static_cast<int64_t *>(buffer);
  }

  int64_t *aux_scratch(size_t bytes) { return grown(aux, aux_bytes, bytes); }
  // as aux_scratch, null where it cannot have that size
  int64_t *aux_if_room(size_t bytes) {
    return grow(aux, aux_bytes, bytes) ? static_cast<int64_t *>(aux)
                                       : nullptr;
  }

  // partial sums of the split key inner product; null where the buffer cannot
  // have that size (the caller then does not split)
  int64_t *partial_sums(size_t bytes) {
    return grow(partial_buf, partial_bytes, bytes)
               ? static_cast<int64_t *>(partial_buf)
               : nullptr;
  }

  int64_t *stash(size_t bytes) {
    return grown(stash_buf, stash_bytes, bytes);
  }

  // CKKSCore::switch_key (src/ckks/core.cpp:1058-1083) of `count` INTT-form
  // duos at moduli_id: key switching of c1, then c0 added to the first half
  // and the second half copied.  Uses the scratch workspace.
  void switch_key_into(int count, int moduli_id, const int64_t *in,
                       const int64_t *key, int key_moduli_id, int64_t *out,
                       bool signed_input = false) {
    const int limbs = params.limbs_at(moduli_id);
    const int ext_limbs = limbs + params.alpha;
    const int64_t N = n();
    KsPlan plan;
    int64_t *ext = ks_scratch(count, moduli_id,
                              int64_t(count) * 2 * ext_limbs * N, plan);
    int64_t *acc = ext + plan.ext_words;
    key_switch(count, moduli_id, key, key_moduli_id, in + limbs * N,
               2 * limbs * N, ext, acc, plan, nullptr, 0, signed_input);
    stage("moddown_add", [&] {
      fhe::launch_moddown_add(tables, acc, in, 2 * limbs * N, 1, out, count,
                              limbs, moduli_id, stream);
    });
  }

  int64_t *scratch(size_t bytes) {
    return grown(workspace, workspace_bytes, bytes);
  }
  bool scratch_fits(size_t bytes) {
    return grow(workspace, workspace_bytes, bytes);
  }

  const fhe::EncodeDevice &encode_tables() {
    if (!encode_ready) {
      std::vector<double> fc, fs, tc, ts;
      params.encode_trig(fc, fs, tc, ts);
      encode.pre = upload(params.encode_pre_permutation(), owned);
      encode.fft_cos = upload(fc, owned);
      encode.fft_sin = upload(fs, owned);
      encode.twist_cos = upload(tc, owned);
      encode.twist_sin = upload(ts, owned);
      encode.log_codec = params.log_n;
      encode_ready = true;
    }
    return encode;
  }

  const fhe::DecodeDevice &decode_tables() {
    if (!decode_ready) {
      std::vector<double> sc, ss, ic, is;
      params.decode_trig(sc, ss, ic, is);
      decode.post = upload(params.decode_post_permutation(), owned);
      decode.skew_cos = upload(sc, owned);
      decode.skew_sin = upload(ss, owned);
      decode.ifft_cos = upload(ic, owned);
      decode.ifft_sin = upload(is, owned);
      decode.log_codec = params.log_n;
      decode_ready = true;
    }
    return decode;
  }

  const fhe::DecodeCrtDevice &decode_crt(int moduli_id) {
    auto it = decode_crt_cache.find(moduli_id);
    if (it != decode_crt_cache.end())
      return it->second;
    const auto h = params.decode_crt(moduli_id);
    require(fhe::decode_crt_supported(h.words),
            "Decode: the modulus product is too wide");
    fhe::DecodeCrtDevice d{};
    d.reverser = upload(h.reverser, owned);
    d.q_product = upload(h.q_product, owned);
    d.q_half = upload(h.q_half, owned);
    d.upper = upload(h.upper, owned);
    d.k = h.k;
    d.words = h.words;
    return decode_crt_cache[moduli_id] = d;
  }

  // Level down of `polys` INTT-form polynomials at `level` (rescaled or not)
  // to dst_level < level; out is not rescaled at dst_level.
  void level_down_into(const int64_t *in, int64_t *out, int polys, int level,
                       bool rescaled, int dst_level) {
    const auto &P = params;
    const int dst_mid = P.moduli_id_of_level(dst_level);
    if (rescaled) {
      // CKKSCore::level_down_after_rescale (src/ckks/core.cpp:743-779): the
      // rescaled input sits at moduli_id_of_level(level) + 1
      const int src_mid = P.moduli_id_of_level(level) + 1;
      const auto c = P.level_down_multiplier_after_rescale(level, dst_level);
      const int limbs = int(c.size());
      require(limbs <= fhe::kMaxEwLimbs, "Level down: too many limbs");
      const int64_t src_poly = int64_t(P.limbs_at(src_mid)) << P.log_n;
      const int64_t dst_poly = int64_t(limbs) << P.log_n;
      const int64_t offset = int64_t(dst_mid - src_mid) << P.log_n;
      stage("elementwise", [&] {
        for (int p = 0; p < polys; p++)
          fhe::launch_elementwise(tables, fhe::kEwEnterReduce,
                                  in + p * src_poly + offset, nullptr,
                                  out + p * dst_poly, limbs, limbs, dst_mid,
                                  c.data(), stream);
      });
    } else {
      // CKKSCore::level_down (src/ckks/core.cpp:792-838)
      const int src_mid = P.moduli_id_of_level(level);
      const int next_mid = P.moduli_id_of_level(level - 1);
      const auto c = P.level_down_multiplier(level, dst_level);
      require(int(c.size()) <= fhe::kMaxEwLimbs, "Level down: too many limbs");
      stage("scalar_rescale", [&] {
        fhe::launch_scalar_rescale(tables, in, out, polys, int(c.size()),
                                   src_mid, c.data(), dst_mid - next_mid,
                                   stream);
      });
    }
  }

  // Chain position of a text at `level`: a rescaled text sits one modulus
  // above the not-rescaled text of its level (the not_rescaled_levels_ /
  // rescaled_levels_ maps, src/ckks/parameters.cpp:60-90).
  int moduli_id_of(int level, bool rescaled) const {
    return params.moduli_id_of_level(level) + (rescaled ? 1 : 0);
  }

  // The engine's form changes of `polys` polynomials at (level, flags), in
  // its order: intt_ first when asked (CKKSEngine::intt_), level_down_ to
  // dst_level <= level (src/ckks/engine_level_down.cpp:5-37: after rescale
  // in the current form, else in the coefficient domain), rescale_ when
  // `rescale` and not yet rescaled (src/ckks/engine_rescale.cpp:5-33), ntt_
  // when `ntt` (src/ckks/engine_ntt.cpp:5-21).  Returns `in` itself when
  // nothing changes, else `out`; t0 and t1 hold polys x limbs(level, flags)
  // x N each, and out may not alias them.
  const int64_t *transform_into(const int64_t *in, int64_t polys, int level,
                                int flags, bool intt_first, int dst_level,
                                bool rescale, bool ntt, int64_t *out,
                                int64_t *t0, int64_t *t1) {
    bool rescaled = (flags & FHE_FLAG_RESCALED) != 0;
    bool is_ntt = (flags & FHE_FLAG_NTT_FORM) != 0;
    const int64_t *cur = in;
    // the steps that write a result, counted first so that the last one
    // writes to out (the others alternate between t0 and t1)
    int steps = 0;
    {
      bool r = rescaled, nt = is_ntt;
      if (intt_first && nt) {
        steps++;
        nt = false;
      }
      if (level > dst_level) {
        steps += (!r && nt) ? 3 : 1;
        r = false;
      }
      if (rescale && !r)
        steps += nt ? 3 : 1;
      if (ntt && !nt)
        steps++;
    }
    int64_t *bufs[2] = {t0, t1};
    int next = 0, done = 0;
    auto target = [&] {
      if (++done == steps)
        return out;
      int64_t *b = bufs[next];
      next ^= 1;
      return b;
    };
    auto to_intt = [&] {
      const int mid = moduli_id_of(level, rescaled);
      const int limbs = params.limbs_at(mid);
      int64_t *y = target();
      stage("intt", [&] {
        fhe::ntt_inverse(tables, cur, y, polys * limbs, limbs, mid,
                         fhe::kInttExit, stream);
      });
      cur = y;
      is_ntt = false;
    };
    auto to_ntt = [&] {
      const int mid = moduli_id_of(level, rescaled);
      const int limbs = params.limbs_at(mid);
      int64_t *y = target();
      stage("ntt", [&] {
        fhe::ntt_forward(tables, cur, y, polys * limbs, limbs, mid, tables.r2,
                         stream);
      });
      cur = y;
      is_ntt = true;
    };
    if (intt_first && is_ntt)
      to_intt();
    if (level > dst_level) {
      // a not-rescaled NTT-form text goes down in the coefficient domain
      // and comes back
      const bool back = !rescaled && is_ntt;
      if (back)
        to_intt();
      int64_t *y = target();
      level_down_into(cur, y, int(polys), level, rescaled, dst_level);
      cur = y;
      rescaled = false;
      level = dst_level;
      if (back)
        to_ntt();
    }
    if (rescale && !rescaled) {
      require(level >= 1, "Rescale: the text should have a positive level.");
      const bool back = is_ntt;
      if (back)
        to_intt();
      const int mid = moduli_id_of(level, false);
      int64_t *y = target();
      stage("rescale", [&] {
        fhe::launch_rescale(tables, cur, y, int(polys), params.limbs_at(mid),
                            mid, stream);
      });
      cur = y;
      rescaled = true;
      if (back)
        to_ntt();
    }
    if (ntt && !is_ntt)
      to_ntt();
    require(done == steps && (steps == 0 || cur == out),
            "internal: form change steps miscounted");
    return steps == 0 ? in : out;
  }

  // CKKSEngine::prepare_for_multiply (src/ckks/engine_multiply.cpp:13-27):
  // intt_ when the level changes, level_down_, rescale_, ntt_.
  const int64_t *prepare_for_multiply_into(const int64_t *in, int64_t polys,
                                           int level, int flags,
                                           int dst_level, int64_t *out,
                                           int64_t *t0, int64_t *t1) {
    return transform_into(in, polys, level, flags, level > dst_level,
                          dst_level, true, true, out, t0, t1);
  }

  // Relinearization of `count` NTT-form trios at moduli_id into INTT-form
  // duos (CKKSCore::relinearize, src/ckks/core.cpp:713-741).  Uses the
  // scratch workspace; the trios are not modified.
  void relinearize_into(int count, int moduli_id, const int64_t *trios,
                        const int64_t *key, int key_moduli_id, int64_t *out) {
    const int limbs = params.limbs_at(moduli_id);
    const int ext_limbs = limbs + params.alpha;
    const int64_t N = n();
    const int64_t trio_l = int64_t(count) * 3 * limbs;
    const int64_t acc_l = int64_t(count) * 2 * ext_limbs;
    KsPlan plan;
    int64_t *trio = ks_scratch(count, moduli_id, (trio_l + acc_l) * N, plan);
    int64_t *ext = trio + trio_l * N, *acc = ext + plan.ext_words;
    const int64_t poly = int64_t(limbs) * N;
    // d0 and d1 are canonicalized by the relinearization add; d2 feeds the
    // representative-sensitive ModUp (the flags are in the accumulators,
    // written after them)
    fhe::LazySpec lazy{lazy_transforms(), reinterpret_cast<uint32_t *>(acc),
                       3};
    stage("intt(trio)", [&] {
      fhe::ntt_inverse(tables, trios, trio, trio_l, limbs, moduli_id,
                       fhe::kInttExit, stream, lazy);
      if (lazy.on)
        fhe::launch_repair_intt(tables, lazy.zero, trios + 2 * poly, 3 * poly,
                                trio + 2 * poly, 3 * poly, count, limbs,
                                moduli_id, stream);
    });
    // the caller's NTT-form d2 provides the partitions' own extended limbs
    key_switch(count, moduli_id, key, key_moduli_id, trio + 2 * limbs * N,
               3 * limbs * N, ext, acc, plan, trios + 2 * limbs * N,
               3 * limbs * N);
    stage("moddown_relin", [&] {
      fhe::launch_moddown_relin(tables, acc, trio, out, count, limbs,
                                moduli_id, stream);
    });
  }

  const int64_t *modup_constants(int moduli_id, int key_moduli_id) {
    auto key = std::make_pair(moduli_id, key_moduli_id);
    auto it = modup_cache.find(key);
    if (it != modup_cache.end())
      return it->second;
    require_not_capturing("constant upload");
    const auto host = params.modup_constants(moduli_id, key_moduli_id);
    void *p = nullptr;
    hip_check(hipMalloc(&p, host.size() * sizeof(int64_t)), "constants");
    hip_check(hipMemcpy(p, host.data(), host.size() * sizeof(int64_t),
                        hipMemcpyHostToDevice),
              "constants upload");
    modup_cache[key] = static_cast<int64_t *>(p);
    return static_cast<int64_t *>(p);
  }

  void check_launch(const char *what) {
    hip_check(hipGetLastError(), what);
  }

  void check_moduli(int moduli_id, int min_limbs, const char *op) {
    require(moduli_id >= 0 && moduli_id < params.chain_count,
            std::string(op) + ": moduli_id out of range.");
    require(params.limbs_at(moduli_id) >= min_limbs,
            std::string(op) + ": the given level is too low.");
  }

  void check_key(int moduli_id, int key_moduli_id, const char *op) {
    require(key_moduli_id >= 0 && key_moduli_id <= moduli_id,
            std::string(op) +
                ": the key level is lower than the ciphertext level.");
    require(params.max_key_switching_level() >=
                params.level_of(key_moduli_id, false),
            std::string(op) + ": the key moduli id is above the key-switching "
                              "level.");
  }

  // Key switching of the INTT-form polynomial src + c * src_stride of each
  // ciphertext c into acc ([count][2][ext][N], INTT form, reduced).
  // own (optional): the NTT form of the same polynomials (limb i of
  // ciphertext c at own + c * own_stride + i * N); the fused path then takes
  // each partition's own extended limbs from it instead of transforming them.
  // signed_input: the source limbs may be any int64 (the signed tile of
  // modulus raising), not residues in [0, 2q): every partition then takes
  // the signed Garner digits and the exact extension.
  // digits (optional): room for the staged ModUp's Garner digits of a group
  // (ks_digits_words) instead of the context's second growable buffer.
  void key_switch(int count, int moduli_id, const int64_t *key,
                  int key_moduli_id, const int64_t *src, int64_t src_stride,
                  int64_t *ext, int64_t *acc, const KsPlan &plan,
                  const int64_t *own = nullptr, int64_t own_stride = 0,
                  bool signed_input = false, int64_t *digits = nullptr) {
    if (plan.group > 0) {
      if (!own_limbs || int(params.partitions(moduli_id, key_moduli_id)
                                .size()) > fhe::kMaxFusedParts)
        own = nullptr;
      for (int c = 0; c < count; c += plan.group) {
        const int here = std::min(plan.group, count - c);
        ks_decompose(here, moduli_id, key_moduli_id, src + c * src_stride,
                     src_stride, ext, own != nullptr, signed_input, digits);
        ks_apply(here, moduli_id, key, key_moduli_id, ext,
                 acc + 2 * c * ext_poly_words(moduli_id),
                 own ? own + c * own_stride : nullptr, own_stride,
                 digits == nullptr);
      }
      return;
    }
    const int limbs = params.limbs_at(moduli_id);
    const int ext_limbs = limbs + params.alpha;
    const int64_t N = n();
    const int key_chain = params.limbs_at(key_moduli_id) + params.alpha;
    const int key_offset = params.limbs_at(key_moduli_id) - limbs;
    const auto parts = params.partitions(moduli_id, key_moduli_id);
    const int64_t *cst = modup_constants(moduli_id, key_moduli_id);
    const int stride = params.ks_stride(moduli_id);
    for (size_t p = 0; p < parts.size(); p++) {
      const auto &part = parts[p];
      fhe::launch_modup(tables, src, src_stride, ext, ext_limbs * N, count,
                        limbs, moduli_id, part.start, part.size,
                        cst + p * stride, params.ks_ext_shoup_offset(moduli_id),
                        !signed_input &&
                            params.modup_non_negative(moduli_id, part),
                        false, stream);
      fhe::ntt_forward(tables, ext, ext, int64_t(count) * ext_limbs,
                       ext_limbs, moduli_id, nullptr, stream);
      const int64_t *key0 =
          key + (int64_t(2 * part.key_index) * key_chain + key_offset) * N;
      const int64_t *key1 =
          key + (int64_t(2 * part.key_index + 1) * key_chain + key_offset) * N;
      fhe::launch_key_inner_product(tables, ext, ext_limbs * N, key0, key1,
                                    acc, 2 * ext_limbs * N, count, ext_limbs,
                                    moduli_id, p == 0, stream);
    }
    fhe::ntt_inverse(tables, acc, acc, int64_t(count) * 2 * ext_limbs,
                     ext_limbs, moduli_id, fhe::kInttExitReduce, stream);
  }

  // The key-independent half of key switching on the fused path
  // (N = 2^13 .. 2^16; any N for a bootstrap key's stages):
  // ModUp of every partition and the first forward NTT pass of every
  // extended limb into ext [count][parts][ext][N] (CKKSCore::decompose,
  // src/ckks/core_key_switch.cpp:434-460, up to its second NTT pass).
  // The extended polynomials, their products with the key and the
  // accumulators are only read by ModDown after the canonicalizing exit,
  // so with lazy_key_switch their arithmetic is lazy.
  // Words of Garner digits the staged ModUp of `count` ciphertexts at
  // moduli_id holds (partitions x partition size rounded to a power of 2).
  int64_t ks_digits_words(int count, int moduli_id) const {
    int maxz = 1;
    while (maxz < params.alpha)
      maxz <<= 1;
    return int64_t(count) * params.partition_count(moduli_id) * maxz *
           params.n;
  }

  void ks_decompose(int count, int moduli_id, int key_moduli_id,
                    const int64_t *src, int64_t src_stride, int64_t *ext,
                    bool skip_own = false, bool signed_input = false,
                    int64_t *digits_ws = nullptr) {
    const int limbs = params.limbs_at(moduli_id);
    const int ext_limbs = limbs + params.alpha;
    const int64_t N = n();
    const auto parts = params.partitions(moduli_id, key_moduli_id);
    const int64_t *cst = modup_constants(moduli_id, key_moduli_id);
    const int stride = params.ks_stride(moduli_id);
    const int np = int(parts.size());
    // exact throughout where the second pass is (N > 2^16): its butterflies
    // take values below 2q, the lazy first pass gives up to 8q
    const fhe::LazySpec lazy{lazy_transforms()};
    int max_size = 0;
    bool is_signed[fhe::kMaxFusedParts] = {};
    std::vector<int> starts(np), sizes(np);
    for (int p = 0; p < np; p++) {
      starts[p] = parts[p].start;
      sizes[p] = parts[p].size;
      if (p < fhe::kMaxFusedParts)
        is_signed[p] = signed_input ||
                       !params.modup_non_negative(moduli_id, parts[p]);
      max_size = std::max(max_size, sizes[p]);
    }
    int64_t *digits = nullptr;
    if (staged_modup && fhe::staged_modup_supported(tables, max_size, np)) {
      int maxz = 1;
      while (maxz < max_size)
        maxz <<= 1;
      // without room for the digits the extension recomputes them
      digits = digits_ws
                   ? digits_ws
                   : aux_if_room(size_t(count) * np * maxz * size_t(N) * 8);
    }
    if (digits) {
      stage("modup_staged(ext)", [&] {
        fhe::launch_staged_modup(tables, src, src_stride, digits, ext, count,
                                 limbs, moduli_id, starts.data(), sizes.data(),
                                 is_signed, np, cst, stride,
                                 params.ks_ext_shoup_offset(moduli_id),
                                 lazy.on, skip_own, stream);
      });
      return;
    }
    for (int p = 0; p < np; p++)
      stage("modup", [&] {
        fhe::launch_modup(tables, src, src_stride,
                          ext + int64_t(p) * ext_limbs * N,
                          int64_t(np) * ext_limbs * N, count, limbs, moduli_id,
                          parts[p].start, parts[p].size, cst + p * stride,
                          params.ks_ext_shoup_offset(moduli_id),
                          !signed_input &&
                              params.modup_non_negative(moduli_id, parts[p]),
                          lazy.on && !signed_input, stream);
      });
    stage("ntt_pass_high(ext)", [&] {
      fhe::ntt_forward_first(tables, ext, ext, int64_t(count) * np * ext_limbs,
                             ext_limbs, moduli_id, nullptr, stream, lazy);
    });
  }

  // The key-dependent half on the fused path: second NTT pass, key inner
  // product over all partitions, both INTT passes (with exit and reduce)
  // into acc [count][2][ext][N].
  void ks_apply(int count, int moduli_id, const int64_t *key,
                int key_moduli_id, const int64_t *ext, int64_t *acc,
                const int64_t *own = nullptr, int64_t own_stride = 0,
                bool may_allocate = true) {
    const int limbs = params.limbs_at(moduli_id);
    const int ext_limbs = limbs + params.alpha;
    const int key_chain = params.limbs_at(key_moduli_id) + params.alpha;
    const int key_offset = params.limbs_at(key_moduli_id) - limbs;
    const auto parts = params.partitions(moduli_id, key_moduli_id);
    const int np = int(parts.size());
    const fhe::LazySpec lazy{lazy_key_switch};
    std::vector<int> starts(np), sizes(np);
    for (int p = 0; p < np; p++) {
      starts[p] = parts[p].start;
      sizes[p] = parts[p].size;
    }
    if (np > fhe::kMaxFusedParts)
      own = nullptr;
    fhe::KsSplit split;
    fhe::PartialSums more;
    int64_t *partials = nullptr;
    if (may_allocate) {
      split = fhe::ks_split(tables, np, count, ext_limbs, lazy_key_switch);
      more.stride = int64_t(count) * 2 * ext_limbs * n();
      more.count = split.groups - 1;
      if (more.count > 0) {
        partials = partial_sums(size_t(more.stride) * more.count * 8);
        if (!partials) {
          split = fhe::KsSplit();
          more.count = 0;
        }
      }
      more.data = partials;
    }
    stage("ks_inner_product_r16", [&] {
      fhe::launch_ks_inner_product_fused(
          tables, ext, key, key_chain, key_offset, parts[0].key_index, np, acc,
          count, ext_limbs, moduli_id, lazy_key_switch, own, own_stride,
          starts.data(), sizes.data(), ks_lazy_accumulate, split, partials,
          stream);
    });
    stage("intt_pass_high(acc)", [&] {
      fhe::ntt_inverse_second(tables, acc, acc, int64_t(count) * 2 * ext_limbs,
                              ext_limbs, moduli_id, fhe::kInttKeyReduce,
                              stream, lazy, more);
    });
  }
};

// Device encoding (context.hip): `count` device messages at `level` into
// out [count][limbs (+ alpha with include_special)][N].
void encode_texts(fhe_context *ctx, const double *values, bool complex_input,
                  int count, int level, bool include_special, int64_t *out);

// The parameters a fhe_params describes (context.hip); twiddles = false
// skips the NTT tables (host-only queries).
fhe::CkksParams resolve_params(const fhe_params *p, bool twiddles = true);

// The batched product, relinearization and, with rescale, rescale pipeline
// (context.hip) of duos in INTT form, or NTT form with a_ntt / b_ntt, on a
// caller-given workspace (limbs of N words, per ciphertext).
struct ProductSpace {
  fhe_context::KsPlan plan;
  int64_t *factors; // the factors' transforms: 4 x limbs
  int64_t *trio;    // the trio in NTT form: 3 x limbs
  int64_t *trio_c;  // and in coefficient form: 3 x limbs
  int64_t *ext;     // plan.ext_words in all
  int64_t *acc;     // 2 x (limbs + alpha)
  int64_t *digits;  // ks_digits_words of a group, or null
  // all but the extended limbs and digits of a batch, one after the other
  static int64_t others(const fhe_context *ctx, int count, int moduli_id);
  static ProductSpace at(const fhe_context *ctx, int count, int moduli_id,
                         const fhe_context::KsPlan &plan, int64_t *ws,
                         int64_t *digits);
};
void hmult_relin_into(fhe_context *ctx, int count, int moduli_id,
                      const int64_t *a, bool a_ntt, const int64_t *b,
                      bool b_ntt, const int64_t *key, int key_moduli_id,
                      bool rescale, int64_t *out, const ProductSpace &space);
// Set-up of the allocation-free entry point on the current device `device`
// (noalloc.hip).
void noalloc_scratch_setup(int device);
