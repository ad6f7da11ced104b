// An allocation-free form of the batched HMult + relinearize + rescale, for
// callers that cannot allocate device memory (code under HIP graph capture,
// tight serving loops, harnesses that forbid allocation).  Its workspace is
// one file-scope device array, `scratch`, of kScratchBytes: every GPU the
// library runs on holds its own copy until the process ends.  Host code
// never uses the array's name as a device address: each device's address
// comes from hipGetSymbolAddress at context creation (with that device
// current) and is kept per device.
//
// Every call on a GPU shares that GPU's array, and the array keeps the last
// call's contents: the pipeline writes every word it reads, so nothing has
// to start at zero.  Calls that overlap on one GPU (two contexts' streams,
// or two host threads) race on the array.
#include <mutex>

#include "context.h"

namespace {

constexpr size_t kScratchBytes = size_t(512) << 20; // 512 MiB
constexpr size_t kScratchWords = kScratchBytes / 8;
constexpr int kMaxDevices = 64;

__device__ __align__(256) int64_t scratch[kScratchWords];

std::mutex scratch_mutex;
int64_t *scratch_address[kMaxDevices] = {};

} // namespace

// The device address of `scratch` on the current device (`device`), looked
// up once per device; called from fhe_context_create.
void noalloc_scratch_setup(int device) {
  require(device >= 0 && device < kMaxDevices,
          "device index beyond the scratch table");
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (scratch_address[device])
    return;
  void *p = nullptr;
  hip_check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)),
            "hipGetSymbolAddress(scratch)");
  scratch_address[device] = static_cast<int64_t *>(p);
}

extern "C" int fhe_hmult_relin_rescale_noalloc(fhe_context *ctx, int count,
                                               int moduli_id,
                                               const int64_t *a,
                                               const int64_t *b,
                                               const int64_t *key,
                                               int key_moduli_id,
                                               int64_t *out) {
  return guarded([&] {
    require(ctx && a && b && key && out, "null argument");
    require(count > 0, "Multiply: empty batch");
    ctx->check_moduli(moduli_id, 3, "Multiply");
    ctx->check_key(moduli_id, key_moduli_id, "Multiply");
    // the one-partition-at-a-time form needs the least workspace where it
    // runs (N != 2^16); batches it holds are accepted, and run in the fused
    // form in as many parts as the fused form's workspace asks for, or, when
    // that holds not even one pair, one partition at a time
    using Plan = fhe_context::KsPlan;
    auto words = [&](int n, const Plan &plan) {
      return ProductSpace::others(ctx, n, moduli_id) + plan.ext_words +
             ctx->ks_digits_words(n, moduli_id);
    };
    const bool whole = ctx->tables.log_n == 16;
    Plan plan = whole ? ctx->ks_groups_of(count, moduli_id)
                      : ctx->ks_one_partition(count, moduli_id);
    const int64_t least = words(count, plan);
    require(size_t(least) <= kScratchWords,
            "Multiply (no allocation): the batch needs " +
                std::to_string(least * 8) +
                " bytes of workspace, above the " +
                std::to_string(kScratchBytes) +
                "-byte scratch; split the batch");
    const int64_t in = int64_t(2) * ctx->params.limbs_at(moduli_id) * ctx->n();
    const int64_t res = in - 2 * ctx->n();
    int part = count;
    if (!whole && ctx->ks_fused(moduli_id)) {
      const Plan one = ctx->ks_groups_of(1, moduli_id);
      const int fit = int(std::min<int64_t>(
          count, int64_t(kScratchWords) / words(1, one)));
      // a part's results may not reach the factors of a later part: an output
      // is never ahead of a factor that starts at or after it (a result is
      // shorter than a factor)
      auto apart = [&](const int64_t *x) {
        return out <= x || out >= x + count * in;
      };
      if (fit >= count || (fit > 0 && apart(a) && apart(b))) {
        part = fit;
        plan = ctx->ks_groups_of(part, moduli_id);
      }
    }
    require(ctx->modup_cache.count({moduli_id, key_moduli_id}) != 0,
            "Multiply (no allocation): no ModUp constants for this key "
            "level (contexts prepare those of the maximum key-switching "
            "level)");
    int64_t *base = nullptr;
    {
      std::lock_guard<std::mutex> lock(scratch_mutex);
      if (ctx->device >= 0 && ctx->device < kMaxDevices)
        base = scratch_address[ctx->device];
    }
    require(base != nullptr, "Multiply (no allocation): no scratch address "
                             "for this device");
    for (int c = 0; c < count; c += part) {
      const int n = std::min(part, count - c);
      hmult_relin_into(
          ctx, n, moduli_id, a + c * in, false, b + c * in, false, key,
          key_moduli_id, true, out + c * res,
          ProductSpace::at(ctx, n, moduli_id, plan, base,
                           base + ProductSpace::others(ctx, n, moduli_id) +
                               plan.ext_words));
    }
    ctx->check_launch("Multiply");
  });
}
