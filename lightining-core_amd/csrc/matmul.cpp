// matmul.cpp -- matmul front-end for the "hip" device.
//
// Mirrors ops::matMulWithPolicy<float> (reference include/lightning_core/
// core/ops.hpp:354-459) and MatMulMetalResidentSession<T> (:1339-1379):
//   * validation: (upload_a && !a) || (upload_b && !b) || (download_out &&
//     !out) || any zero dim -> kInvalidValue (:367-370);
//   * workload hint m*k*n in the op_dispatch trace (:366);
//   * resident protocol start (upload, no download, no sync), run (launch
//     only), finish (download + sync), sync (sync only), and the batched
//     launch-only forms (:207-352, policy.hpp:37-71);
//   * buffers of the policy-level API live in one backend-global slot, as the
//     reference's Metal context (matmul_metal.mm:1836-1937); sessions own
//     their own buffers instead.
// 16-bit compute rounds the fp32 host data once at upload (RNE) and lays B out
// K-contiguous (transposed), the layout the MFMA GEMM reads.
#include <algorithm>
#include <climits>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <iterator>
#include <limits>
#include <string>
#include <vector>

#include "ops_internal.hpp"
#include "tune.hpp"

namespace lchip {

GuardArgs beginGuard(HipContext* ctx, int* slot, int which) {
  if (ctx->guard_host.get() == nullptr) {
    const std::size_t bytes = 2 * kGuardSlots * sizeof(int);
    if (ctx->guard_words.ensure(bytes, true) != Status::kSuccess ||
        ctx->guard_host.ensure(bytes) != Status::kSuccess) {
      return GuardArgs{nullptr, nullptr, 0};
    }
    std::memset(ctx->guard_host.get(), 0, bytes);
    for (int i = kGuardSlots - 1; i >= 0; --i) {
      ctx->guard_free.push_back(i);
    }
  }
  if (*slot < 0 && !ctx->guard_free.empty()) {
    *slot = ctx->guard_free.back();
    ctx->guard_free.pop_back();
  }
  if (*slot < 0 || ctx->guard_epoch == INT_MAX) {
    return GuardArgs{nullptr, nullptr, 0};
  }
  const int at = 2 * *slot + which;
  return GuardArgs{ctx->guard_words.as<int>() + at, static_cast<int*>(ctx->guard_host.device()) + at,
                   ++ctx->guard_epoch};
}

void releaseGuard(HipContext* ctx, int* slot) {
  if (*slot >= 0) {
    ctx->guard_free.push_back(*slot);
    *slot = -1;
  }
}

bool knownUnfit(const HipContext* ctx, int slot, int which, int epoch) {
  return epoch == 0 || static_cast<const volatile int*>(ctx->guard_host.get())[2 * slot + which] == epoch;
}

namespace {

// The guard of an fp32 operand about to be uploaded (`which` 0: A, 1: B).
GuardArgs beginUpload(HipContext* ctx, MatMulResident& r, int which) {
  const GuardArgs g = beginGuard(ctx, &r.guard_slot, which);
  (which == 0 ? r.epoch_a : r.epoch_b) = g.epoch;
  (which == 0 ? r.has_planes_a : r.has_planes_b) = false;
  r.planes_denied = 0;
  return g;
}

bool knownUnsafe(const HipContext* ctx, const MatMulResident& r) {
  return knownUnfit(ctx, r.guard_slot, 0, r.epoch_a) || knownUnfit(ctx, r.guard_slot, 1, r.epoch_b);
}

Status uploadA(HipContext* ctx, MatMulResident& r, const float* a) {
  if (!isHalf(r.dtype)) {
    // fp32: A [roundup(M, 64), roundup(K, 64)], zero pads
    const std::size_t mp = roundUp(r.m, kern::kF32GemmBM);
    const std::size_t kp = roundUp(r.k, kern::kF32GemmBK);
    LC_TRY(r.stage.ensure(r.m * r.k * sizeof(float)));
    LC_TRY(r.a.ensure(mp * kp * sizeof(float)));
    LC_TRY(upload(ctx, r.stage.get(), a, r.m * r.k * sizeof(float)));
    const GuardArgs g = beginUpload(ctx, r, 0);
    const hipError_t e = kern::padCopyF32(r.stage.as<float>(), r.a.as<float>(), static_cast<int>(r.m),
                                          static_cast<int>(r.k), r.k, static_cast<int>(mp), static_cast<int>(kp),
                                          ctx->stream, g.word, g.host, g.epoch);
    return e == hipSuccess ? Status::kSuccess : failHip(e, "matmul upload padding (A)");
  }
  const std::size_t mp = roundUp(r.m, kern::kHalfGemmBM);
  const std::size_t kp = roundUp(r.k, kern::kHalfGemmBK);
  LC_TRY(r.stage.ensure(r.m * r.k * sizeof(float)));
  LC_TRY(r.a.ensure(mp * kp * sizeof(uint16_t)));
  LC_TRY(upload(ctx, r.stage.get(), a, r.m * r.k * sizeof(float)));
  const hipError_t e = kern::convertPad(r.stage.as<float>(), r.a.as<uint16_t>(), 1, static_cast<int>(r.m),
                                        static_cast<int>(r.k), r.k, static_cast<int>(mp), static_cast<int>(kp), 0, 0,
                                        halfOf(r.dtype), ctx->stream);
  return e == hipSuccess ? Status::kSuccess : failHip(e, "matmul upload conversion (A)");
}

Status uploadB(HipContext* ctx, MatMulResident& r, const float* b) {
  if (!isHalf(r.dtype)) {
    // fp32: B [roundup(K, 64), roundup(N, 64)], zero pads
    const std::size_t kp = roundUp(r.k, kern::kF32GemmBK);
    const std::size_t np = roundUp(r.n, kern::kF32GemmBN);
    LC_TRY(r.stage.ensure(r.k * r.n * sizeof(float)));
    LC_TRY(r.b.ensure(kp * np * sizeof(float)));
    LC_TRY(upload(ctx, r.stage.get(), b, r.k * r.n * sizeof(float)));
    const GuardArgs g = beginUpload(ctx, r, 1);
    const hipError_t e = kern::padCopyF32(r.stage.as<float>(), r.b.as<float>(), static_cast<int>(r.k),
                                          static_cast<int>(r.n), r.n, static_cast<int>(kp), static_cast<int>(np),
                                          ctx->stream, g.word, g.host, g.epoch);
    return e == hipSuccess ? Status::kSuccess : failHip(e, "matmul upload padding (B)");
  }
  const std::size_t np = roundUp(r.n, kern::kHalfGemmBN);
  const std::size_t kp = roundUp(r.k, kern::kHalfGemmBK);
  LC_TRY(r.stage.ensure(r.k * r.n * sizeof(float)));
  LC_TRY(r.b.ensure(np * kp * sizeof(uint16_t)));
  LC_TRY(upload(ctx, r.stage.get(), b, r.k * r.n * sizeof(float)));
  // B [K, N] -> Bt [N_pad, K_pad]
  const hipError_t e = kern::convertTransposePad(r.stage.as<float>(), r.b.as<uint16_t>(), 1, static_cast<int>(r.k),
                                                 static_cast<int>(r.n), r.n, static_cast<int>(kp),
                                                 static_cast<int>(np), 0, 0, halfOf(r.dtype), ctx->stream);
  return e == hipSuccess ? Status::kSuccess : failHip(e, "matmul upload conversion (B)");
}

// Tune-cache names of the GEMM variants and the configuration each stands
// for (block tile M x N x K, waves, K-split of a stage between wave groups).
struct VariantInfo {
  int variant;
  const char* name;
  int tile_m, tile_n, tile_k, waves, split_k;
  const char* hip_kernel;  // the __global__ function that runs it
};

constexpr VariantInfo kF32Variants[] = {
    {static_cast<int>(kern::GemmF32Variant::kDataParallel), "f32_dp_64x64x64", 64, 64, 64, 8, 2,
     "gemm_f32_lds_kernel"},
    {static_cast<int>(kern::GemmF32Variant::kStreamK), "f32_streamk_64x64x64", 64, 64, 64, 8, 2,
     "gemm_f32_lds_kernel"},
    {static_cast<int>(kern::GemmF32Variant::kDataParallelBK32), "f32_dp_64x64x32", 64, 64, 32, 8, 2,
     "gemm_f32_lds_kernel"},
    {static_cast<int>(kern::GemmF32Variant::kSplit64), "f32_split_64x64", 64, 64, 32, 4, 4, "gemm_f32_split_kernel"},
    {static_cast<int>(kern::GemmF32Variant::kSplit80), "f32_split_80x64", 80, 64, 32, 4, 4, "gemm_f32_split_kernel"},
    {static_cast<int>(kern::GemmF32Variant::kSplit128), "f32_split_128x128", 128, 128, 32, 4, 1,
     "gemm_f32_split128_kernel"},
};

constexpr VariantInfo kHalfVariants[] = {
    {static_cast<int>(kern::GemmHalfVariant::kW4), "half_w4_256x256", 256, 256, 32, 4, 1, "gemm_half_tn_w4_kernel"},
    {static_cast<int>(kern::GemmHalfVariant::kW4D), "half_w4d_256x256", 256, 256, 64, 4, 1,
     "gemm_half_tn_w4d_kernel"},
    {static_cast<int>(kern::GemmHalfVariant::kW4R), "half_w4r_256x256", 256, 256, 64, 4, 1,
     "gemm_half_tn_w4r_kernel"},
    {static_cast<int>(kern::GemmHalfVariant::kW4H), "half_w4h_256x256", 256, 256, 64, 4, 1,
     "gemm_half_tn_w4h_kernel"},
    {static_cast<int>(kern::GemmHalfVariant::kLds), "half_lds_256x256", 256, 256, 64, 8, 1,
     "gemm_half_tn_lds_kernel"},
    {static_cast<int>(kern::GemmHalfVariant::kBig8), "half_big8_256x256", 256, 256, 64, 8, 1, "gemm_half_tn_kernel"},
    {static_cast<int>(kern::GemmHalfVariant::kBig4), "half_big4_256x256", 256, 256, 64, 4, 1, "gemm_half_tn_kernel"},
    {static_cast<int>(kern::GemmHalfVariant::kMid), "half_mid_128x128", 128, 128, 64, 4, 1, "gemm_half_tn_kernel"},
    {static_cast<int>(kern::GemmHalfVariant::kSmall), "half_small_64x64", 64, 64, 64, 4, 1, "gemm_half_tn_kernel"},
    {static_cast<int>(kern::GemmHalfVariant::kR128), "half_r4_128x128", 128, 128, 64, 4, 1, "gemm_half_tn_r4_kernel"},
    {static_cast<int>(kern::GemmHalfVariant::kR96), "half_r4_96x128", 96, 128, 64, 4, 1, "gemm_half_tn_r4_kernel"},
    {static_cast<int>(kern::GemmHalfVariant::kR64x128), "half_r4_64x128", 64, 128, 64, 4, 1, "gemm_half_tn_r4_kernel"},
    {static_cast<int>(kern::GemmHalfVariant::kR64), "half_r4_64x64", 64, 64, 64, 4, 1, "gemm_half_tn_r4_kernel"},
    {static_cast<int>(kern::GemmHalfVariant::kR32), "half_r4_32x64", 32, 64, 64, 4, 1, "gemm_half_tn_r4_kernel"},
    {static_cast<int>(kern::GemmHalfVariant::kSkinny), "half_skinny_16x64", 16, 64, 256, 8, 2, "gemm_skinny_kernel"},
};

struct VariantTable {
  const VariantInfo* first;
  const VariantInfo* last;
  const VariantInfo* begin() const { return first; }
  const VariantInfo* end() const { return last; }
};

VariantTable variants(bool half) {
  return half ? VariantTable{std::begin(kHalfVariants), std::end(kHalfVariants)}
              : VariantTable{std::begin(kF32Variants), std::end(kF32Variants)};
}

const VariantInfo* infoOf(bool half, int variant) {
  for (const VariantInfo& v : variants(half)) {
    if (v.variant == variant) {
      return &v;
    }
  }
  return nullptr;
}

bool isSplit(int variant) { return variant >= static_cast<int>(kern::GemmF32Variant::kSplit64); }

// The variants of a shape (0: not settled).  fp32 has two: `once` for a call
// that uploads an operand and launches once, never one of the split GEMM, and
// `resident` for every other launch.  The tune cache's row names one variant
// for both ("A"), or "once|resident", or "once|" before a resident launch was
// timed; a row that names a split variant alone leaves `once` open.
struct Choices {
  int once = 0;
  int resident = 0;
};

TuneEntry entryFor(bool half, const Choices& c) {
  const VariantInfo* once = infoOf(half, c.once);
  const VariantInfo* resident = infoOf(half, c.resident);
  const VariantInfo* v = resident != nullptr ? resident : once;  // the row's figures
  TuneEntry e;
  e.kernel = c.once == c.resident ? v->name
                                  : std::string(once->name) + "|" + (resident != nullptr ? resident->name : "");
  e.tile_m = v->tile_m;
  e.tile_n = v->tile_n;
  e.tile_k = v->tile_k;
  e.waves = v->waves;
  e.split_k = v->split_k;
  return e;
}

// The variant a cached row names, 0 unless this shape can run it.
int variantFromName(const std::string& name, bool half, std::size_t m, std::size_t k) {
  const long long k_pad = static_cast<long long>(roundUp(k, kern::kHalfGemmBK));
  for (const VariantInfo& v : variants(half)) {
    if (name == v.name) {
      const bool skinny = v.variant == static_cast<int>(kern::GemmHalfVariant::kSkinny);
      if (half && skinny != (m <= 16)) {
        return 0;
      }
      if (half && kern::isR4(static_cast<kern::GemmHalfVariant>(v.variant)) && !kern::gemmHalfR4Fits(k_pad, k_pad)) {
        return 0;
      }
      return v.variant;
    }
  }
  return 0;
}

Choices cachedChoices(HipContext* ctx, const MatMulResident& r) {
  const bool half = isHalf(r.dtype);
  Choices c;
  TuneEntry e;
  if (!tuneLookup(r.m, r.k, r.n, static_cast<int>(r.dtype), baseArch(ctx), &e)) {
    return c;
  }
  const std::size_t bar = e.kernel.find('|');
  c.once = variantFromName(e.kernel.substr(0, bar), half, r.m, r.k);
  c.resident = bar == std::string::npos ? c.once : variantFromName(e.kernel.substr(bar + 1), half, r.m, r.k);
  if (!half && isSplit(c.once)) {
    c.once = 0;
  }
  return c;
}

int cuCount(const HipContext* ctx) {
  return ctx->props.multiProcessorCount > 0 ? ctx->props.multiProcessorCount : 256;
}

// The split GEMM keeps 6 bytes more per operand value; past an eighth of the
// device's memory, or past the kernels' 32-bit offsets along k (160 bytes a k),
// the fp32 kernels run instead.  The planes are given up when another
// allocation needs their memory.
bool splitFits(const HipContext* ctx, std::size_t m, std::size_t k, std::size_t n) {
  const std::size_t kp = roundUp(k, kern::kF32GemmBK);
  const std::size_t rows = roundUp(m, kern::kF32GemmBM) + roundUp(n, kern::kF32GemmBN);
  return kp <= (std::size_t{1} << 23) && 3 * sizeof(uint16_t) * rows * kp <= ctx->props.totalGlobalMem / 8;
}

// The GEMM of a split variant (its planes made first if they are stale);
// false when its buffers cannot be had, and nothing was launched.
bool launchSplitGemm(HipContext* ctx, MatMulResident& r, kern::GemmF32Variant variant, hipError_t* result) {
  const int M = static_cast<int>(r.m);
  const int N = static_cast<int>(r.n);
  const int kp = static_cast<int>(roundUp(r.k, kern::kF32GemmBK));
  const int np = static_cast<int>(roundUp(r.n, kern::kF32GemmBN));
  const int mp = static_cast<int>(roundUp(r.m, kern::kF32GemmBM));
  const int splits = kern::gemmF32SplitCount(variant, M, N, kp, cuCount(ctx));
  kern::SplitKWork work{nullptr, nullptr};
  if (splits > 1) {
    const std::size_t tiles = kern::gemmF32SplitTiles(variant, M, N);
    if (ctx->splitk_part.ensure(tiles * splits * kern::gemmF32SplitPartFloats(variant) * sizeof(float)) !=
            Status::kSuccess ||
        ctx->splitk_counters.ensure(tiles * sizeof(int), true) != Status::kSuccess) {
      return false;
    }
    work = kern::SplitKWork{ctx->splitk_part.as<float>(), ctx->splitk_counters.as<int>()};
  }
  const std::size_t na = 3 * static_cast<std::size_t>(mp) * kp;
  const std::size_t nb = 3 * static_cast<std::size_t>(np) * kp;
  if (r.planes.size() < (na + nb) * sizeof(uint16_t)) {
    r.has_planes_a = r.has_planes_b = false;  // never made, too small, or freed for another allocation
  }
  if (r.planes_denied == ctx->frees) {
    return false;
  }
  if (r.planes.ensureSpare(ctx, (na + nb) * sizeof(uint16_t)) != Status::kSuccess) {
    r.planes_denied = ctx->frees;
    return false;
  }
  r.planes_denied = 0;
  const kern::SplitOperandF32 a{r.a.as<float>(), kp, mp / 16, r.planes.as<uint16_t>()};
  const kern::SplitOperandF32 b{r.b.as<float>(), np, np / 16, r.planes.as<uint16_t>() + na};
  if (!r.has_planes_a || !r.has_planes_b) {
    kern::SplitOperandF32 new_a = a, new_b = b;
    new_a.src = r.has_planes_a ? nullptr : a.src;
    new_b.src = r.has_planes_b ? nullptr : b.src;
    *result = kern::splitPlanesF32(new_a, new_b, kp, ctx->stream);
    if (*result != hipSuccess) {
      return true;
    }
    r.has_planes_a = r.has_planes_b = true;
  }
  const int* words = ctx->guard_words.as<int>() + 2 * r.guard_slot;
  const kern::SplitGuardF32 guard{words, words + 1, r.epoch_a, r.epoch_b};
  *result = kern::gemmF32Split(a, b, r.c.as<float>(), M, N, kp, N, guard, work, variant, splits, ctx->stream);
  return true;
}

hipError_t launchGemm(HipContext* ctx, MatMulResident& r, int variant) {
  const int M = static_cast<int>(r.m);
  const int K = static_cast<int>(r.k);
  const int N = static_cast<int>(r.n);
  if (!isHalf(r.dtype)) {
    const int kp = static_cast<int>(roundUp(r.k, kern::kF32GemmBK));
    const int np = static_cast<int>(roundUp(r.n, kern::kF32GemmBN));
    if (isSplit(variant)) {
      hipError_t e = hipSuccess;
      if (!knownUnsafe(ctx, r) && splitFits(ctx, r.m, r.k, r.n) &&
          launchSplitGemm(ctx, r, static_cast<kern::GemmF32Variant>(variant), &e)) {
        return e;
      }
      variant = r.once;
    }
    // stream-K: one workgroup per CU (a whole-tile grid may hold two per CU)
    const int groups = cuCount(ctx);
    const bool fresh_fail = ctx->gemm_fail.get() == nullptr;
    if (ctx->gemm_part.ensure(static_cast<std::size_t>(groups) * 4096 * sizeof(float)) != Status::kSuccess ||
        ctx->gemm_flags.ensure(static_cast<std::size_t>(groups) * sizeof(int), true) != Status::kSuccess ||
        ctx->gemm_fail.ensure(sizeof(int)) != Status::kSuccess) {
      return hipErrorOutOfMemory;
    }
    if (fresh_fail) {
      *static_cast<int*>(ctx->gemm_fail.get()) = 0;
    }
    kern::StreamKSync sync{ctx->gemm_part.as<float>(), ctx->gemm_flags.as<int>(),
                           static_cast<int*>(ctx->gemm_fail.device()), 0, streamKSpinLimit()};
    if (nextStreamKEpoch(ctx, &sync.epoch) != Status::kSuccess) {
      return hipErrorUnknown;
    }
    return kern::gemmF32Padded(r.a.as<float>(), r.b.as<float>(), r.c.as<float>(), M, N, kp, kp, np, N, sync, groups,
                               static_cast<kern::GemmF32Variant>(variant), ctx->stream);
  }
  const int kp = static_cast<int>(roundUp(r.k, kern::kHalfGemmBK));
  if (kern::isR4(static_cast<kern::GemmHalfVariant>(variant))) {
    return kern::gemmHalfR4(r.a.as<uint16_t>(), r.b.as<uint16_t>(), r.c.as<float>(), M, N, kp, kp, kp, N,
                            halfOf(r.dtype), static_cast<kern::GemmHalfVariant>(variant), ctx->stream);
  }
  kern::SkinnyWork skinny{nullptr, nullptr, 0, 0, 0};
  if (M <= 16) {
    const int tiles = static_cast<int>(roundUp(r.n, 64) / 64);
    if (ctx->skinny_part.ensure(static_cast<std::size_t>(kern::kSkinnyMaxSplits) * tiles * kern::kSkinnyPartFloats *
                                sizeof(float)) != Status::kSuccess ||
        ctx->skinny_counters.ensure(static_cast<std::size_t>(tiles) * sizeof(int), true) != Status::kSuccess) {
      return hipErrorOutOfMemory;
    }
    skinny = kern::SkinnyWork{ctx->skinny_part.as<float>(), ctx->skinny_counters.as<int>(),
                              static_cast<int>(ctx->skinny_counters.size() / sizeof(int)), kern::kSkinnyMaxSplits,
                              ctx->props.multiProcessorCount > 0 ? ctx->props.multiProcessorCount : 256};
  }
  return kern::gemmHalfTN(r.a.as<uint16_t>(), r.b.as<uint16_t>(), r.c.as<float>(), M, N, kp, kp, kp, N,
                          halfOf(r.dtype), static_cast<kern::GemmHalfVariant>(variant), ctx->stream, &skinny);
}

// Times the candidates round-robin (so clock and thermal drift spread over
// all of them): one warm-up round, then 5 rounds of 2 back-to-back launches
// per candidate timed with HIP events on the context stream; the median per
// candidate counts (the reference's autoTuneTile takes a 5-sample median,
// src/ops/matmul_metal.mm:1687-1710).  16-bit candidates that take over 1.5 times
// the first timed round's fastest, where that is 20 us or more a launch, keep that
// one sample (ms to set up a session, with all samples / so: bf16 8192^3 165 / 82,
// 4096^3 24.7 / 15.9, 1500x3000x2000 9.4 / 6.9).
Status timeVariants(HipContext* ctx, MatMulResident& r, const std::vector<int>& cands, std::vector<float>* ms) {
  constexpr int kRounds = 5;
  constexpr int kLaunches = 2;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  LC_HIP_TRY(hipEventCreate(&e0));
  if (hipEventCreate(&e1) != hipSuccess) {
    (void)hipEventDestroy(e0);
    return failHip(hipErrorOutOfMemory, "matmul autotune events");
  }
  std::vector<std::vector<float>> samples(cands.size());
  float slowest = std::numeric_limits<float>::max();  // whose first sample is above it takes no more
  hipError_t e = hipSuccess;
  for (int round = -1; round < kRounds && e == hipSuccess; ++round) {
    for (std::size_t c = 0; c < cands.size() && e == hipSuccess; ++c) {
      if (!samples[c].empty() && samples[c][0] > slowest) {
        continue;
      }
      e = hipEventRecord(e0, ctx->stream);
      for (int l = 0; l < kLaunches && e == hipSuccess; ++l) {
        e = launchGemm(ctx, r, cands[c]);
      }
      if (e == hipSuccess) e = hipEventRecord(e1, ctx->stream);
      if (e == hipSuccess) e = hipEventSynchronize(e1);
      float t = 0.0f;
      if (e == hipSuccess) e = hipEventElapsedTime(&t, e0, e1);
      if (round >= 0) {
        samples[c].push_back(t);
      }
    }
    if (round == 0 && e == hipSuccess && isHalf(r.dtype)) {
      float best = samples[0][0];
      for (const auto& v : samples) {
        best = std::min(best, v[0]);
      }
      if (best >= 0.02f * kLaunches) {
        slowest = 1.5f * best;
      }
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (e != hipSuccess) {
    return failHip(e, "matmul autotune");
  }
  ms->clear();
  for (auto& v : samples) {
    std::sort(v.begin(), v.end());
    ms->push_back(v[v.size() / 2]);
  }
  return Status::kSuccess;
}

// fp32: the split GEMM where its planes fit, else whole tiles or stream-K, and
// those as well for the shortest k, where loads and stores are all there is: one
// 64-deep step in at most one 64x64 tile per CU, or up to three in more tiles
// whose rows no 16-byte store fits (us, them / the split GEMM): 948x45x631 5.7 /
// 6.9, 710x51x1918 8.3 / 11.6, 3144x74x1342 21.7 / 30.6; past the lines
// 1024x32x2816 11.4 / 9.7, 2048x80x1056 14.5 / 13.3.
// Over 500 shapes 0.2% behind the better of the two, 15% at worst.
int defaultF32Variant(const HipContext* ctx, std::size_t m, std::size_t k, std::size_t n) {
  const int M = static_cast<int>(m);
  const int N = static_cast<int>(n);
  const std::size_t kp = roundUp(k, kern::kF32GemmBK);
  const bool one_round = ((m + 63) / 64) * ((n + 63) / 64) <= static_cast<std::size_t>(cuCount(ctx));
  const bool short_k = one_round ? kp <= 64 : n % 4 != 0 && kp <= 192;
  if (short_k || !splitFits(ctx, m, k, n)) {
    return static_cast<int>(kern::gemmF32Choose(M, N, cuCount(ctx)));
  }
  return static_cast<int>(kern::gemmF32SplitChoose(M, N, static_cast<int>(kp), cuCount(ctx)));
}

// 16 bits: the skinny kernel up to 16 rows, 256x256 tiles while there is one
// per CU, else the smaller tiles of gemm_half.hip (within its 32-bit offsets)
// unless the product is mostly stores: few k steps, or rows of C that no 16-byte
// store fits, in more than a few tiles.  There the register-staged kernels,
// several workgroups a CU, hide the stores (us, them / the ring tiles):
// 7044x157x1759 19.7 / 44.7, 1360x581x6939 29.0 / 42.9, 6208x64x832 9.4 / 12.5,
// 2304x384x5760 24.9 / 29.1; past the lines 13568x384x704 21.8 / 22.6,
// 1920x640x6656 34.1 / 37.5, 1500x3000x2000 39.6 / 22.9.  Over 440 shapes the rule's
// choice is 0.5% behind the better of the two, 14% at worst.
int defaultHalfVariant(const HipContext* ctx, std::size_t m, std::size_t k, std::size_t n) {
  const int M = static_cast<int>(m);
  const int N = static_cast<int>(n);
  const kern::GemmHalfVariant v = kern::gemmHalfChoose(M, N);
  const int kp = static_cast<int>(roundUp(k, kern::kHalfGemmBK));
  if ((v == kern::GemmHalfVariant::kMid || v == kern::GemmHalfVariant::kSmall) && kern::gemmHalfR4Fits(kp, kp)) {
    const bool stores = ((m + 127) / 128) * ((n + 127) / 128) >= 64 && kp <= (n % 4 == 0 ? 384 : 1280);
    if (!stores) {
      return static_cast<int>(kern::gemmHalfR4Choose(M, N, kp, cuCount(ctx)));
    }
  }
  return static_cast<int>(v);
}

bool forcedVariant(bool half) { return std::getenv(half ? "CJ_HIP_GEMM_TILE" : "CJ_HIP_GEMM_F32") != nullptr; }

// `preferred` (the heuristic's choice) unless another candidate is clearly
// faster (3%: below that the measurement cannot tell them apart); candidates
// past `accept` do not count.
template <typename Accept>
int fastest(const std::vector<int>& cands, const std::vector<float>& ms, int preferred, Accept accept) {
  float ref_ms = 0.0f;
  for (std::size_t c = 0; c < ms.size(); ++c) {
    if (cands[c] == preferred) {
      ref_ms = ms[c];
    }
  }
  int best = preferred;
  float best_ms = ref_ms > 0.0f ? ref_ms * 0.97f : 0.0f;
  for (std::size_t c = 0; c < ms.size(); ++c) {
    if (accept(cands[c]) && (best_ms <= 0.0f || ms[c] < best_ms)) {
      best_ms = ms[c];
      best = cands[c];
    }
  }
  return best;
}

int defaultOnceVariant(const HipContext* ctx, const MatMulResident& r) {
  return static_cast<int>(kern::gemmF32Choose(static_cast<int>(r.m), static_cast<int>(r.n), cuCount(ctx)));
}

void recordChoices(HipContext* ctx, const MatMulResident& r, const Choices& c) {
  if (infoOf(isHalf(r.dtype), c.once) == nullptr) {
    return;
  }
  tuneRecord(r.m, r.k, r.n, static_cast<int>(r.dtype), baseArch(ctx), entryFor(isHalf(r.dtype), c));
}

// Settles r.once (fp32): a tune-cache entry, else (CJ_MATMUL_AUTOTUNE not off)
// the faster of whole tiles and stream-K, else the heuristic; the choice is
// recorded.  CJ_HIP_GEMM_F32 (a sweep override) bypasses all of it.
Status settleOnce(HipContext* ctx, MatMulResident& r) {
  if (r.once_tuned) {
    return Status::kSuccess;
  }
  r.once = 0;
  if (!forcedVariant(false)) {
    Choices c = cachedChoices(ctx, r);
    if (c.once == 0) {
      const std::vector<int> cands = {static_cast<int>(kern::GemmF32Variant::kDataParallel),
                                      static_cast<int>(kern::GemmF32Variant::kStreamK)};
      std::vector<float> ms;
      if (autotuneEnabled("CJ_MATMUL_AUTOTUNE")) {
        LC_TRY(timeVariants(ctx, r, cands, &ms));
      }
      c.once = fastest(cands, ms, defaultOnceVariant(ctx, r), [](int) { return true; });
      recordChoices(ctx, r, c);
    }
    r.once = c.once;
  }
  r.once_tuned = true;
  return Status::kSuccess;
}

// Settles r.variant likewise, over every candidate for the shape and dtype.
// CJ_HIP_GEMM_F32 / CJ_HIP_GEMM_TILE bypass it.
Status settleVariant(HipContext* ctx, MatMulResident& r) {
  if (r.tuned) {
    return Status::kSuccess;
  }
  const bool half = isHalf(r.dtype);
  r.variant = 0;
  if (forcedVariant(half)) {
    r.tuned = true;
    return Status::kSuccess;
  }
  Choices c = cachedChoices(ctx, r);
  if (c.resident != 0) {
    r.variant = c.resident;
    r.tuned = true;
    return Status::kSuccess;
  }
  const bool timed = autotuneEnabled("CJ_MATMUL_AUTOTUNE");
  std::vector<int> cands;
  if (!half) {
    cands = {static_cast<int>(kern::GemmF32Variant::kDataParallel), static_cast<int>(kern::GemmF32Variant::kStreamK)};
    if (splitFits(ctx, r.m, r.k, r.n)) {
      if (timed) {
        // A split variant's time is that of operands it takes.  With others (the
        // scans of both have run after this sync) nothing is settled or recorded.
        LC_TRY(syncStream(ctx));
        if (knownUnsafe(ctx, r)) {
          LC_TRY(settleOnce(ctx, r));
          r.variant = r.once;
          return Status::kSuccess;
        }
      }
      for (const VariantInfo& v : kF32Variants) {
        if (isSplit(v.variant)) {
          cands.push_back(v.variant);
        }
      }
    }
  } else if (r.m > 16) {
    // w4, w4d, big8 and big4 were never more than 3% ahead of all of these over
    // 440 shapes (17-16384 x 64-8192 x 64-8192); they stay for a tune cache or
    // CJ_HIP_GEMM_TILE that names them.
    cands = {static_cast<int>(kern::GemmHalfVariant::kW4H), static_cast<int>(kern::GemmHalfVariant::kW4R),
             static_cast<int>(kern::GemmHalfVariant::kLds), static_cast<int>(kern::GemmHalfVariant::kMid),
             static_cast<int>(kern::GemmHalfVariant::kSmall)};
    const long long k_pad = static_cast<long long>(roundUp(r.k, kern::kHalfGemmBK));
    for (const VariantInfo& v : kHalfVariants) {
      if (kern::isR4(static_cast<kern::GemmHalfVariant>(v.variant)) && kern::gemmHalfR4Fits(k_pad, k_pad)) {
        cands.push_back(v.variant);
      }
    }
  }
  std::vector<float> ms;
  if (cands.size() > 1 && timed) {
    LC_TRY(timeVariants(ctx, r, cands, &ms));
  }
  c.resident = fastest(cands, ms, half ? defaultHalfVariant(ctx, r.m, r.k, r.n) : defaultF32Variant(ctx, r.m, r.k, r.n),
                       [](int) { return true; });
  if (half) {
    c.once = c.resident;
  } else if (c.once == 0) {
    c.once = fastest(cands, ms, defaultOnceVariant(ctx, r), [](int v) { return !isSplit(v); });
  }
  recordChoices(ctx, r, c);
  r.variant = c.resident;
  r.tuned = true;
  return Status::kSuccess;
}

// The variant of a launch.  A call that uploads an fp32 operand and launches
// once keeps the fp32 instruction below 2^32 products: the planes of a new
// operand cost 5 us (256^3) to 12 us (2048^3), more than the split GEMM saves
// there (1024^3: 6.4 + 16.1 us against 22.3).  That depends on the call alone,
// so equal calls give equal bits whatever ran before them.
Status launchVariant(HipContext* ctx, MatMulResident& r, bool one_shot, int* variant) {
  if (one_shot && !isHalf(r.dtype) && r.m * r.k * r.n < (std::size_t{1} << 32)) {
    LC_TRY(settleOnce(ctx, r));
    *variant = r.once;
    return Status::kSuccess;
  }
  if (!isHalf(r.dtype) && knownUnsafe(ctx, r) && (!r.tuned || isSplit(r.variant))) {
    LC_TRY(settleOnce(ctx, r));
    *variant = r.once;
    return Status::kSuccess;
  }
  LC_TRY(settleVariant(ctx, r));
  *variant = r.variant;
  return Status::kSuccess;
}

// Small fp32 calls that upload both operands and download the product (the
// plain matmul2d call) spend most of their time in per-copy overhead: two
// pageable uploads and a pageable download at ~10 us each, and the stream
// sync.  Here A and B are packed into pinned staging and the padding kernels
// read them through its device alias (each value crosses the bus once); after
// the GEMM one kernel copies C into the staging and raises the host-mapped
// completion flag, which the call waits for instead of a stream sync.
constexpr std::size_t kQuickMatMulElems = std::size_t{1} << 18;  // per operand and the product

bool quickMatMulEnabled() {
  static const bool on = [] {
    const char* v = std::getenv("CJ_HIP_MATMUL_QUICK");
    return v == nullptr || std::string(v) != "0";
  }();
  return on;
}

Status matmulQuick(HipContext* ctx, MatMulResident& r, const float* a, const float* b, float* out) {
  const std::size_t na = r.m * r.k, nb = r.k * r.n, nc = r.m * r.n;
  const std::size_t b_at = roundUp(na, 64);  // 256-byte aligned parts
  const std::size_t c_at = roundUp(b_at + nb, 64);
  const std::size_t mp = roundUp(r.m, kern::kF32GemmBM);
  const std::size_t kp = roundUp(r.k, kern::kF32GemmBK);
  const std::size_t np = roundUp(r.n, kern::kF32GemmBN);
  LC_TRY(ctx->pinned.ensure((c_at + nc) * sizeof(float)));
  LC_TRY(r.a.ensure(mp * kp * sizeof(float)));
  LC_TRY(r.b.ensure(kp * np * sizeof(float)));
  LC_TRY(r.c.ensure(nc * sizeof(float)));
  float* stage = static_cast<float*>(ctx->pinned.get());
  float* dev = static_cast<float*>(ctx->pinned.device());
  std::memcpy(stage, a, na * sizeof(float));
  std::memcpy(stage + b_at, b, nb * sizeof(float));
  const GuardArgs ga = beginUpload(ctx, r, 0);
  const GuardArgs gb = beginUpload(ctx, r, 1);
  hipError_t e = kern::padCopyF32(dev, r.a.as<float>(), static_cast<int>(r.m), static_cast<int>(r.k), r.k,
                                  static_cast<int>(mp), static_cast<int>(kp), ctx->stream, ga.word, ga.host,
                                  ga.epoch);
  if (e == hipSuccess) {
    e = kern::padCopyF32(dev + b_at, r.b.as<float>(), static_cast<int>(r.k), static_cast<int>(r.n), r.n,
                         static_cast<int>(kp), static_cast<int>(np), ctx->stream, gb.word, gb.host, gb.epoch);
  }
  if (e != hipSuccess) {
    return failHip(e, "matmul upload padding");
  }
  r.has_a = r.has_b = true;
  int variant = 0;
  LC_TRY(launchVariant(ctx, r, true, &variant));
  unsigned* flag_dev = nullptr;
  unsigned* count_dev = nullptr;
  unsigned seq = 0;
  LC_TRY(prepareDoneFlag(ctx, &flag_dev, &count_dev, &seq));
  traceOpDispatch(TraceOp::kMatMul, Device::kHIP, Device::kHIP, false, r.m * r.k * r.n);
  e = launchGemm(ctx, r, variant);
  if (e != hipSuccess) {
    return failHip(e, "matmul kernel launch");
  }
  r.has_c = true;
  e = kern::copyOutFlagF32(r.c.as<float>(), dev + c_at, nc, count_dev, flag_dev, seq, ctx->stream);
  if (e != hipSuccess) {
    return failHip(e, "matmul output copy");
  }
  LC_TRY(waitDoneFlag(ctx, seq));
  std::memcpy(out, stage + c_at, nc * sizeof(float));
  return Status::kSuccess;
}

}  // namespace

Status matmulResident(HipContext* ctx, MatMulResident& r, std::size_t m, std::size_t k, std::size_t n,
                      lcDataType dtype, const float* a, const float* b, float* out, const lcMatMulIoPolicy& policy,
                      std::size_t repeat) {
  if ((policy.upload_a && a == nullptr) || (policy.upload_b && b == nullptr) ||
      (policy.download_out && out == nullptr) || m == 0 || k == 0 || n == 0) {
    return fail(Status::kInvalidValue, "matmul: null pointer required by the io policy or zero dimension");
  }
  if (!validDtype(dtype)) {
    return fail(Status::kInvalidValue, "matmul: unknown compute dtype");
  }
  if (m > (1u << 30) / 1 || k > (1u << 30) || n > (1u << 30) || m * k > (std::size_t(1) << 34) ||
      k * n > (std::size_t(1) << 34) || m * n > (std::size_t(1) << 34)) {
    return fail(Status::kNotSupported, "matmul: shape too large");
  }
  if (r.m != m || r.k != k || r.n != n || r.dtype != dtype) {
    r.has_a = r.has_b = r.has_c = false;
    r.tuned = r.once_tuned = false;
    r.variant = r.once = 0;
    r.m = m;
    r.k = k;
    r.n = n;
    r.dtype = dtype;
  }
  if ((!policy.upload_a && !r.has_a) || (!policy.upload_b && !r.has_b)) {
    return fail(Status::kInvalidValue, "matmul: no resident input for an operand the policy does not upload");
  }
  if (!isHalf(dtype) && repeat == 1 && policy.upload_a && policy.upload_b && policy.download_out &&
      std::max({m * k, k * n, m * n}) <= kQuickMatMulElems && quickMatMulEnabled()) {
    return matmulQuick(ctx, r, a, b, out);
  }
  if (policy.upload_a) {
    LC_TRY(uploadA(ctx, r, a));
    r.has_a = true;
  }
  if (policy.upload_b) {
    LC_TRY(uploadB(ctx, r, b));
    r.has_b = true;
  }
  LC_TRY(r.c.ensure(m * n * sizeof(float)));
  const std::size_t hint = m * k * n;
  int variant = 0;
  if (repeat > 0) {
    const bool one_shot = repeat == 1 && policy.download_out && (policy.upload_a || policy.upload_b);
    LC_TRY(launchVariant(ctx, r, one_shot, &variant));
  }
  for (std::size_t i = 0; i < repeat; ++i) {
    traceOpDispatch(TraceOp::kMatMul, Device::kHIP, Device::kHIP, false, hint);
    const hipError_t e = launchGemm(ctx, r, variant);
    if (e != hipSuccess) {
      return failHip(e, "matmul kernel launch");
    }
  }
  r.has_c = true;
  if (policy.download_out && m * n <= kStagedDownloadMax && quickMatMulEnabled()) {
    const StagedOut o{r.c.as<float>(), out, m * n};
    return stagedDownload(ctx, &o, 1);
  }
  if (policy.download_out) {
    LC_TRY(download(ctx, out, r.c.get(), m * n * sizeof(float)));
  }
  if (policy.download_out || policy.synchronize) {
    LC_TRY(syncStream(ctx));
  } else if (repeat > 0) {
    LC_TRY(noteEnqueued(ctx, TraceOp::kMatMul, repeat));
  }
  return Status::kSuccess;
}

namespace {

MatMulResident& globalMatMulResident() {
  static MatMulResident* r = new MatMulResident();  // process lifetime
  return *r;
}

Status matmulPolicyEntry(const float* a, const float* b, float* out, std::size_t m, std::size_t k, std::size_t n,
                         lcDeviceKind device, const lcMatMulIoPolicy& policy, std::size_t repeat,
                         lcDataType dtype) {
  if ((policy.upload_a && a == nullptr) || (policy.upload_b && b == nullptr) ||
      (policy.download_out && out == nullptr) || m == 0 || k == 0 || n == 0) {
    return fail(Status::kInvalidValue, "matmul: null pointer required by the io policy or zero dimension");
  }
  HipContext* ctx = nullptr;
  LC_TRY(requireHip(device, "matmul", &ctx));
  std::lock_guard<std::recursive_mutex> lock(ctx->mu);
  return matmulResident(ctx, globalMatMulResident(), m, k, n, dtype, a, b, out, policy, repeat);
}

}  // namespace
}  // namespace lchip

using namespace lchip;

struct lcMatMulResidentSession {
  MatMulResident res;
  std::size_t m = 0, k = 0, n = 0;
  lcDataType dtype = LC_DTYPE_F32;
};

namespace {

lcMatMulIoPolicy makePolicy(int ua, int ub, int dl, int sync) {
  lcMatMulIoPolicy p{};
  p.upload_a = ua;
  p.upload_b = ub;
  p.download_out = dl;
  p.synchronize = sync;
  return p;
}

lcError_t sessionCall(lcMatMulResidentSession* s, const float* a, const float* b, float* out,
                      const lcMatMulIoPolicy& p, std::size_t repeat) {
  if (s == nullptr) {
    return toLc(fail(Status::kInvalidValue, "matmul session: null session"));
  }
  HipContext* ctx = nullptr;
  Status st = requireHip(LC_DEVICE_HIP, "matmul session", &ctx);
  if (st != Status::kSuccess) {
    return toLc(st);
  }
  std::lock_guard<std::recursive_mutex> lock(ctx->mu);
  return toLc(matmulResident(ctx, s->res, s->m, s->k, s->n, s->dtype, a, b, out, p, repeat));
}

}  // namespace

extern "C" {

lcMatMulIoPolicy lcMatMulIoPolicyDefault(void) { return makePolicy(1, 1, 1, 1); }

lcError_t lcMatMul(const float* a, const float* b, float* out, size_t m, size_t k, size_t n, lcDeviceKind device) {
  return toLc(matmulPolicyEntry(a, b, out, m, k, n, device, makePolicy(1, 1, 1, 1), 1, LC_DTYPE_F32));
}

lcError_t lcMatMulWithPolicy(const float* a, const float* b, float* out, size_t m, size_t k, size_t n,
                             lcDeviceKind device, const lcMatMulIoPolicy* policy) {
  const lcMatMulIoPolicy p = policy ? *policy : makePolicy(1, 1, 1, 1);
  return toLc(matmulPolicyEntry(a, b, out, m, k, n, device, p, 1, LC_DTYPE_F32));
}

lcError_t lcMatMulWithPolicyBatched(const float* a, const float* b, float* out, size_t m, size_t k, size_t n,
                                    lcDeviceKind device, const lcMatMulIoPolicy* policy, size_t repeat_count) {
  if (repeat_count == 0) {
    return toLc(fail(Status::kInvalidValue, "matmul: repeat_count must be > 0"));
  }
  const lcMatMulIoPolicy p = policy ? *policy : makePolicy(1, 1, 1, 1);
  return toLc(matmulPolicyEntry(a, b, out, m, k, n, device, p, repeat_count, LC_DTYPE_F32));
}

lcError_t lcMatMulResidentSessionCreate(size_t m, size_t k, size_t n, lcDataType compute_dtype,
                                        lcMatMulResidentSession** out) {
  if (out == nullptr || m == 0 || k == 0 || n == 0 || !validDtype(compute_dtype)) {
    return toLc(fail(Status::kInvalidValue, "matmul session: invalid arguments"));
  }
  HipContext* ctx = nullptr;
  Status st = requireHip(LC_DEVICE_HIP, "matmul session", &ctx);
  if (st != Status::kSuccess) {
    return toLc(st);
  }
  auto* s = new lcMatMulResidentSession();
  s->m = m;
  s->k = k;
  s->n = n;
  s->dtype = compute_dtype;
  *out = s;
  return LC_SUCCESS;
}

lcError_t lcMatMulResidentSessionDestroy(lcMatMulResidentSession* s) {
  if (s == nullptr) {
    return LC_INVALID_VALUE;
  }
  Status st = Status::kSuccess;
  HipContext* ctx = hipContext(&st);
  if (ctx != nullptr) {
    std::lock_guard<std::recursive_mutex> lock(ctx->mu);
    (void)hipStreamSynchronize(ctx->stream);
    releaseGuard(ctx, &s->res.guard_slot);
    dropSpare(ctx, &s->res.planes);
  }
  delete s;
  return LC_SUCCESS;
}

// ops.hpp:207-216 / policy.hpp:37-44: upload both, no download, no sync.
lcError_t lcMatMulResidentSessionStart(lcMatMulResidentSession* s, const float* a, const float* b, float* out) {
  return sessionCall(s, a, b, out, makePolicy(1, 1, 0, 0), 1);
}
// ops.hpp:218-227 / policy.hpp:46-53: launch only.
lcError_t lcMatMulResidentSessionRun(lcMatMulResidentSession* s, const float* a, const float* b, float* out) {
  return sessionCall(s, a, b, out, makePolicy(0, 0, 0, 0), 1);
}
// ops.hpp:229-238 / policy.hpp:55-62: launch, download, sync.
lcError_t lcMatMulResidentSessionFinish(lcMatMulResidentSession* s, const float* a, const float* b, float* out) {
  return sessionCall(s, a, b, out, makePolicy(0, 0, 1, 1), 1);
}
// ops.hpp:240-249 / policy.hpp:64-71: launch, sync, no download.
lcError_t lcMatMulResidentSessionSync(lcMatMulResidentSession* s, const float* a, const float* b, float* out) {
  return sessionCall(s, a, b, out, makePolicy(0, 0, 0, 1), 1);
}
// ops.hpp:251-299: repeat launches over the resident inputs, then sync.  As
// in the reference (upload=false, download=false, sync=true passed to the
// batched backend), the pointers must be non-null but are not read or written;
// finish() downloads the result.
lcError_t lcMatMulResidentSessionRunBatchSync(lcMatMulResidentSession* s, const float* a, const float* b, float* out,
                                              size_t repeat_count) {
  if (repeat_count == 0 || a == nullptr || b == nullptr || out == nullptr) {
    return toLc(fail(Status::kInvalidValue, "matmul session: run_batch_sync needs pointers and repeat_count > 0"));
  }
  return sessionCall(s, nullptr, nullptr, nullptr, makePolicy(0, 0, 0, 1), repeat_count);
}
// ops.hpp:301-352: repeat launches, sync, no download.
lcError_t lcMatMulResidentSessionRunBatchSyncNoDownload(lcMatMulResidentSession* s, const float* a, const float* b,
                                                        float* out, size_t repeat_count) {
  (void)a;
  (void)b;
  (void)out;
  if (repeat_count == 0) {
    return toLc(fail(Status::kInvalidValue, "matmul session: repeat_count must be > 0"));
  }
  return sessionCall(s, nullptr, nullptr, nullptr, makePolicy(0, 0, 0, 1), repeat_count);
}
// ops.hpp:1371-1373: the same with null pointers.
lcError_t lcMatMulResidentSessionRunBatchSyncCachedNoDownload(lcMatMulResidentSession* s, size_t repeat_count) {
  return lcMatMulResidentSessionRunBatchSyncNoDownload(s, nullptr, nullptr, nullptr, repeat_count);
}

lcError_t lcMatMulResidentSessionTimeLaunches(lcMatMulResidentSession* s, size_t count, float* ms_out) {
  if (s == nullptr || count == 0 || ms_out == nullptr) {
    return toLc(fail(Status::kInvalidValue, "matmul session: null session or output, or count 0"));
  }
  HipContext* ctx = nullptr;
  Status st = requireHip(LC_DEVICE_HIP, "matmul session", &ctx);
  if (st != Status::kSuccess) {
    return toLc(st);
  }
  std::lock_guard<std::recursive_mutex> lock(ctx->mu);
  MatMulResident& r = s->res;
  if (!r.has_a || !r.has_b || r.m != s->m || r.k != s->k || r.n != s->n || r.dtype != s->dtype) {
    return toLc(fail(Status::kInvalidValue, "matmul session: no resident inputs to time (start the session first)"));
  }
  int variant = 0;
  st = launchVariant(ctx, r, false, &variant);
  if (st != Status::kSuccess) {
    return toLc(st);
  }
  std::vector<hipEvent_t> ev(2 * count, nullptr);
  hipError_t e = hipSuccess;
  for (std::size_t i = 0; i < ev.size() && e == hipSuccess; ++i) {
    e = hipEventCreate(&ev[i]);
  }
  for (std::size_t i = 0; i < count && e == hipSuccess; ++i) {
    e = hipEventRecord(ev[2 * i], ctx->stream);
    if (e == hipSuccess) {
      traceOpDispatch(TraceOp::kMatMul, Device::kHIP, Device::kHIP, false, r.m * r.k * r.n);
      e = launchGemm(ctx, r, variant);
    }
    if (e == hipSuccess) {
      e = hipEventRecord(ev[2 * i + 1], ctx->stream);
    }
  }
  if (e == hipSuccess) {
    e = hipStreamSynchronize(ctx->stream);
  }
  for (std::size_t i = 0; i < count && e == hipSuccess; ++i) {
    e = hipEventElapsedTime(&ms_out[i], ev[2 * i], ev[2 * i + 1]);
  }
  for (hipEvent_t x : ev) {
    if (x != nullptr) {
      (void)hipEventDestroy(x);
    }
  }
  if (e != hipSuccess) {
    return toLc(failHip(e, "matmul session: timed launches"));
  }
  r.has_c = true;
  return toLc(syncStream(ctx));
}

lcError_t lcMatMulResidentSessionKernelName(lcMatMulResidentSession* s, char* buf, size_t cap) {
  if (s == nullptr || buf == nullptr || cap == 0) {
    return toLc(fail(Status::kInvalidValue, "matmul session: null session or buffer"));
  }
  HipContext* ctx = nullptr;
  Status st = requireHip(LC_DEVICE_HIP, "matmul session", &ctx);
  if (st != Status::kSuccess) {
    return toLc(st);
  }
  std::lock_guard<std::recursive_mutex> lock(ctx->mu);
  const bool half = isHalf(s->dtype);
  const MatMulResident& r = s->res;
  int v = r.tuned ? r.variant : 0;
  if (v == 0) {
    v = half ? defaultHalfVariant(ctx, s->m, s->k, s->n) : defaultF32Variant(ctx, s->m, s->k, s->n);
  }
  // Operands the split GEMM does not take, planes past their limit or without
  // memory: the fp32 instruction's variant runs.
  if (!half && isSplit(v) &&
      (!splitFits(ctx, s->m, s->k, s->n) || r.planes_denied == ctx->frees || (r.has_a && r.has_b && knownUnsafe(ctx, r)))) {
    v = r.once;
    if (v == 0) {
      v = static_cast<int>(kern::gemmF32Choose(static_cast<int>(s->m), static_cast<int>(s->n), cuCount(ctx)));
    }
  }
  std::string text;
  for (const VariantInfo& info : variants(half)) {
    if (info.variant == v) {
      text = std::string(info.name) + " " + info.hip_kernel;
    }
  }
  if (text.empty()) {
    return toLc(fail(Status::kUnknown, "matmul session: unknown variant"));
  }
  std::snprintf(buf, cap, "%s", text.c_str());
  return LC_SUCCESS;
}

}  // extern "C"
