// gemm_half.hip -- 16-bit TN GEMM (C = A . Bt^T, fp32 accumulate and output)
// for problems with too few 256x256 tiles to fill the chip, and for few rows.
#include <type_traits>

#include "../kernels.hpp"
#include "gemm_tiles.hpp"
#include "kcommon.hpp"

namespace lchip::k {

// ---------------------------------------------------------------------------
// Four waves in 2 x 2, each 16 RM x 16 CN of a 32 RM x 32 CN tile; LDS is a
// ring of four 64-deep stages (128-byte rows, chunk c of row r at
// c ^ ((r >> 1) & 7), as in gemm_half_tn_w4h_kernel).  A wave reads all of a
// stage's fragments into registers during the stage before it, so a stage is
// one barrier and its slot is free for the copies of the stage four ahead as
// soon as the barrier is passed.
// Bound: LDS bandwidth for the 128- and 96-row tiles (a stage reads and writes
// 84-96 KB for 24-32 MFMAs a wave, 670-770 cycles at 128 bytes a cycle against
// 384-512 of MFMA; measured 0.43-0.45 us a stage), the stream of Bt from HBM
// for few rows.  The k order of every accumulator is that of the 256x256
// kernels, so results agree bit for bit.
// Measured against the best of the register-staged kernels and w4h, f16
// (M x K x N, us): 1500x3000x2000 38.4 -> 24.4 (96x128); 2048^3 32.7 -> 23.5
// (128x128); 1000x4096x4096 56.8 -> 38.6; 1024^3 8.6 -> 6.0 (64x64);
// 200x1000x5000 10.9 -> 7.4 (64x128); 64x8192x8192 70.6 -> 25.1 (32x64, Bt at
// 5.4 TB/s); 32x4096x8192 37 -> 13.0.  Sharing a tile's k range between two
// workgroups gained only at 128x4096x4096 (13.8 -> 12.4 with 64x64, where the
// 32x64 tile already takes 12.7), so tiles are never split.
// A has rows_a and Bt rows_b readable rows (tile rows past them read the last
// one and are never stored); K is padded to 64; 32-bit lane offsets (the host
// keeps 256 * ld * 2 bytes below 2^31).
// ---------------------------------------------------------------------------
template <typename T, int RM, int CN>
__global__ __launch_bounds__(256) void gemm_half_tn_r4_kernel(const uint16_t* __restrict__ A,
                                                              const uint16_t* __restrict__ Bt, float* __restrict__ C,
                                                              int M, int N, int K, int rows_a, int rows_b,
                                                              int lda, int ldb, int ldc, int tiles_m, int tiles_n,
                                                              int vec4) {
  constexpr int BM = 32 * RM;
  constexpr int BN = 32 * CN;
  constexpr int NS = 4;
  constexpr int A_BYTES = BM * 128;
  constexpr int STAGE = A_BYTES + BN * 128;
  constexpr int CPS = RM + CN;  // copies a wave makes of a stage (8 rows each)
  __shared__ __attribute__((aligned(16))) char smem[NS * STAGE];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1;
  const int wn = wave & 1;
  const int lr = lane & 15;
  const int lq = lane >> 4;
  int bm, bn;
  tile_origin<8>(tiles_m, tiles_n, BM, BN, bm, bn);
  const int S = K / 64;

  // Copy j of this wave fills rows 8 (wave RM + j) .. + 7 of the A part, then
  // rows 8 (wave CN + j - RM) .. of the Bt part.
  const int crow = lane >> 3;
  const int pch = lane & 7;
  uint32_t off[CPS];
#pragma unroll
  for (int j = 0; j < CPS; ++j) {
    const int row = j < RM ? 8 * (wave * RM + j) + crow : 8 * (wave * CN + j - RM) + crow;
    const int lch = pch ^ ((row >> 1) & 7);
    const int src = j < RM ? min(bm + row, rows_a - 1) - bm : min(bn + row, rows_b - 1) - bn;
    off[j] = static_cast<uint32_t>(src * (j < RM ? lda : ldb) + lch * 8) * 2u;
  }
  const char* a_tile = reinterpret_cast<const char*>(A + static_cast<size_t>(bm) * lda);
  const char* b_tile = reinterpret_cast<const char*>(Bt + static_cast<size_t>(bn) * ldb);
  const uint32_t lds0 = lds_addr(smem);
  auto copy = [&](int j, int s, int slot) {  // stages past the last: that one again, unused
    const size_t k = static_cast<size_t>(min(s, S - 1)) * 128;
    const uint32_t dst = lds0 + static_cast<uint32_t>(slot * STAGE) +
                         (j < RM ? static_cast<uint32_t>(wave * RM + j) * 1024u
                                 : A_BYTES + static_cast<uint32_t>(wave * CN + j - RM) * 1024u);
    load_lds16_sbase(off[j], (j < RM ? a_tile : b_tile) + k, dst);
  };

  floatx4 acc[RM][CN];
#pragma unroll
  for (int i = 0; i < RM; ++i) {
#pragma unroll
    for (int j = 0; j < CN; ++j) {
      acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  // Fragment f of a stage: k step f / (RM + CN), then the wave's A blocks, then
  // its Bt blocks; lane l reads row l % 16, chunk 4 step + l / 16.
  typedef __attribute__((address_space(3))) const char lds_char;
  typedef __attribute__((address_space(3))) const u32x4 lds_u32x4;
  lds_char* fa[2];
  lds_char* fb[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const int o = lr * 128 + (((4 * kk + lq) ^ ((lr >> 1) & 7)) << 4);
    fa[kk] = (lds_char*)(smem) + wm * RM * 2048 + o;
    fb[kk] = (lds_char*)(smem) + A_BYTES + wn * CN * 2048 + o;
  }
  constexpr int NF = 2 * CPS;
  auto frag = [&](int f, int slot) -> u32x4 {
    const int kk = f / CPS;
    const int b = f % CPS;
    return *reinterpret_cast<lds_u32x4*>((b < RM ? fa[kk] + b * 2048 : fb[kk] + (b - RM) * 2048) + slot * STAGE);
  };
#pragma unroll
  for (int s = 0; s < NS; ++s) {
#pragma unroll
    for (int j = 0; j < CPS; ++j) {
      copy(j, s, s);
    }
  }
  wait_vmcnt<(NS - 1) * CPS>();
  __builtin_amdgcn_s_waitcnt(0xc07f);  // no scalar load pending in the loop
  stage_barrier();
  u32x4 fr[2][NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    fr[0][f] = frag(f, 0);
  }
  auto body = [&](auto phase, int s) {
    constexpr int SL = decltype(phase)::value;  // s % NS
    constexpr int P = SL % 2;
    constexpr int NM = 2 * RM * CN;
    wait_vmcnt<(NS - 2) * CPS>();  // this wave's copies of stage s + 1 have landed
    wait_lgkmcnt<0>();             // and its reads of stage s are done
    stage_barrier();
#pragma unroll
    for (int g = 0; g < NM; ++g) {
      const int kk = g / (RM * CN);
      const int i = g / CN % RM;
      const int j = g % CN;
      // Bt is the MFMAs' first operand: a lane holds four columns of one row
      acc[i][j] = mfma16x16x32<T>(fr[P][kk * CPS + RM + j], fr[P][kk * CPS + i], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int f = g * NF / NM; f < (g + 1) * NF / NM; ++f) {
        fr[P ^ 1][f] = frag(f, (SL + 1) % NS);
      }
#pragma unroll
      for (int c = g * CPS / NM; c < (g + 1) * CPS / NM; ++c) {
        copy(c, s + NS, SL);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (int s = 0; s < S; s += NS) {
    body(std::integral_constant<int, 0>{}, s);
    if (s + 1 < S) body(std::integral_constant<int, 1>{}, s + 1);
    if (s + 2 < S) body(std::integral_constant<int, 2>{}, s + 2);
    if (s + 3 < S) body(std::integral_constant<int, 3>{}, s + 3);
  }
  wait_vmcnt<0>();  // no copy may still be writing LDS
#pragma unroll
  for (int i = 0; i < RM; ++i) {
#pragma unroll
    for (int j = 0; j < CN; ++j) {
      store_c4(C, ldc, bm + 16 * (wm * RM + i) + lr, bn + 16 * (wn * CN + j) + 4 * lq, M, N, vec4, acc[i][j]);
    }
  }
}

template <typename T, int RM, int CN>
static hipError_t launch_r4(const uint16_t* A, const uint16_t* Bt, float* C, int M, int N, int K, int lda, int ldb,
                            int ldc, hipStream_t stream) {
  const int tiles_m = (M + 32 * RM - 1) / (32 * RM);
  const int tiles_n = (N + 32 * CN - 1) / (32 * CN);
  const int vec4 = (ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0) ? 1 : 0;
  hipLaunchKernelGGL((gemm_half_tn_r4_kernel<T, RM, CN>), dim3(tiles_m * tiles_n), dim3(256), 0, stream, A, Bt,
                     C, M, N, K, (M + kern::kHalfGemmBM - 1) / kern::kHalfGemmBM * kern::kHalfGemmBM,
                     (N + kern::kHalfGemmBN - 1) / kern::kHalfGemmBN * kern::kHalfGemmBN, lda, ldb, ldc, tiles_m,
                     tiles_n, vec4);
  return hipGetLastError();
}

template <typename T>
static hipError_t launch_r4_variant(kern::GemmHalfVariant v, const uint16_t* A, const uint16_t* Bt, float* C, int M,
                                    int N, int K, int lda, int ldb, int ldc, hipStream_t stream) {
  switch (v) {
    case kern::GemmHalfVariant::kR128:
      return launch_r4<T, 4, 4>(A, Bt, C, M, N, K, lda, ldb, ldc, stream);
    case kern::GemmHalfVariant::kR96:
      return launch_r4<T, 3, 4>(A, Bt, C, M, N, K, lda, ldb, ldc, stream);
    case kern::GemmHalfVariant::kR64x128:
      return launch_r4<T, 2, 4>(A, Bt, C, M, N, K, lda, ldb, ldc, stream);
    case kern::GemmHalfVariant::kR64:
      return launch_r4<T, 2, 2>(A, Bt, C, M, N, K, lda, ldb, ldc, stream);
    case kern::GemmHalfVariant::kR32:
      return launch_r4<T, 1, 2>(A, Bt, C, M, N, K, lda, ldb, ldc, stream);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace lchip::k

namespace lchip::kern {

GemmHalfVariant gemmHalfR4Choose(int M, int N, int K, int cus) {
  // A model of the measured times (us): per round of the workgroups that fit
  // the chip at once, a prologue and the stages; a tile whose workgroups have
  // CUs of their own runs a stage faster than one that shares them.
  struct Tile {
    GemmHalfVariant variant;
    int rows, cols, per_cu;
    double alone, shared;  // a stage
  };
  constexpr Tile kTiles[] = {{GemmHalfVariant::kR128, 128, 128, 1, 0.45, 0.45},
                             {GemmHalfVariant::kR96, 96, 128, 1, 0.42, 0.42},
                             {GemmHalfVariant::kR64x128, 64, 128, 1, 0.28, 0.30},
                             {GemmHalfVariant::kR64, 64, 64, 2, 0.19, 0.37},
                             {GemmHalfVariant::kR32, 32, 64, 3, 0.15, 0.40}};
  GemmHalfVariant best = GemmHalfVariant::kR128;
  double best_us = 0.0;
  for (const Tile& t : kTiles) {
    const long long tiles =
        static_cast<long long>((M + t.rows - 1) / t.rows) * ((N + t.cols - 1) / t.cols);
    const long long slots = static_cast<long long>(cus) * (tiles <= cus ? 1 : t.per_cu);
    const double us = static_cast<double>((tiles + slots - 1) / slots) *
                      (1.5 + (tiles <= cus ? t.alone : t.shared) * (K / 64));
    if (best_us == 0.0 || us < best_us) {
      best = t.variant;
      best_us = us;
    }
  }
  return best;
}

hipError_t gemmHalfR4(const uint16_t* A, const uint16_t* Bt, float* C, int M, int N, int K, int lda, int ldb, int ldc,
                      Half t, GemmHalfVariant variant, hipStream_t stream) {
  if (K <= 0 || K % kHalfGemmBK != 0 || M <= 0 || N <= 0 || !gemmHalfR4Fits(lda, ldb)) {
    return hipErrorInvalidValue;
  }
  return t == Half::kBF16
             ? k::launch_r4_variant<k::BF16>(variant, A, Bt, C, M, N, K, lda, ldb, ldc, stream)
             : k::launch_r4_variant<k::F16>(variant, A, Bt, C, M, N, K, lda, ldb, ldc, stream);
}

}  // namespace lchip::kern
