// gemm_half.hip -- 16-bit TN GEMM (C = A . Bt^T, fp32 accumulate and output)
// for problems with too few 256x256 tiles to fill the chip, and for few rows.
#include <type_traits>

#include "../kernels.hpp"
#include "gemm_tiles.hpp"
#include "kcommon.hpp"

namespace lchip::k {

// What happens to four consecutive columns n .. n + 3 of row m: row(m) and
// col(n) hold what the store needs of each, worked out once per lane and block.
struct StoreF32 {
  float* C;
  int ldc;
  int M, N;
  int vec4;  // C is 16-byte aligned and ldc % 4 == 0
  __device__ __forceinline__ int row(int m) const { return m; }
  __device__ __forceinline__ int col(int n) const { return n; }
  __device__ __forceinline__ void store(int m, int n, floatx4 v) const { store_c4(C, ldc, m, n, M, N, vec4, v); }
};

// relu(C) in 16 bits; N and ldc multiples of 4.
template <typename T>
struct StoreReluHalf {
  uint16_t* C;
  int ldc;
  int M, N;
  __device__ __forceinline__ int row(int m) const { return m; }
  __device__ __forceinline__ int col(int n) const { return n; }
  __device__ __forceinline__ void store(int m, int n, floatx4 v) const {
    if (m < M && n < N) {
      // (a comparison, as a NaN stays one)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = v[i] < 0.0f ? 0.0f : v[i];
      }
      u32x2 w;
      w[0] = pack2<T>(v[0], v[1]);
      w[1] = pack2<T>(v[2], v[3]);
      *reinterpret_cast<u32x2*>(C + static_cast<size_t>(m) * ldc + n) = w;
    }
  }
};

// Row m = b T_ + t, column n = which E + h Dh + d of the QKV projection to Q
// and K [b H + h][t][d] or V^T [b H + h][d][t]; Dh a multiple of 4.  A lane's
// four columns are one 8-byte store to Q or K; to V^T, 16 lanes of a row block
// write 32 contiguous bytes of each d.
template <typename T>
struct StoreQkv {
  uint16_t* q;
  uint16_t* k;
  uint16_t* vt;
  int M, T_, E, H, Dh, S_pad;
  struct Row {
    size_t image;  // b H S_pad Dh
    int t;         // -1: past the last row
  };
  struct Col {
    uint16_t* base;  // the head's part of Q, K or V^T
    int d;
    bool v;
  };
  __device__ __forceinline__ Row row(int m) const {
    const int b = m / T_;
    return {static_cast<size_t>(b) * H * S_pad * Dh, m < M ? m - b * T_ : -1};
  }
  __device__ __forceinline__ Col col(int n) const {
    const int which = n / E;
    const int r = n - which * E;
    const int h = r / Dh;
    return {(which == 0 ? q : which == 1 ? k : vt) + static_cast<size_t>(h) * S_pad * Dh, which < 3 ? r - h * Dh : -1,
            which == 2};
  }
  __device__ __forceinline__ void store(const Row& r, const Col& c, floatx4 x) const {
    if (r.t < 0 || c.d < 0) {
      return;
    }
    u32x2 w;
    w[0] = pack2<T>(x[0], x[1]);
    w[1] = pack2<T>(x[2], x[3]);
    uint16_t* p = c.base + r.image;
    if (!c.v) {
      *reinterpret_cast<u32x2*>(p + static_cast<size_t>(r.t) * Dh + c.d) = w;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[static_cast<size_t>(c.d + i) * S_pad + r.t] = static_cast<uint16_t>(w[i >> 1] >> (16 * (i & 1)));
      }
    }
  }
};

// ---------------------------------------------------------------------------
// Four waves in 2 x 2, each 16 RM x 16 CN of a 32 RM x 32 CN tile; LDS is a
// ring of four 64-deep stages (128-byte rows, chunk c of row r at
// c ^ ((r >> 1) & 7), as in gemm_half_tn_w4h_kernel).  A wave reads all of a
// stage's fragments into registers during the stage before it, so a stage is
// one barrier and its slot is free for the copies of the stage four ahead as
// soon as the barrier is passed.
// Bound: the copies and the barrier of each stage for the 128- and 96-row tiles
// (24-32 MFMAs a wave, 384-512 cycles, in a stage of 0.43-0.45 us: one wave per
// SIMD, MFMAs busy 50-55% of a CU's cycles and LDS reads 30%, no bank conflicts,
// at 1500x3000x2000), the stream of Bt from HBM for few rows.  The k order of
// every accumulator is that of the 256x256 kernels, so results agree bit for bit.
// Measured against the best of the register-staged kernels and w4h, f16
// (M x K x N, us): 1500x3000x2000 38.4 -> 24.4 (96x128); 2048^3 32.7 -> 23.5
// (128x128); 1000x4096x4096 56.8 -> 38.6; 1024^3 8.6 -> 6.0 (64x64);
// 200x1000x5000 10.9 -> 7.4 (64x128); 64x8192x8192 70.6 -> 25.1 (32x64, Bt at
// 5.4 TB/s); 32x4096x8192 37 -> 13.0.  Sharing a tile's k range between two
// workgroups gained only at 128x4096x4096 (13.8 -> 12.4 with 64x64, where the
// 32x64 tile already takes 12.7), so tiles are never split.
// The ViT block's GEMMs (M x 768 x 768, x 2304 for QKV) with these epilogues and
// a separate attention kernel, against 128-row tiles of 12 stages of their own
// and one kernel for QKV and attention (18.8 us already for one image, its
// serial chain; 64 us for 32, three rounds): block of 224 x 224 images 30.9 ->
// 18.8 us (batch 1), 32.7 -> 26.4 (4), 36.0 -> 33.9 (8), 67.7 -> 51 (16), 105.6
// -> 93 (32); of 112 x 112 images 24.1 -> 17.3 (1), 25.3 -> 19.4 (8), 49.5 ->
// 33.0 (32).
// A has rows_a and Bt rows_b readable rows (tile rows past them read the last
// one and are never stored); K is padded to 64; 32-bit lane offsets (the host
// keeps 256 * ld * 2 bytes below 2^31).
// ---------------------------------------------------------------------------
template <typename T, int RM, int CN, typename Epi>
__global__ __launch_bounds__(256) void gemm_half_tn_r4_kernel(const uint16_t* __restrict__ A,
                                                              const uint16_t* __restrict__ Bt, int K, int rows_a,
                                                              int rows_b, int lda, int ldb, int tiles_m, int tiles_n,
                                                              Epi epi) {
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
  decltype(epi.col(0)) col[CN];
#pragma unroll
  for (int j = 0; j < CN; ++j) {
    col[j] = epi.col(bn + 16 * (wn * CN + j) + 4 * lq);
  }
#pragma unroll
  for (int i = 0; i < RM; ++i) {
    const auto row = epi.row(bm + 16 * (wm * RM + i) + lr);
#pragma unroll
    for (int j = 0; j < CN; ++j) {
      epi.store(row, col[j], acc[i][j]);
    }
  }
}

template <typename T, int RM, int CN, typename Epi>
static hipError_t launch_r4(const uint16_t* A, const uint16_t* Bt, int M, int N, int K, int lda, int ldb, Epi epi,
                            hipStream_t stream) {
  const int tiles_m = (M + 32 * RM - 1) / (32 * RM);
  const int tiles_n = (N + 32 * CN - 1) / (32 * CN);
  hipLaunchKernelGGL((gemm_half_tn_r4_kernel<T, RM, CN, Epi>), dim3(tiles_m * tiles_n), dim3(256), 0, stream, A, Bt, K,
                     (M + kern::kHalfGemmBM - 1) / kern::kHalfGemmBM * kern::kHalfGemmBM,
                     (N + kern::kHalfGemmBN - 1) / kern::kHalfGemmBN * kern::kHalfGemmBN, lda, ldb, tiles_m, tiles_n,
                     epi);
  return hipGetLastError();
}

template <typename T, typename Epi>
static hipError_t launch_r4_variant(kern::GemmHalfVariant v, const uint16_t* A, const uint16_t* Bt, int M, int N, int K,
                                    int lda, int ldb, Epi epi, hipStream_t stream) {
  if (K <= 0 || K % kern::kHalfGemmBK != 0 || M <= 0 || N <= 0 || !kern::gemmHalfR4Fits(lda, ldb)) {
    return hipErrorInvalidValue;
  }
  switch (v) {
    case kern::GemmHalfVariant::kR128:
      return launch_r4<T, 4, 4>(A, Bt, M, N, K, lda, ldb, epi, stream);
    case kern::GemmHalfVariant::kR96:
      return launch_r4<T, 3, 4>(A, Bt, M, N, K, lda, ldb, epi, stream);
    case kern::GemmHalfVariant::kR64x128:
      return launch_r4<T, 2, 4>(A, Bt, M, N, K, lda, ldb, epi, stream);
    case kern::GemmHalfVariant::kR64:
      return launch_r4<T, 2, 2>(A, Bt, M, N, K, lda, ldb, epi, stream);
    case kern::GemmHalfVariant::kR32:
      return launch_r4<T, 1, 2>(A, Bt, M, N, K, lda, ldb, epi, stream);
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
  const int vec4 = (ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0) ? 1 : 0;
  const k::StoreF32 epi{C, ldc, M, N, vec4};
  return t == Half::kBF16 ? k::launch_r4_variant<k::BF16>(variant, A, Bt, M, N, K, lda, ldb, epi, stream)
                          : k::launch_r4_variant<k::F16>(variant, A, Bt, M, N, K, lda, ldb, epi, stream);
}

hipError_t gemmHalfR4Relu(const uint16_t* A, const uint16_t* Bt, uint16_t* C, int M, int N, int K, int lda, int ldb,
                          int ldc, Half t, int cus, hipStream_t stream) {
  if (N % 4 != 0 || ldc % 4 != 0) {
    return hipErrorInvalidValue;
  }
  const GemmHalfVariant v = gemmHalfR4Choose(M, N, K, cus);
  return t == Half::kBF16
             ? k::launch_r4_variant<k::BF16>(v, A, Bt, M, N, K, lda, ldb, k::StoreReluHalf<k::BF16>{C, ldc, M, N}, stream)
             : k::launch_r4_variant<k::F16>(v, A, Bt, M, N, K, lda, ldb, k::StoreReluHalf<k::F16>{C, ldc, M, N}, stream);
}

hipError_t gemmHalfR4Qkv(const uint16_t* tokens, const uint16_t* Wqkv_t, uint16_t* q, uint16_t* k_, uint16_t* vt, int B,
                         int T_, int E, int H, int S_pad, Half t, int cus, hipStream_t stream) {
  const int M = B * T_;
  const int Dh = E / H;
  if (E % H != 0 || Dh % 4 != 0) {
    return hipErrorInvalidValue;
  }
  const GemmHalfVariant v = gemmHalfR4Choose(M, 3 * E, E, cus);
  return t == Half::kBF16 ? k::launch_r4_variant<k::BF16>(v, tokens, Wqkv_t, M, 3 * E, E, E, E,
                                                          k::StoreQkv<k::BF16>{q, k_, vt, M, T_, E, H, Dh, S_pad}, stream)
                          : k::launch_r4_variant<k::F16>(v, tokens, Wqkv_t, M, 3 * E, E, E, E,
                                                         k::StoreQkv<k::F16>{q, k_, vt, M, T_, E, H, Dh, S_pad}, stream);
}

}  // namespace lchip::kern
