// gemm_f32.hip -- fp32 GEMM on the bf16 matrix cores, every fp32 operand as
// an exact sum of three bf16 values.
//
// An fp32 value x has 24 significant bits and a bf16 value 8, so
//   h = bf16(x), m = bf16(x - h), l = bf16(x - h - m)   (round to nearest)
// hold x exactly: x = h + m + l.  The product of two such sums needs six of
// the nine bf16 products (hh, hm, mh, mm, hl, lh): the dropped three together
// stay below 2^-24 of |a b|, half an fp32 ulp of each term (0.87 of that at most
// over 4 million pairs, 0.09 on average, as often up as down).
//
// The split is exact for finite values whose low parts stay normal bf16
// numbers; SplitGuardF32 says which operands are not (an infinity, a NaN, a
// value outside [2^-100, 2^50]): such a launch runs the same tiles on
// v_mfma_f32_16x16x4_f32 with the fp32 operands.
#include <type_traits>

#include "../kernels.hpp"
#include "gemm_tiles.hpp"
#include "kcommon.hpp"

namespace lchip::k {

using kern::SplitGuardF32;
using kern::SplitOperandF32;

// ---------------------------------------------------------------------------
// The planes of an operand: [h, m, l][band of 16 rows][32-deep k step][lane]
// with 16 bytes a lane: row l % 16 of the band, k = 8 (l / 16) .. + 7 of the
// step, the fragment of v_mfma_f32_16x16x32_bf16.  A wave's fragment load is
// then 1 KB of contiguous memory.  Rows are A's rows (ROWS_K: k contiguous in
// the source) or B's columns.
// ---------------------------------------------------------------------------
template <bool ROWS_K>
__device__ __forceinline__ void split_block(const float* __restrict__ src, int ld, uint16_t* __restrict__ dst,
                                            size_t plane, int band, int step, int nk, int lane) {
  const int row = band * 16 + (lane & 15);
  const int k = step * 32 + 8 * (lane >> 4);
  float v[8];
  if constexpr (ROWS_K) {
    const floatx4* p = reinterpret_cast<const floatx4*>(src + static_cast<size_t>(row) * ld + k);
    const floatx4 lo = p[0];
    const floatx4 hi = p[1];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = lo[j];
      v[4 + j] = hi[j];
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[j] = src[static_cast<size_t>(k + j) * ld + row];
    }
  }
  uint16_t* out = dst + ((static_cast<size_t>(band) * nk + step) * 64 + lane) * 8;
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    u32x4 w;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      w[j] = pack2<BF16>(v[2 * j], v[2 * j + 1]);
      v[2 * j] -= __builtin_bit_cast(float, w[j] << 16);
      v[2 * j + 1] -= __builtin_bit_cast(float, w[j] & 0xffff0000u);
    }
    *reinterpret_cast<u32x4*>(out + p * plane) = w;
  }
}

// Both operands (whose pointer is not null) in one launch, a wave per block.
__global__ __launch_bounds__(256) void split_planes_kernel(SplitOperandF32 a, SplitOperandF32 b, int nk) {
  const int lane = threadIdx.x & 63;
  const long long na = a.src != nullptr ? static_cast<long long>(a.bands) * nk : 0;
  const long long total = na + (b.src != nullptr ? static_cast<long long>(b.bands) * nk : 0);
  for (long long i = static_cast<long long>(blockIdx.x) * 4 + (threadIdx.x >> 6); i < total; i += gridDim.x * 4ll) {
    // consecutive blocks: k steps of one band of A (its rows are contiguous
    // along k), bands of one k step of B
    if (i < na) {
      split_block<true>(a.src, a.ld, a.planes, static_cast<size_t>(a.bands) * nk * 512, static_cast<int>(i / nk),
                        static_cast<int>(i % nk), nk, lane);
    } else {
      const long long j = i - na;
      split_block<false>(b.src, b.ld, b.planes, static_cast<size_t>(b.bands) * nk * 512,
                         static_cast<int>(j % b.bands), static_cast<int>(j / b.bands), nk, lane);
    }
  }
}

// Buffer loads: a wave-uniform base, a 32-bit lane offset that never changes,
// a uniform offset that moves with the k step (SALU).
__device__ __forceinline__ u32x4 load16(__amdgpu_buffer_rsrc_t rsrc, uint32_t lane_off, int uniform_off) {
  return __builtin_bit_cast(
      u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, static_cast<int>(lane_off), uniform_off, 0));
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_at(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0x7fffffff, 0x00027000);
}

// The step of wave-uniform index t of a 16 R x 64 block on the fp32 matrix
// instruction, for operands the planes cannot hold.
template <int R>
__device__ __forceinline__ void f32_step(const SplitOperandF32& A, const SplitOperandF32& B, int step, int row0,
                                         int col0, int lane, floatx4 (&acc)[R][4]) {
  const int lr = lane & 15;
  const int k = step * 32 + 8 * (lane >> 4);
  float bv[4][8];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int col = min(col0 + 16 * j, (B.bands - 1) * 16) + lr;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      bv[j][e] = B.src[static_cast<size_t>(k + e) * B.ld + col];
    }
  }
#pragma unroll
  for (int b = 0; b < R; ++b) {
    const int row = min(row0 + 16 * b, (A.bands - 1) * 16) + lr;
    const floatx4* p = reinterpret_cast<const floatx4*>(A.src + static_cast<size_t>(row) * A.ld + k);
    const floatx4 lo = p[0];
    const floatx4 hi = p[1];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        acc[b][j] =
            __builtin_amdgcn_mfma_f32_16x16x4f32(bv[j][e], e < 4 ? lo[e & 3] : hi[e & 3], acc[b][j], 0, 0, 0);
      }
    }
  }
}

// Accumulators start as zeros the compiler cannot see through: known zeros
// make it keep the loop's accumulators in vector registers and copy them to
// and from the accumulation registers in every iteration (64x64 tile: 192
// moves per 192 MFMAs).
template <int R>
__device__ __forceinline__ void zero_acc(floatx4 (&acc)[R][4]) {
#pragma unroll
  for (int b = 0; b < R; ++b) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc[b][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
      asm volatile("" : "+a"(acc[b][j]));
    }
  }
}
template <int R>
__device__ __forceinline__ void add_acc(floatx4 (&acc)[R][4], floatx4 (&low)[R][4]) {
#pragma unroll
  for (int b = 0; b < R; ++b) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      asm volatile("" : "+a"(acc[b][j]), "+a"(low[b][j]));
      acc[b][j] += low[b][j];
    }
  }
}

// The six products (plane of A, plane of B; 0 = h), the small ones first.
constexpr int kProdA[6] = {2, 0, 1, 1, 0, 0};
constexpr int kProdB[6] = {0, 2, 1, 0, 1, 0};

// One 16 RB x 64 tile a workgroup, four waves along k (each multiplies the
// whole tile over every fourth k step); gridDim.y workgroups share a tile's k
// range.  No LDS in the loop: no fragment is used by two waves, and a block of
// the planes is one contiguous 1 KB load straight into registers, a step
// ahead of its MFMAs.
// Bound: the loads.  A 64x64 tile needs 24 KB per wave and 96 MFMAs (1536
// cycles), 64 bytes a cycle and CU at the matrix rate; measured about 41
// (loading two steps ahead instead of one changed nothing), so a k step takes
// 1.0-1.2 us where the MFMAs alone need 0.7.  Splitting the fp32 values in
// the loop instead (43 bytes a cycle, no planes) was bound by its VALU work:
// 17.5 against 16.1 us at 1024^3.
// Measured against the fp32 matrix instruction's kernels (1024^3 / 512x2048x512
// / 256^3 / 897x2841x1092): 22.2 / 19.0 / 7.9 / 60.3 -> 16.0 / 16.5 / 6.7 /
// 34.9 us; relative error against 64 bits 2.9e-7 / 2.1e-7 / 0.9e-7 / 4.0e-7 ->
// 1.0e-7 / 0.9e-7 / 0.6e-7 / 1.6e-7 (normal values).
template <int RB>
__global__ __launch_bounds__(256, 1) void gemm_f32_split_kernel(SplitOperandF32 A, SplitOperandF32 B,
                                                                float* __restrict__ C, int M, int N, int ldc,
                                                                int tiles_m, int tiles_n, int nk_all,
                                                                SplitGuardF32 guard, SplitKWork work, int vec4) {
  constexpr int WK = 4;
  constexpr int BM = 16 * RB;
  constexpr int BN = 64;
  __shared__ floatx4 red[WK * RB * 4 * 64];
  __shared__ int last;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int kq = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15;
  const int lq = lane >> 4;

  int bm, bn;
  tile_origin<8>(tiles_m, tiles_n, BM, BN, bm, bn);
  // k steps [k0, k1) of this workgroup, of which wave kq takes every fourth.
  const int k0 = static_cast<int>(static_cast<long long>(blockIdx.y) * nk_all / gridDim.y);
  const int k1 = static_cast<int>(static_cast<long long>(blockIdx.y + 1) * nk_all / gridDim.y);
  const int steps = (k1 - k0 - kq + WK - 1) / WK;  // <= 0: none

  const size_t plane_a = static_cast<size_t>(A.bands) * nk_all * 1024;  // bytes
  const size_t plane_b = static_cast<size_t>(B.bands) * nk_all * 1024;
  const char* a0 = reinterpret_cast<const char*>(A.planes) + static_cast<size_t>(bm / 16) * nk_all * 1024;
  const char* b0 = reinterpret_cast<const char*>(B.planes) + static_cast<size_t>(bn / 16) * nk_all * 1024;
  __amdgpu_buffer_rsrc_t ra[3], rb[3];
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    ra[p] = buffer_at(a0 + p * plane_a);
    rb[p] = buffer_at(b0 + p * plane_b);
  }
  const uint32_t voff = lane * 16u;
  int a_band[RB];  // bytes from the tile's first band; past the last band: that band again (never stored)
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    a_band[b] = min(b, A.bands - 1 - bm / 16) * nk_all * 1024;
  }
  const int b_band = nk_all * 1024;
  constexpr int NF = (RB + 4) * 3;
  // fragment f of step t: A block f / 3, plane f % 3 for f < 3 RB, then B;
  // steps past the last re-load the operand's last one (unused)
  auto load = [&](int f, int t) {
    const int at = min(k0 + kq + t * WK, nk_all - 1) * 1024;
    if (f < 3 * RB) {
      return load16(ra[f % 3], voff, a_band[f / 3] + at);
    }
    return load16(rb[f % 3], voff, (f / 3 - RB) * b_band + at);
  };
  u32x4 fr[2][NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    fr[0][f] = load(f, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
  floatx4 acc[RB][4];
  zero_acc(acc);
  if (guard.unsafe()) {
    for (int t = 0; t < steps; ++t) {
      f32_step(A, B, k0 + kq + t * WK, bm, bn, lane, acc);
    }
  } else {
    floatx4 low[RB][4];
    zero_acc(low);
    // The hh products go to `acc`, the five small ones to `low`: `acc` is
    // rounded once per k step instead of six times.
    auto body = [&](auto phase, int t) {
      constexpr int P = decltype(phase)::value;  // t % 2
#pragma unroll
      for (int g = 0; g < 24 * RB; ++g) {
        const int q = g / (4 * RB);
        const int b = g / 4 % RB;
        const int j = g % 4;
        floatx4& d = q < 5 ? low[b][j] : acc[b][j];
        // B is the MFMAs' first operand: a lane holds four columns of one row
        d = mfma16x16x32<BF16>(fr[P][3 * RB + 3 * j + kProdB[q]], fr[P][3 * b + kProdA[q]], d);
        __builtin_amdgcn_sched_barrier(0);
        if (g % 2 == 0 && g / 2 < NF) {
          fr[P ^ 1][g / 2] = load(g / 2, t + 1);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    for (int t = 0; t < steps; t += 2) {
      body(std::integral_constant<int, 0>{}, t);
      if (t + 1 < steps) {
        body(std::integral_constant<int, 1>{}, t + 1);
      }
    }
    add_acc(acc, low);
  }

  // acc[b][j]: row bm + 16 b + lane % 16, columns bn + 16 j + 4 (lane / 16) .. + 3.
  // The four waves' parts of a row block meet in LDS; wave w sums (in wave
  // order) and stores blocks w and w + 4.
  constexpr int MINE = (RB + 3) / 4;
  auto slot = [&](int k, int b, int j) { return ((k * RB + b) * 4 + j) * 64 + lane; };
#pragma unroll
  for (int b = 0; b < RB; ++b) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      red[slot(kq, b, j)] = acc[b][j];
    }
  }
  __syncthreads();
  floatx4 mine[MINE][4];
#pragma unroll
  for (int s = 0; s < MINE; ++s) {
    const int b = min(kq + 4 * s, RB - 1);  // a wave without a second block sums (and never stores) the last one
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      mine[s][j] = red[slot(0, b, j)];
#pragma unroll
      for (int k = 1; k < WK; ++k) {
        mine[s][j] += red[slot(k, b, j)];
      }
    }
  }
  if (gridDim.y > 1 && !sum_splits(work, lane, kq, &last, mine)) {
    return;
  }
#pragma unroll
  for (int s = 0; s < MINE; ++s) {
    if (kq + 4 * s < RB) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        store_c4(C, ldc, bm + 16 * (kq + 4 * s) + lr, bn + 16 * j + 4 * lq, M, N, vec4, mine[s][j]);
      }
    }
  }
}

// One 128 x 128 tile a workgroup, four waves of 64 x 64; the planes of a
// 32-deep k step of both operands (48 KB) pass through a ring of three LDS
// slots.  gridDim.y workgroups share a tile's k range.
// A fragment serves two waves and six products serve each plane three or two
// times, so a CU reads 32 bytes a cycle from the caches and 64 from LDS at the
// matrix rate.  A step's fragments are read into registers during the step
// before it, so its slot is refilled as soon as everyone has passed the one
// barrier of the step, two steps before the copies are needed.  A workgroup
// fills a CU (144 KB of LDS).
// Bound: the matrix cores at the clock they reach under load (a step 1.06 us,
// 60% of the nominal rate), plus about 4 us of prologue and C stores a tile.
// Measured against the fp32 matrix instruction's kernel, 4096x1024x4096 /
// 2048^3 / 3072^3: 270 / 134 / 440 -> 152 / 75 / 274 us; relative error
// against 64 bits 2.9e-7 / 4.1e-7 / 5.0e-7 -> 1.9e-7 / 2.7e-7 / 3.4e-7.
__global__ __launch_bounds__(256, 1) void gemm_f32_split128_kernel(SplitOperandF32 A, SplitOperandF32 B,
                                                                   float* __restrict__ C, int M, int N, int ldc,
                                                                   int tiles_m, int tiles_n, int nk_all,
                                                                   SplitGuardF32 guard, SplitKWork work, int vec4) {
  constexpr int SLOT = 48 * 1024;  // bytes: A bands 0-7 (3 planes each), then B's
  __shared__ __attribute__((aligned(16))) char smem[3 * SLOT];
  __shared__ int last;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave >> 1) * 4;  // first band of this wave's rows and columns
  const int wn = (wave & 1) * 4;
  const int lr = lane & 15;
  const int lq = lane >> 4;
  int bm, bn;
  tile_origin<4>(tiles_m, tiles_n, 128, 128, bm, bn);
  const int k0 = static_cast<int>(static_cast<long long>(blockIdx.y) * nk_all / gridDim.y);
  const int k1 = static_cast<int>(static_cast<long long>(blockIdx.y + 1) * nk_all / gridDim.y);
  const int steps = k1 - k0;

  // Copy c (0..11) of this wave fills 1 KB block 12 * wave + c of a slot:
  // block i = (band i / 3 of A, then of B; plane i % 3).  Bands past the
  // operand's last are read as that one (never stored).
  const size_t plane_a = static_cast<size_t>(A.bands) * nk_all * 1024;  // bytes
  const size_t plane_b = static_cast<size_t>(B.bands) * nk_all * 1024;
  const char* src[4];  // plane 0 of this wave's four bands, at step k0
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int band = 4 * wave + i;
    const int at = wave < 2 ? min(bm / 16 + band, A.bands - 1) : min(bn / 16 + band - 8, B.bands - 1);
    src[i] = reinterpret_cast<const char*>(wave < 2 ? A.planes : B.planes) +
             (static_cast<size_t>(at) * nk_all + k0) * 1024;
  }
  const size_t plane = wave < 2 ? plane_a : plane_b;
  const uint32_t voff = lane * 16u;
  const uint32_t wave_lds = lds_addr(smem) + static_cast<uint32_t>(wave) * 12288u;
  auto copy = [&](int c, int t, int slot) {
    const int st = min(t, steps - 1);
    load_lds16_sbase(voff, src[c / 3] + (c % 3) * plane + static_cast<size_t>(st) * 1024,
                     wave_lds + static_cast<uint32_t>(slot * SLOT + c * 1024));
  };
  floatx4 acc[4][4];
  zero_acc(acc);
  if (guard.unsafe()) {
    // four chains along k, as the fp32 kernels and the smaller tiles have
    for (int c = 0; c < 4; ++c) {
      floatx4 part[4][4];
      zero_acc(part);
      for (int t = c * steps / 4; t < (c + 1) * steps / 4; ++t) {
        f32_step(A, B, k0 + t, bm + 16 * wm, bn + 16 * wn, lane, part);
      }
      add_acc(acc, part);
    }
  } else if (steps > 0) {
    floatx4 low[4][4];
    zero_acc(low);
#pragma unroll
    for (int t = 0; t < 3; ++t) {
#pragma unroll
      for (int c = 0; c < 12; ++c) {
        copy(c, t, t);
      }
    }
    typedef __attribute__((address_space(3))) const char lds_char;
    typedef __attribute__((address_space(3))) const u32x4 lds_u32x4;
    lds_char* la = (lds_char*)(smem) + (wm * 3) * 1024 + lane * 16;
    lds_char* lb = (lds_char*)(smem) + (24 + wn * 3) * 1024 + lane * 16;
    // fragment f (0..11: A band f / 3, plane f % 3; 12..23: B) of `slot`
    auto frag = [&](int slot, int f) -> u32x4 {
      return *reinterpret_cast<lds_u32x4*>((f < 12 ? la + f * 1024 : lb + (f - 12) * 1024) + slot * SLOT);
    };
    __builtin_amdgcn_s_waitcnt(0xc07f);
    wait_vmcnt<24>();
    stage_barrier();
    u32x4 fr[2][24];
#pragma unroll
    for (int f = 0; f < 24; ++f) {
      fr[0][f] = frag(0, f);
    }
    // Step t: its fragments are in fr[P]; slot (t + 1) % 3 is read into
    // fr[P ^ 1], and slot t % 3, which everyone has read, is refilled with
    // step t + 3.
    auto body = [&](auto phase, int t) {
      constexpr int PH = decltype(phase)::value;  // t % 6
      constexpr int P = PH % 2;
      constexpr int SL = PH % 3;
      wait_vmcnt<12>();    // this wave's copies of step t + 1 have landed
      wait_lgkmcnt<0>();   // and its reads of step t are done
      stage_barrier();
#pragma unroll
      for (int g = 0; g < 96; ++g) {
        const int q = g / 16;
        const int b = g / 4 % 4;
        const int j = g % 4;
        floatx4& d = q < 5 ? low[b][j] : acc[b][j];
        d = mfma16x16x32<BF16>(fr[P][12 + 3 * j + kProdB[q]], fr[P][3 * b + kProdA[q]], d);
        __builtin_amdgcn_sched_barrier(0);
        if (g % 3 == 0 && g < 72) {
          fr[P ^ 1][g / 3] = frag((SL + 1) % 3, g / 3);
        }
        if (g % 8 == 4) {
          copy(g / 8, t + 3, SL);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    for (int t = 0; t < steps; t += 6) {
      body(std::integral_constant<int, 0>{}, t);
      if (t + 1 < steps) body(std::integral_constant<int, 1>{}, t + 1);
      if (t + 2 < steps) body(std::integral_constant<int, 2>{}, t + 2);
      if (t + 3 < steps) body(std::integral_constant<int, 3>{}, t + 3);
      if (t + 4 < steps) body(std::integral_constant<int, 4>{}, t + 4);
      if (t + 5 < steps) body(std::integral_constant<int, 5>{}, t + 5);
    }
    wait_vmcnt<0>();  // no copy may still be writing LDS
    add_acc(acc, low);
  }
  // acc[b][j]: row bm + 16 (wm + b) + lane % 16, columns bn + 16 (wn + j) + 4 (lane / 16) .. + 3
  if (gridDim.y > 1 && !sum_splits(work, lane, wave, &last, acc)) {
    return;
  }
#pragma unroll
  for (int b = 0; b < 4; ++b) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      store_c4(C, ldc, bm + 16 * (wm + b) + lr, bn + 16 * (wn + j) + 4 * lq, M, N, vec4, acc[b][j]);
    }
  }
}

template <int RB>
static hipError_t launch_split(const SplitOperandF32& A, const SplitOperandF32& B, float* C, int M, int N, int K,
                               int ldc, const SplitGuardF32& guard, const SplitKWork& work, int splits,
                               hipStream_t stream) {
  const int tiles_m = (M + 16 * RB - 1) / (16 * RB);
  const int tiles_n = (N + 63) / 64;
  const int vec4 = (ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0) ? 1 : 0;
  hipLaunchKernelGGL((gemm_f32_split_kernel<RB>), dim3(tiles_m * tiles_n, splits), dim3(256), 0, stream, A, B, C, M,
                     N, ldc, tiles_m, tiles_n, K / 32, guard, work, vec4);
  return hipGetLastError();
}

}  // namespace lchip::k

namespace lchip::kern {

using namespace lchip::k;

hipError_t splitPlanesF32(const SplitOperandF32& a, const SplitOperandF32& b, int K, hipStream_t stream) {
  const int nk = K / 32;
  const long long total =
      ((a.src != nullptr ? static_cast<long long>(a.bands) : 0) + (b.src != nullptr ? b.bands : 0)) * nk;
  if (total == 0) {
    return hipSuccess;
  }
  const long long blocks = (total + 3) / 4;
  hipLaunchKernelGGL(split_planes_kernel, dim3(static_cast<unsigned>(blocks < 8192 ? blocks : 8192)), dim3(256), 0,
                     stream, a, b, nk);
  return hipGetLastError();
}

int gemmF32SplitTiles(GemmF32Variant variant, int M, int N) {
  const int rows = variant == GemmF32Variant::kSplit64 ? 64 : variant == GemmF32Variant::kSplit80 ? 80 : 128;
  const int cols = variant == GemmF32Variant::kSplit128 ? 128 : 64;
  return ((M + rows - 1) / rows) * ((N + cols - 1) / cols);
}

int gemmF32SplitCount(GemmF32Variant variant, int M, int N, int K, int cus) {
  // Sharing a tile's k range costs its partial sums a round trip (about 2.5
  // us) and pays only where CUs are idle: each workgroup keeps at least
  // eight k steps.  512x2048x512 (64 tiles):
  // 21.5 us whole, 16.8 halved, 16.4 quartered; 1024^3 (256 tiles): 16.1 us
  // whole, 22.1 halved; with 128x128 tiles (64) 30.5, 23.4 and 21.8 us.
  const int tiles = gemmF32SplitTiles(variant, M, N);
  constexpr int least = 8;  // k steps of a workgroup
  int splits = 1;
  while (splits < 8 && tiles * splits * 2 <= cus && K / 32 >= least * splits * 2) {
    splits *= 2;
  }
  return splits;
}

GemmF32Variant gemmF32SplitChoose(int M, int N, int K, int cus) {
  // A model of the measured times (us): a launch of one round, then per round
  // of workgroups its k steps.  The 128x128 tile runs a step at 1.06 us and
  // has the longer prologue; the smaller ones read more than twice the bytes
  // per product and are bound by their loads (64 rows 1.2 us per four k
  // steps, 80 rows 1.35).  Measured (64 / 80 / 128): 1024^3 16.1 / 17.3 /
  // 21.8 us; 1000x777x1030 23.6 / 16.2 / 24.5; 2048^3 86 / 95 / 73;
  // 4096x1024x4096 192 / 185 / 153.
  const GemmF32Variant all[3] = {GemmF32Variant::kSplit64, GemmF32Variant::kSplit80, GemmF32Variant::kSplit128};
  const double step[3] = {0.30, 0.34, 1.06};
  const double round[3] = {2.5, 2.7, 4.0};
  GemmF32Variant best = all[0];
  double best_us = 0.0;
  for (int i = 0; i < 3; ++i) {
    const int splits = gemmF32SplitCount(all[i], M, N, K, cus);
    const long long groups = static_cast<long long>(gemmF32SplitTiles(all[i], M, N)) * splits;
    const double us = static_cast<double>((groups + cus - 1) / cus) * (round[i] + step[i] * (K / 32) / splits) +
                      (splits > 1 ? 2.5 : 0.0);
    if (i == 0 || us < best_us) {
      best = all[i];
      best_us = us;
    }
  }
  return best;
}

size_t gemmF32SplitPartFloats(GemmF32Variant variant) {
  return variant == GemmF32Variant::kSplit64 ? 4096 : variant == GemmF32Variant::kSplit80 ? 8192 : 16384;
}

hipError_t gemmF32Split(const SplitOperandF32& A, const SplitOperandF32& B, float* C, int M, int N, int K, int ldc,
                        const SplitGuardF32& guard, const SplitKWork& work, GemmF32Variant variant, int splits,
                        hipStream_t stream) {
  if (K <= 0 || K % kF32GemmBK != 0 || M <= 0 || N <= 0 || splits < 1) {
    return hipErrorInvalidValue;
  }
  switch (variant) {
    case GemmF32Variant::kSplit64:
      return launch_split<4>(A, B, C, M, N, K, ldc, guard, work, splits, stream);
    case GemmF32Variant::kSplit80:
      return launch_split<5>(A, B, C, M, N, K, ldc, guard, work, splits, stream);
    case GemmF32Variant::kSplit128: {
      const int tiles_m = (M + 127) / 128;
      const int tiles_n = (N + 127) / 128;
      const int vec4 = (ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0) ? 1 : 0;
      hipLaunchKernelGGL(gemm_f32_split128_kernel, dim3(tiles_m * tiles_n, splits), dim3(256), 0, stream, A, B, C, M,
                         N, ldc, tiles_m, tiles_n, K / 32, guard, work, vec4);
      return hipGetLastError();
    }
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace lchip::kern
