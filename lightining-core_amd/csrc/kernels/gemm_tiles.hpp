// gemm_tiles.hpp -- tile order, the sum over workgroups that share a tile's k
// range, and masked C stores of the GEMM kernels that take k splits.
#pragma once

#include "../kernels.hpp"
#include "kcommon.hpp"

namespace lchip::k {

using kern::SplitKWork;

// Tile of workgroup w: w runs on XCD w % 8, and each XCD gets a contiguous
// range of an order that walks groups of GROUP tile rows.
template <int GROUP>
__device__ __forceinline__ void tile_origin(int tiles_m, int tiles_n, int tile_h, int tile_w, int& bm, int& bn) {
  const int full = (tiles_m * tiles_n) & ~7;
  int pid = blockIdx.x;
  if (pid < full) {
    pid = (pid & 7) * (full >> 3) + (pid >> 3);
  }
  const int group_size = GROUP * tiles_n;
  const int group = pid / group_size;
  const int first_m = group * GROUP;
  const int gm = min(tiles_m - first_m, GROUP);
  const int in_group = pid - group * group_size;
  bm = (first_m + in_group % gm) * tile_h;
  bn = (in_group / gm) * tile_w;
}

// C[m][n .. n + 3] = v, masked to [M, N].
__device__ __forceinline__ void store_c4(float* C, int ldc, int m, int n, int M, int N, int vec4, floatx4 v) {
  if (m >= M) {
    return;
  }
  float* p = C + static_cast<size_t>(m) * ldc + n;
  if (vec4 && n + 3 < N) {
    *reinterpret_cast<floatx4*>(p) = v;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (n + i < N) {
        p[i] = v[i];
      }
    }
  }
}

// The sum of acc over the gridDim.y workgroups of a tile, in k order, in the
// workgroup that finishes last (false in the others); every wave sums its own
// R x J blocks of 16 x 16.  Partials move with device-scope (sc1) stores and loads,
// coherent across the XCDs' L2s; the vmcnt wait orders the stores before the
// counter bump.  No workgroup waits for another, and the last one leaves the
// tile's counter at zero.
template <int R, int J>
__device__ __forceinline__ bool sum_splits(const SplitKWork& work, int lane, int wave, int* last,
                                           floatx4 (&acc)[R][J]) {
  const size_t tile = blockIdx.x;
  const int splits = gridDim.y;
  auto part = [&](int y, int b, int j) {
    return work.part + (((tile * splits + y) * 4 + wave) * R + b) * (J * 256) + j * 256 + lane;
  };
#pragma unroll
  for (int b = 0; b < R; ++b) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        __hip_atomic_store(part(blockIdx.y, b, j) + i * 64, acc[b][j][i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  wait_vmcnt<0>();
  __syncthreads();
  if (threadIdx.x == 0) {
    *last = __hip_atomic_fetch_add(work.counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == splits - 1;
  }
  __syncthreads();
  if (*last == 0) {
    return false;
  }
#pragma unroll
  for (int b = 0; b < R; ++b) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
      acc[b][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  for (int y = 0; y < splits; ++y) {
#pragma unroll
    for (int b = 0; b < R; ++b) {
#pragma unroll
      for (int j = 0; j < J; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc[b][j][i] += __hip_atomic_load(part(y, b, j) + i * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    }
  }
  if (threadIdx.x == 0) {
    __hip_atomic_store(work.counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  return true;
}

}  // namespace lchip::k
