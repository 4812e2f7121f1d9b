// attention_f32.hip -- fp32 attention forward on the bf16 matrix cores, every
// fp32 value as an exact sum of three bf16 values (see gemm_f32.hip: h, m, l
// and the six products that matter; operands the parts cannot hold run on
// v_mfma_f32_16x16x4_f32 instead).
//
// Formulation as in attention.hip: scores transposed, S^T = K . Q^T, so a lane
// holds scores of one query per 16-query block, the output transposed,
// O^T = V^T . P^T, and the probabilities go from the first product's
// accumulators into the second's operand without leaving the lane: with 16x16
// tiles lane l holds, of every 32 keys, keys 4 (l / 16) + i and 16 + 4 (l / 16)
// + i (i < 4) of query l % 16, and V's planes are laid out in that key order.
#include <math.h>

#include "../kernels.hpp"
#include "kcommon.hpp"

namespace lchip::k {

using kern::AttnPlanesF32;

namespace {
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kMaskValue = -1e30f;
constexpr int kQBlock = 128;  // queries per workgroup, 32 per wave
constexpr int kPA[6] = {2, 0, 1, 1, 0, 0};  // the six products (plane of the first operand, of the second), small first
constexpr int kPB[6] = {0, 2, 1, 0, 1, 0};
}  // namespace

// ---------------------------------------------------------------------------
// Planes.  A block is 1 KB: lane l holds 8 bf16, the fragment of
// v_mfma_f32_16x16x32_bf16.  Per head (nt = ceil(S / 32) tiles of 32 rows,
// DK = D / 32):
//   q:  [band of 16 queries (2 nt)][plane][k step DK]
//   kv: [tile of 32 keys (nt)] of 12 DK blocks: K [plane][band 2][k step DK],
//       then V^T [plane][band of 16 columns (2 DK)]
// K and Q lanes hold row l % 16, d = 32 step + 8 (l / 16) + j; V lanes column
// l % 16, keys 16 (j / 4) + 4 (l / 16) + j % 4.  Rows past S are zero.  Every
// value is checked on the way (`guard` words as padCopyF32's).
// ---------------------------------------------------------------------------
template <int DK>
__global__ __launch_bounds__(256) void attn_planes_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                          const float* __restrict__ v, uint16_t* __restrict__ pq,
                                                          uint16_t* __restrict__ pkv, int bh, int S, int nt,
                                                          int* __restrict__ guard, int* __restrict__ guard_host,
                                                          int epoch) {
  constexpr int D = 32 * DK;
  const int lane = threadIdx.x & 63;
  const int lr = lane & 15;
  const int lq = lane >> 4;
  const long long per = static_cast<long long>(nt) * 2 * DK;  // blocks of one plane of one tensor of a head
  const long long total = 3 * per * bh;
  bool odd = false;
  for (long long i = static_cast<long long>(blockIdx.x) * 4 + (threadIdx.x >> 6); i < total; i += gridDim.x * 4ll) {
    const int head = static_cast<int>(i / (3 * per));
    const long long r = i - 3 * per * head;
    const int which = static_cast<int>(r / per);  // 0 Q, 1 K, 2 V
    const int b = static_cast<int>(r - per * which);
    const size_t src = static_cast<size_t>(head) * S * D;
    float x[8];
    uint16_t* dst;
    size_t plane;
    if (which < 2) {
      const int band = b / DK;
      const int step = b - band * DK;
      const int row = band * 16 + lr;
      const float* p = (which == 0 ? q : k) + src + static_cast<size_t>(row) * D + 32 * step + 8 * lq;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        x[j] = row < S ? p[j] : 0.0f;
      }
      if (which == 0) {
        dst = pq + ((static_cast<size_t>(head) * 2 * nt + band) * 3 * DK + step) * 512;
        plane = DK * 512;
      } else {
        dst = pkv + ((static_cast<size_t>(head) * nt + band / 2) * 12 * DK + (band & 1) * DK + step) * 512;
        plane = 2 * DK * 512;
      }
    } else {
      const int tile = b / (2 * DK);
      const int band = b - tile * 2 * DK;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = tile * 32 + 16 * (j / 4) + 4 * lq + j % 4;
        x[j] = key < S ? v[src + static_cast<size_t>(key) * D + band * 16 + lr] : 0.0f;
      }
      dst = pkv + ((static_cast<size_t>(head) * nt + tile) * 12 * DK + 6 * DK + band) * 512;
      plane = 2 * DK * 512;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t mag = __builtin_bit_cast(uint32_t, x[j]) & 0x7fffffffu;
      odd |= mag != 0 && (mag < 0x0d800000u || mag > 0x58800000u);  // 2^-100, 2^50
    }
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      u32x4 w;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        w[j] = pack2<BF16>(x[2 * j], x[2 * j + 1]);
        x[2 * j] -= __builtin_bit_cast(float, w[j] << 16);
        x[2 * j + 1] -= __builtin_bit_cast(float, w[j] & 0xffff0000u);
      }
      *reinterpret_cast<u32x4*>(dst + p * plane + lane * 8) = w;
    }
  }
  if (odd) {
    *guard = epoch;
    __hip_atomic_store(guard_host, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// max over the four lanes that share a query.
__device__ __forceinline__ float max_quads(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  return max_xor32(max_of_swap(__builtin_amdgcn_permlane16_swap(u, u, false, false)));
}

// ---------------------------------------------------------------------------
// 128 queries a workgroup, 32 a wave; KG groups of four waves take alternate
// 32-key tiles, each group through a ring of three tiles in LDS (copied two
// tiles ahead, one barrier a tile).  Q's fragments stay in registers; a K or V
// fragment (1 KB, contiguous in LDS and in memory) serves one wave's 32
// queries.  The output's hh products and the five small ones have accumulators
// of their own.
// Bound: a tile is 96 MFMAs (D = 64, 1536 cycles), about 250 VALU instructions
// and the LDS latencies between them, which one wave per SIMD cannot hide
// (1.8 us a tile) and two halve; small problems pay the partials of the key
// split besides.  Two waves per SIMD need 256 registers, so they stop at D = 64.
// Measured against attn_fwd_f32_kernel (batch x heads, S, D; us): 1x8 1000 64
// causal 67 -> 24.7; 4x16 512 64 causal 77 -> 31; 4x12 2048 64 774 -> 255;
// 4x16 512 128 277 -> 70; 4x16 2048 128 causal 2133 -> 842; 2x4 300 96 causal
// 30 -> 19.  Relative error against 64 bits 2.8e-7 / 2.8e-7 / 8.7e-7 / 5.7e-7 /
// 4.6e-7 / 2.7e-7 -> 1.6e-7 / 1.5e-7 / 3.5e-7 / 3.2e-7 / 2.7e-7 / 1.9e-7.
// (Computing tile t + 1's scores while tile t's become probabilities, in one
// wave, gained nothing and spilled at D >= 64.)
// ---------------------------------------------------------------------------
template <int DK, int KG>
__global__ __launch_bounds__(256 * KG, DK <= 2 ? 2 : 1) void attn_fwd_f32_split_kernel(
    AttnPlanesF32 in, float* __restrict__ out, int S, int nt, int causal, float scale, float post_scale,
    float post_bias, int post_relu, int split_tiles, float* __restrict__ ws) {
  constexpr int D = 32 * DK;
  constexpr int DB = 2 * DK;               // 16-column bands of V
  constexpr int TILE = 12 * DK * 1024;     // bytes of a tile's planes
  constexpr int CPW = 3 * DK;              // 1 KB copies a wave makes of a tile
  __shared__ __attribute__((aligned(16))) char smem[3 * KG * TILE];

  const int lane = threadIdx.x & 63;
  const int wave8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wave8 & 3;  // its queries
  const int kg = wave8 >> 2;   // its tiles: every KG-th
  const int lr = lane & 15;
  const int lq = lane >> 4;
  const int head = blockIdx.y;
  // Heaviest (causal) blocks first.  Key split as in attn_fwd_f32_kernel:
  // workgroup z takes tiles [z, z + 1) * split_tiles and writes its
  // unnormalised O, m, l to ws.
  const bool split = split_tiles > 0;
  const int qb = static_cast<int>(gridDim.x) - 1 - static_cast<int>(blockIdx.x);
  const int q0 = qb * kQBlock + wave * 32;
  const int t0 = split ? static_cast<int>(blockIdx.z) * split_tiles : 0;
  int t1 = causal ? min(nt, (qb + 1) * (kQBlock / 32)) : nt;
  if (split) {
    t1 = min(t1, t0 + split_tiles);
  }
  const int n = (t1 - t0 + KG - 1) / KG;  // iterations; iteration t: tile t0 + t * KG + kg
  // The wave's last tile: up to its queries' diagonal.  Only that tile can need
  // masks (queries and tiles are both cut at multiples of 32), so a non-finite V
  // row reaches no query before its own tile.
  const int edge_tile = causal ? min(nt - 1, q0 / 32) : nt - 1;
  const int last_tile = min(edge_tile, t1 - 1);

  floatx4 o[2][DB], ol[2][DB];  // hh products; the small ones
  float m_run[2], l_run[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    m_run[c] = kMaskValue;
    l_run[c] = 0.0f;
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      o[c][d] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
      ol[c][d] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }

  // Scores of a tile -> probabilities in st and the new row maxima; `edge`:
  // keys past S or (causal) past the query are masked.
  const float sl = scale * kLog2e;
  auto probabilities = [&](floatx4 (&st)[2][2], float (&mt)[2], bool edge, int j0) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      mt[c] = m_run[c];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float x = st[r][c][i] * sl;
          if (edge) {
            const int key = j0 + 16 * r + 4 * lq + i;
            x = key >= S || (causal && key > q0 + 16 * c + lr) ? kMaskValue : x;
          }
          st[r][c][i] = x;
          mt[c] = fmaxf(mt[c], x);
        }
      }
      mt[c] = max_quads(mt[c]);
#pragma unroll
      for (int r = 0; r < 2; ++r) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          st[r][c][i] = __builtin_amdgcn_exp2f(st[r][c][i] - mt[c]);
        }
      }
    }
  };
  // The state moves to the new maxima (most tiles leave them alone).
  auto rescale = [&](const floatx4 (&st)[2][2], const float (&mt)[2]) {
    if (__any(mt[0] > m_run[0] || mt[1] > m_run[1])) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const float alpha = __builtin_amdgcn_exp2f(m_run[c] - mt[c]);
        m_run[c] = mt[c];
        l_run[c] *= alpha;
#pragma unroll
        for (int d = 0; d < DB; ++d) {
          o[c][d] *= alpha;
          ol[c][d] *= alpha;
        }
      }
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      l_run[c] += ((st[0][c][0] + st[0][c][1]) + (st[0][c][2] + st[0][c][3])) +
                  ((st[1][c][0] + st[1][c][1]) + (st[1][c][2] + st[1][c][3]));
    }
  };

  if (*in.guard == in.epoch) {
    // The fp32 operands, straight from memory, each tile's K and Q rows as
    // float4 (one launch: the host then knows and takes attn_fwd_f32_kernel).
    // Bound: the latency of those loads, few waves in flight.  Measured against
    // that kernel (with its combine / with the planes and the combine here, us):
    // 1x1024x128 43.6 -> 45.0, 1x600x128 39.1 -> 37.4, 8x1000x64 causal 71 -> 46,
    // 48x2048x64 865 -> 693, 64x512x128 321 -> 144, 16x1500x96 causal 324 -> 262.
    const size_t base = static_cast<size_t>(head) * S * D;
    const float* qp[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      qp[c] = in.q + base + static_cast<size_t>(min(q0 + 16 * c + lr, S - 1)) * D + 8 * lq;
    }
    for (int t = t0 + kg; t <= last_tile; t += KG) {
      const int j0 = t * 32;
      floatx4 st[2][2];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          st[r][c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        }
      }
      const float* kp[2];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        kp[r] = in.k + base + static_cast<size_t>(min(j0 + 16 * r + lr, S - 1)) * D + 8 * lq;
      }
#pragma unroll
      for (int s = 0; s < DK; ++s) {
        floatx4 kf[2][2], qf[2][2];  // rows, halves of eight values
#pragma unroll
        for (int r = 0; r < 2; ++r) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            kf[r][h] = *reinterpret_cast<const floatx4*>(kp[r] + 32 * s + 4 * h);
            qf[r][h] = *reinterpret_cast<const floatx4*>(qp[r] + 32 * s + 4 * h);
          }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
#pragma unroll
          for (int r = 0; r < 2; ++r) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
              st[r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[r][e / 4][e % 4], qf[c][e / 4][e % 4], st[r][c], 0, 0, 0);
            }
          }
        }
      }
      // V's loads of two bands go out before the probabilities are needed
      const float* vp = in.v + base + lr;
      auto band = [&](int d, float (&x)[8]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int key = j0 + 16 * (e / 4) + 4 * lq + e % 4;
          x[e] = key < S ? vp[static_cast<size_t>(key) * D + 16 * d] : 0.0f;
        }
      };
      float vx[2][8];
      band(0, vx[0]);
      band(1, vx[1]);
      float mt[2];
      probabilities(st, mt, true, j0);
      rescale(st, mt);
#pragma unroll
      for (int d = 0; d < DB; ++d) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            o[c][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vx[d % 2][e], st[e / 4][c][e % 4], o[c][d], 0, 0, 0);
          }
        }
        if (d + 2 < DB) {
          band(d + 2, vx[d % 2]);
        }
      }
    }
  } else if (n > 0) {
    const char* kv = reinterpret_cast<const char*>(in.planes_kv) + static_cast<size_t>(head) * nt * TILE +
                     wave * (CPW * 1024);
    const uint32_t ring = lds_addr(smem) + static_cast<uint32_t>(kg * 3 * TILE);
    const uint32_t lds0 = ring + static_cast<uint32_t>(wave) * (CPW * 1024u);
    const uint32_t voff = lane * 16u;
    auto copy = [&](int t, int slot) {  // tiles past the last: that one again, unused
      const char* src = kv + static_cast<size_t>(min(t0 + t * KG + kg, nt - 1)) * TILE;
#pragma unroll
      for (int c = 0; c < CPW; ++c) {
        load_lds16_sbase(voff, src + c * 1024, lds0 + static_cast<uint32_t>(slot * TILE + c * 1024));
      }
    };
    copy(0, 0);
    copy(1, 1);
    // Q's fragments stay in registers (query tiles past the last: that one, not stored)
    u32x4 qf[2][3][DK];
    {
      const int band = min(q0 / 16, 2 * nt - 2);
      const u32x4* qp = reinterpret_cast<const u32x4*>(in.planes_q) +
                        (static_cast<size_t>(head) * 2 * nt + band) * 3 * DK * 64 + lane;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
          for (int s = 0; s < DK; ++s) {
            qf[c][p][s] = qp[((c * 3 + p) * DK + s) * 64];
          }
        }
      }
    }
    typedef __attribute__((address_space(3))) const char lds_char;
    typedef __attribute__((address_space(3))) const u32x4 lds_u32x4;
    lds_char* lbase = (lds_char*)(smem) + kg * 3 * TILE + lane * 16;
    auto scores = [&](int slot, floatx4 (&st)[2][2]) {
      lds_char* tile = lbase + slot * TILE;
#pragma unroll
      for (int r = 0; r < 2; ++r) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          st[r][c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        }
      }
#pragma unroll
      for (int s = 0; s < DK; ++s) {
        u32x4 kf[2][3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
          for (int r = 0; r < 2; ++r) {
            kf[r][p] = *reinterpret_cast<lds_u32x4*>(tile + ((p * 2 + r) * DK + s) * 1024);
          }
        }
#pragma unroll
        for (int x = 0; x < 6; ++x) {
#pragma unroll
          for (int r = 0; r < 2; ++r) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
              st[r][c] = mfma16x16x32<BF16>(kf[r][kPA[x]], qf[c][kPB[x]][s], st[r][c]);
            }
          }
        }
      }
    };
    auto accumulate = [&](int slot, const floatx4 (&st)[2][2]) {
      lds_char* tile = lbase + slot * TILE + 6 * DK * 1024;
      u32x4 pf[2][3];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float x = st[j / 2][c][2 * (j & 1)];
          float y = st[j / 2][c][2 * (j & 1) + 1];
#pragma unroll
          for (int p = 0; p < 3; ++p) {
            // opaque: from the plain conversion the compiler makes a second
            // one for the value it subtracts
            uint32_t w = pack2<BF16>(x, y);
            asm("" : "+v"(w));
            pf[c][p][j] = w;
            x -= __builtin_bit_cast(float, w << 16);
            y -= __builtin_bit_cast(float, w & 0xffff0000u);
          }
        }
      }
#pragma unroll
      for (int d = 0; d < DB; d += 2) {  // two bands: four independent accumulators in turn
        u32x4 vf[2][3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            vf[e][p] = *reinterpret_cast<lds_u32x4*>(tile + (p * DB + d + e) * 1024);
          }
        }
#pragma unroll
        for (int x = 0; x < 6; ++x) {
#pragma unroll
          for (int e = 0; e < 2; ++e) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
              floatx4& acc = x < 5 ? ol[c][d + e] : o[c][d + e];
              acc = mfma16x16x32<BF16>(vf[e][kPA[x]], pf[c][kPB[x]], acc);
            }
          }
        }
      }
    };
    int slot = 0;
    for (int t = 0; t < n; ++t) {
      wait_vmcnt<CPW>();  // this wave's copies of iteration t have landed
      stage_barrier();    // everyone's; and everyone has read iteration t - 1, whose slot is refilled
      copy(t + 2, slot == 0 ? 2 : slot - 1);
      const int tile = t0 + t * KG + kg;
      if (tile <= last_tile) {
        floatx4 st[2][2];
        float mt[2];
        scores(slot, st);
        if (tile == edge_tile) {
          probabilities(st, mt, true, tile * 32);
        } else {
          probabilities(st, mt, false, 0);
        }
        rescale(st, mt);
        accumulate(slot, st);
      }
      slot = slot == 2 ? 0 : slot + 1;
    }
    wait_vmcnt<0>();  // no copy may still be writing LDS
  }

  // The wave's sums: o + ol, l over the four lanes of a query.
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    l_run[c] += __shfl_xor(l_run[c], 16);
    l_run[c] += __shfl_xor(l_run[c], 32);
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      o[c][d] += ol[c][d];
    }
  }
  if constexpr (KG == 2) {
    // The two key groups' states meet in LDS (every copy has landed).
    floatx4* os = reinterpret_cast<floatx4*>(smem) + wave * (2 * DB * 64) + lane;
    float* mls = reinterpret_cast<float*>(smem + 4 * 2 * DB * 1024) + wave * 64 * 4 + lane;
    __syncthreads();
    if (kg == 1) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        mls[128 * c] = m_run[c];
        mls[128 * c + 64] = l_run[c];
#pragma unroll
        for (int d = 0; d < DB; ++d) {
          os[(c * DB + d) * 64] = o[c][d];
        }
      }
    }
    __syncthreads();
    if (kg == 1) {
      return;
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const float m1 = mls[128 * c];
      const float m = fmaxf(m_run[c], m1);
      const float f0 = __builtin_amdgcn_exp2f(m_run[c] - m);
      const float f1 = __builtin_amdgcn_exp2f(m1 - m);
      m_run[c] = m;
      l_run[c] = l_run[c] * f0 + mls[128 * c + 64] * f1;
#pragma unroll
      for (int d = 0; d < DB; ++d) {
        o[c][d] = o[c][d] * f0 + os[(c * DB + d) * 64] * f1;
      }
    }
  }
  float* dst = out + static_cast<size_t>(head) * S * D;
  float* ml = nullptr;
  if (split) {
    const size_t heads = gridDim.y;
    dst = ws + (static_cast<size_t>(blockIdx.z) * heads + head) * S * D;
    ml = ws + static_cast<size_t>(gridDim.z) * heads * S * D +
         (static_cast<size_t>(blockIdx.z) * heads + head) * S * 2;
  }
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int qi = q0 + 16 * c + lr;
    if (qi >= S) {
      continue;
    }
    if (split && lq == 0) {
      ml[qi * 2] = m_run[c];
      ml[qi * 2 + 1] = l_run[c];
    }
    const float inv = split ? 1.0f : 1.0f / l_run[c];
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      floatx4 x = o[c][d];
      if (!split) {
        x *= inv;
        if (post_scale != 1.0f || post_bias != 0.0f || post_relu) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            x[i] = x[i] * post_scale + post_bias;
            if (post_relu && x[i] < 0.0f) {
              x[i] = 0.0f;
            }
          }
        }
      }
      *reinterpret_cast<floatx4*>(dst + static_cast<size_t>(qi) * D + 16 * d + 4 * lq) = x;
    }
  }
}

}  // namespace lchip::k

namespace lchip::kern {

using namespace lchip::k;

bool attentionF32SplitFits(int S, int D) { return D % 32 == 0 && D <= 128 && S >= 1; }

size_t attentionF32PlanesHalves(int bh, int S, int D) {
  const size_t nt = (S + 31) / 32;
  return static_cast<size_t>(bh) * nt * 32 * D * 9;  // three planes of q, k and v
}

hipError_t attentionF32Planes(const float* q, const float* k, const float* v, uint16_t* planes, int bh, int S, int D,
                              int* guard, int* guard_host, int epoch, hipStream_t stream) {
  if (!attentionF32SplitFits(S, D) || bh <= 0) {
    return hipErrorInvalidValue;
  }
  const int nt = (S + 31) / 32;
  uint16_t* pkv = planes + static_cast<size_t>(bh) * nt * 32 * D * 3;
  const long long blocks = (static_cast<long long>(bh) * nt * 2 * (D / 32) * 3 + 3) / 4;
  const dim3 grid(static_cast<unsigned>(blocks < 8192 ? blocks : 8192));
  switch (D / 32) {
    case 1:
      hipLaunchKernelGGL((attn_planes_kernel<1>), grid, dim3(256), 0, stream, q, k, v, planes, pkv, bh, S, nt, guard,
                         guard_host, epoch);
      break;
    case 2:
      hipLaunchKernelGGL((attn_planes_kernel<2>), grid, dim3(256), 0, stream, q, k, v, planes, pkv, bh, S, nt, guard,
                         guard_host, epoch);
      break;
    case 3:
      hipLaunchKernelGGL((attn_planes_kernel<3>), grid, dim3(256), 0, stream, q, k, v, planes, pkv, bh, S, nt, guard,
                         guard_host, epoch);
      break;
    default:
      hipLaunchKernelGGL((attn_planes_kernel<4>), grid, dim3(256), 0, stream, q, k, v, planes, pkv, bh, S, nt, guard,
                         guard_host, epoch);
      break;
  }
  return hipGetLastError();
}

namespace {

// Key groups within a workgroup (waves of one SIMD on alternate tiles) and
// tiles per key split (0: none) of a problem.
struct SplitPlan {
  int groups;
  int tiles;
};
SplitPlan planOf(int bh, int S, int D, int cus) {
  const int nt = (S + 31) / 32;
  const long long base = static_cast<long long>((S + kQBlock - 1) / kQBlock) * bh;
  // Two key groups while one workgroup of four waves would leave each SIMD a
  // single wave (8 heads of S = 1000, D = 64: 26.2 -> 24.7 us, 64 heads of 512:
  // 34.5 -> 31.3); their two rings fit LDS up to D = 64.
  const int groups = D <= 64 && base <= cus && nt >= 4 ? 2 : 1;
  // Key splits while CUs are idle and a wave keeps two tiles; each adds
  // partials that the combine kernel reads (8 heads of S = 1000: 1, 2, 4
  // splits 43, 31, 24.7 us; one head of 2048: 4, 8, 16 splits 28, 23, 28 us).
  int z = 1;
  while (z < 8 && base * z * 2 <= cus && nt / (2 * z * groups) >= 2) {
    z *= 2;
  }
  return SplitPlan{groups, z > 1 ? (nt + z - 1) / z : 0};
}

}  // namespace

size_t attentionF32SplitWorkFloats(int bh, int S, int D, int cus) {
  const int tiles = planOf(bh, S, D, cus).tiles;
  if (tiles == 0) {
    return 0;
  }
  const size_t z = ((S + 31) / 32 + tiles - 1) / tiles;
  return z * bh * static_cast<size_t>(S) * (D + 2);
}

hipError_t attentionF32Split(const AttnPlanesF32& in, float* out, int bh, int S, int D, bool causal, float post_scale,
                             float post_bias, int post_relu, float* ws, size_t ws_floats, int cus,
                             hipStream_t stream) {
  if (!attentionF32SplitFits(S, D) || bh <= 0 || bh > 65535) {
    return hipErrorInvalidValue;
  }
  const int nt = (S + 31) / 32;
  const SplitPlan plan = planOf(bh, S, D, cus);
  int tiles = plan.tiles;
  if (ws == nullptr || ws_floats < attentionF32SplitWorkFloats(bh, S, D, cus)) {
    tiles = 0;
  }
  const int z = tiles > 0 ? (nt + tiles - 1) / tiles : 1;
  const dim3 grid((S + kQBlock - 1) / kQBlock, bh, z);
  const float scale = 1.0f / sqrtf(static_cast<float>(D));
  const int cz = causal ? 1 : 0;
#define LC_ATTN_SPLIT(DK_, KG_)                                                                                     \
  hipLaunchKernelGGL((attn_fwd_f32_split_kernel<DK_, KG_>), grid, dim3(256 * (KG_)), 0, stream, in, out, S, nt, cz, \
                     scale, post_scale, post_bias, post_relu, tiles, ws)
  switch (D / 32) {
    case 1: if (plan.groups == 2) { LC_ATTN_SPLIT(1, 2); } else { LC_ATTN_SPLIT(1, 1); } break;
    case 2: if (plan.groups == 2) { LC_ATTN_SPLIT(2, 2); } else { LC_ATTN_SPLIT(2, 1); } break;
    case 3: LC_ATTN_SPLIT(3, 1); break;
    default: LC_ATTN_SPLIT(4, 1); break;
  }
#undef LC_ATTN_SPLIT
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || z == 1) {
    return e;
  }
  return attentionF32Combine(ws, out, bh, S, D, z, post_scale, post_bias, post_relu, stream);
}

}  // namespace lchip::kern
