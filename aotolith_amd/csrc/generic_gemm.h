// The graph plans' matrix product on the matrix cores: out = alpha * A @ B (+ beta * bias),
// batched, any strides, f32 accumulation, one rounding to the output type.
//
// bf16 x bf16 runs v_mfma_f32_32x32x16_bf16 (the products of bf16 values are exact in its f32
// accumulators), every other float pair v_mfma_f32_32x32x2_f32 on f32 operands: the precision of the
// f32 FMA loop this replaces, in another summation order.
//
// A block owns a (64 MT) x (64 NT) tile, four waves of (32 MT) x (32 NT) per k-group. KG k-groups
// take the k-steps (128 bytes of k: 64 bf16 or 32 f32) in turn, each with its own double-buffered
// stage, and sum through LDS at the end: the graphs' grids are small (512 x 896 outputs are 112 tiles
// of 64 x 64 on 256 CUs), so a block's four groups stand in for the blocks that a larger grid would
// have. Operands go global -> registers -> LDS one step ahead, rows of 8 16-byte chunks with the chunk
// index XORed by the row (conflict-free for the 32-row operand reads).
//
// Bound: latency (few tiles, 4 to 19 trips of one load round trip each) and, in large grids, the MFMA
// pipe. 512 rows, bf16, traced in a block, against the f32 FMA kernel with per-element typed loads that
// this replaces: 896 -> 128 126.7 -> 13.2 us, 896 -> 896 138.3 -> 13.8, 896 -> 4864 169.9 -> 17.7.
//
// MODE says how a step's chunks are read:
//   kVec   both operands contiguous along k: 16-byte loads (K, strides and bases multiples of 16 bytes)
//   kCols  B contiguous along n instead (a product with an untransposed right operand): loads along n
//          (pairs of columns for bf16), transposed in registers
//   kAny   element loads through the strides, of any float type: odd sizes, other layouts
#pragma once

#include "aoto_hip.h"
#include "common.h"
#include "generic.h"
#include "generic_args.h"

namespace aoto {

typedef float f32x16_t __attribute__((ext_vector_type(16)));

enum { kVec = 0, kCols = 1, kAny = 2 };

template <typename T>
AOTO_DEVICE uint4 gemm_chunk_any(const void* p, int dtype, long long off, long long step, int count) {
  constexpr int E = 16 / (int)sizeof(T);
  uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int e = 0; e < E; ++e) {
    if (e < count) {
      if (sizeof(T) == 2)
        w[e >> 1] |= (uint32_t) static_cast<const uint16_t*>(p)[off + e * step] << (16 * (e & 1));
      else
        w[e & 3] = __float_as_uint(load_float(p, dtype, off + e * step));
    }
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

template <typename T, int MODE, int MT, int NT, int KG>
__device__ __forceinline__ void generic_gemm_body(const GemmArgs& g) {
  constexpr int E = 16 / (int)sizeof(T);    // elements of a chunk
  constexpr int BK = 8 * E;                 // k of a step
  constexpr int BM = 64 * MT, BN = 64 * NT;
  constexpr int RA = BM / 32, RB = BN / 32;  // chunks of A / B a thread of the group stages
  constexpr int kStage = (BM + BN) * 8;      // chunks of one buffer
  constexpr int kRed = KG > 1 ? (KG - 1) * 4 * MT * NT * 16 * 64 / 4 : 0;  // chunks of the groups' sums
  constexpr int kLds = KG * 2 * kStage > kRed ? KG * 2 * kStage : kRed;
  __shared__ uint4 lds[kLds];

  const int t = threadIdx.x & 255, group = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const long long batch = blockIdx.z;
  const long long m0 = (long long)blockIdx.y * BM, n0 = (long long)blockIdx.x * BN;
  const char* ab = static_cast<const char*>(g.a);
  const char* bb = static_cast<const char*>(g.b);
  uint4* stage = lds + group * 2 * kStage;

  const int steps = (int)((g.k + BK - 1) / BK);
  const int trips = (steps + KG - 1) / KG;
  const int row = t >> 3, c = t & 7;

  uint4 ra[RA], rb[RB];
  auto load = [&](int step) {
    const long long k = (long long)step * BK + c * E;
    if (MODE != kAny) {
      // (K is a whole number of chunks: a chunk past K reads in bounds and becomes zeros)
      const bool live = k < g.k;
      const long long kc = live ? k : 0;
#pragma unroll
      for (int i = 0; i < RA; ++i) {
        const long long r = min(m0 + row + 32 * i, g.m - 1);
        const uint4 v = *reinterpret_cast<const uint4*>(ab + (batch * g.sa_b + r * g.sa_m + kc) * (long long)sizeof(T));
        ra[i] = live ? v : make_uint4(0u, 0u, 0u, 0u);
      }
    } else {
      const int count = (int)min((long long)E, g.k - k);
#pragma unroll
      for (int i = 0; i < RA; ++i) {
        const long long r = min(m0 + row + 32 * i, g.m - 1);
        ra[i] = gemm_chunk_any<T>(g.a, g.a_dtype, batch * g.sa_b + r * g.sa_m + k * g.sa_k, g.sa_k, count);
      }
    }
    if (MODE == kVec) {
      const bool live = k < g.k;
      const long long kc = live ? k : 0;
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const long long n = min(n0 + row + 32 * i, g.n - 1);
        const uint4 v = *reinterpret_cast<const uint4*>(bb + (batch * g.sb_b + n * g.sb_n + kc) * (long long)sizeof(T));
        rb[i] = live ? v : make_uint4(0u, 0u, 0u, 0u);
      }
    } else if (MODE == kAny) {
      const int count = (int)min((long long)E, g.k - k);
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const long long n = min(n0 + row + 32 * i, g.n - 1);
        rb[i] = gemm_chunk_any<T>(g.b, g.b_dtype, batch * g.sb_b + k * g.sb_k + n * g.sb_n, g.sb_k, count);
      }
    } else if (sizeof(T) == 2) {
      // a thread owns column pairs (2p, 2p + 1) of one chunk of 8 k: 8 dword loads, 128 bytes of a
      // row per half wave, then the two columns' chunks by byte permutes
      const int p = t & 31, ck = t >> 5;
#pragma unroll
      for (int i = 0; i < RB / 2; ++i) {
        const long long n = min(n0 + 2 * p + 64 * i, g.n - 2);
        uint32_t w[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const long long kk = (long long)step * BK + ck * 8 + e;
          const uint32_t v = *reinterpret_cast<const uint32_t*>(
              bb + (batch * g.sb_b + min(kk, g.k - 1) * g.sb_k + n) * 2);
          w[e] = kk < g.k ? v : 0u;
        }
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          lo[e] = __builtin_amdgcn_perm(w[2 * e + 1], w[2 * e], 0x05040100u);
          hi[e] = __builtin_amdgcn_perm(w[2 * e + 1], w[2 * e], 0x07060302u);
        }
        rb[2 * i] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        rb[2 * i + 1] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
      }
    } else {
      // f32: a thread owns column p of one chunk of 4 k
      const int p = t & 31, ck = t >> 5;
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const long long n = min(n0 + p + 32 * i, g.n - 1);
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const long long kk = (long long)step * BK + ck * 4 + e;
          const uint32_t v = *reinterpret_cast<const uint32_t*>(
              bb + (batch * g.sb_b + min(kk, g.k - 1) * g.sb_k + n) * 4);
          w[e] = kk < g.k ? v : 0u;
        }
        rb[i] = make_uint4(w[0], w[1], w[2], w[3]);
      }
    }
  };
  auto store = [&](uint4* buf) {
#pragma unroll
    for (int i = 0; i < RA; ++i) {
      const int r = row + 32 * i;
      buf[r * 8 + (c ^ (r & 7))] = ra[i];
    }
    uint4* bufb = buf + BM * 8;
    if (MODE != kCols) {
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const int r = row + 32 * i;
        bufb[r * 8 + (c ^ (r & 7))] = rb[i];
      }
    } else {
      const int p = t & 31, ck = t >> 5;
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const int r = sizeof(T) == 2 ? 2 * p + (i & 1) + 64 * (i >> 1) : p + 32 * i;
        bufb[r * 8 + (ck ^ (r & 7))] = rb[i];
      }
    }
  };

  const int wm = (wave >> 1) * 32 * MT, wn = (wave & 1) * 32 * NT;
  const int lr = lane & 31, half = lane >> 5;
  f32x16_t acc[MT][NT] = {};
  auto compute = [&](const uint4* buf) {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      uint4 av[MT], bv[NT];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int r = wm + 32 * i + lr;
        av[i] = buf[r * 8 + ((2 * kk + half) ^ (r & 7))];
      }
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int r = wn + 32 * j + lr;
        bv[j] = buf[BM * 8 + r * 8 + ((2 * kk + half) ^ (r & 7))];
      }
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          if (sizeof(T) == 2) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                __builtin_bit_cast(bf16x8_t, av[i]), __builtin_bit_cast(bf16x8_t, bv[j]), acc[i][j], 0, 0, 0);
          } else {
            // the halves' chunks hold k 8kk .. 8kk+3 and 8kk+4 .. 8kk+7: product e takes one of each,
            // for both operands alike
            const uint32_t aw[4] = {av[i].x, av[i].y, av[i].z, av[i].w}, bw[4] = {bv[j].x, bv[j].y, bv[j].z, bv[j].w};
#pragma unroll
            for (int e = 0; e < 4; ++e)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(aw[e]), __uint_as_float(bw[e]),
                                                               acc[i][j], 0, 0, 0);
          }
        }
    }
  };

  if (trips > 0) {
    load(group);
    store(stage);
  }
  __syncthreads();
  for (int s = 0; s < trips; ++s) {
    const bool more = s + 1 < trips;  // uniform; a step past the last loads zeros
    if (more) load((s + 1) * KG + group);
    compute(stage + (s & 1) * kStage);
    if (more) store(stage + ((s + 1) & 1) * kStage);
    __syncthreads();
  }

  if (KG > 1) {
    float* red = reinterpret_cast<float*>(lds);
    if (group > 0) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            red[((((group - 1) * 4 + wave) * MT * NT + i * NT + j) * 16 + r) * 64 + lane] = acc[i][j][r];
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int other = 0; other < KG - 1; ++other)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            acc[i][j][r] += red[(((other * 4 + wave) * MT * NT + i * NT + j) * 16 + r) * 64 + lane];
  }

#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const long long n = n0 + wn + 32 * j + lr;
    if (n >= g.n) continue;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const long long m = m0 + wm + 32 * i + 8 * (r >> 2) + 4 * half + (r & 3);
        if (m >= g.m) continue;
        float v = acc[i][j][r];
        if (g.alpha != 1.f) v *= g.alpha;
        if (g.bias) {
          const float b = (float)load_value(g.bias, g.bias_dtype, batch * g.sbias_b + m * g.sbias_m + n * g.sbias_n);
          v = g.beta == 1.f ? v + b : v + g.beta * b;
        }
        store_float_type(g.c, g.c_dtype, batch * g.sc_b + m * g.sc_m + n * g.sc_n, v);
      }
  }
}

}  // namespace aoto

#define AOTO_GENERIC_GEMM(TYPE, T, LETTER, MODE, TILES, KG)                              \
  extern "C" __global__ __launch_bounds__(256 * KG) void                                 \
      aoto_generic_gemm_##TYPE##_##LETTER##_t##TILES##k##KG(aoto::GemmArgs g) {          \
    aoto::generic_gemm_body<T, MODE, TILES, TILES, KG>(g);                               \
  }
#define AOTO_GENERIC_GEMM_MODE(TYPE, T, LETTER, MODE)   \
  AOTO_GENERIC_GEMM(TYPE, T, LETTER, MODE, 1, 1)        \
  AOTO_GENERIC_GEMM(TYPE, T, LETTER, MODE, 1, 2)        \
  AOTO_GENERIC_GEMM(TYPE, T, LETTER, MODE, 1, 4)        \
  AOTO_GENERIC_GEMM(TYPE, T, LETTER, MODE, 2, 1)
