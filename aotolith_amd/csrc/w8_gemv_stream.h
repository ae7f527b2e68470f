// Wave-persistent, software-pipelined form of the int8 decode GEMV: the semantics and rounding points of
// w8.h's kernel in the structure of w4_gemv_stream.h's block-staged one.
//
// w8.h's kernel stages x behind two block barriers before its first weight load and waits for every chunk of
// a row group before the next one's loads, so a layer projection ran at 2 to 3 TB/s. Here
//   * x goes out first, the first tile's weights right behind it, and x is normalized, rounded and staged once
//     per 4-wave block while they land;
//   * LPR lanes share a row, each with CPL 16-byte chunks (16 codes) of it; single projections keep the x
//     chunks a lane meets in registers, the paired form, with two weight sets, reads them from LDS;
//   * two register sets alternate over a wave's row tiles, the next tile's words, scales and bias loaded while
//     this one's are reduced, all unconditional (clamped), so the waits count the same loads on every path;
//   * scales and bias are read as the aligned 32-bit pair that holds the element (even group counts).
// Bound: HBM for wide outputs, launch and latency else. us over rotating weights, w8.h's kernel -> this: 512 -> 512
// 3.5 -> 2.4, 2048 -> 2048 4.4 -> 3.5, 5120 -> 5120 12.3 -> 7.5, 13824 -> 5120 25.6 -> 17.5, paired 5120 -> 13824
// 36.0 -> 28.1 (5.2 TB/s), 2048 -> 151936 61.1 -> 56.8 (5.6 TB/s).
#pragma once

#include "common.h"
#include "w4_gemv_stream.h"
#include "w8.h"

namespace aoto {

// Dot of one chunk's 16 codes (offset by 128, see chunk_dot_w8) with x in registers or LDS.
AOTO_DEVICE float chunk_dot_w8_xs(const uint4 q, const uint4 xa, const uint4 xb) {
  const uint4 x[2] = {xa, xb};
  return chunk_dot_w8(q, x);
}

template <int LPR, int CPL, int XV, bool NORM, bool PAIRED, bool BIAS>
__device__ __forceinline__ void w8_gemv_stream_body(const uint4* __restrict__ words,
                                                    const uint16_t* __restrict__ scales,
                                                    const uint16_t* __restrict__ x,
                                                    const uint16_t* __restrict__ norm_w, int K, int N, int group_shift,
                                                    const uint16_t* __restrict__ bias,
                                                    const uint4* __restrict__ up_words,
                                                    const uint16_t* __restrict__ up_scales, float eps, float alpha,
                                                    float beta, uint16_t* __restrict__ y) {
  extern __shared__ uint4 lds[];
  __shared__ float scratch[kGemvThreads / 64];
  constexpr int RPW = 64 / LPR;
  constexpr bool XREG = !PAIRED;
  const int nchunks = K >> 4, vecs = K >> 3, ngroups = nchunks >> group_shift;
  uint4* xs = lds;                                      // [nchunks][2], natural order
  float* csum = reinterpret_cast<float*>(lds + vecs);   // 128 x the chunk's sum
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & (LPR - 1), rsub = lane / LPR;
  const int tiles = (N + RPW - 1) / RPW, total_waves = gridDim.x * 4;

  int cidx[CPL], shalf[CPL];
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    cidx[j] = min(li + LPR * j, nchunks - 1);
    shalf[j] = (cidx[j] >> group_shift) & 1;
  }
  struct Regs {
    uint4 q[CPL], u[PAIRED ? CPL : 1];
    uint32_t s[CPL], us[PAIRED ? CPL : 1], b;
  };
  const uint32_t* scale_words = reinterpret_cast<const uint32_t*>(scales);
  const uint32_t* up_scale_words = reinterpret_cast<const uint32_t*>(up_scales);
  auto pair_half = [](uint32_t pair, int high) { return __uint_as_float(high ? (pair & 0xFFFF0000u) : (pair << 16)); };
  auto load = [&](int tile, Regs& r) {
    const int row = min(min(tile, tiles - 1) * RPW + rsub, N - 1);
    const size_t w = (size_t)row * nchunks, g = (size_t)row * (ngroups >> 1);
#pragma unroll
    for (int j = 0; j < CPL; ++j) r.q[j] = words[w + cidx[j]];
    if (PAIRED) {
#pragma unroll
      for (int j = 0; j < CPL; ++j) r.u[j] = up_words[w + cidx[j]];
    }
#pragma unroll
    for (int j = 0; j < CPL; ++j) r.s[j] = scale_words[g + (cidx[j] >> (group_shift + 1))];
    if (PAIRED) {
#pragma unroll
      for (int j = 0; j < CPL; ++j) r.us[j] = up_scale_words[g + (cidx[j] >> (group_shift + 1))];
    }
    if (BIAS) r.b = reinterpret_cast<const uint32_t*>(bias)[row >> 1];
  };

  uint4 raw[XV], wraw[NORM ? XV : 1];
#pragma unroll
  for (int i = 0; i < XV; ++i)
    raw[i] = reinterpret_cast<const uint4*>(x)[min((int)threadIdx.x + kGemvThreads * i, vecs - 1)];
  if (NORM) {
#pragma unroll
    for (int i = 0; i < XV; ++i)
      wraw[i] = reinterpret_cast<const uint4*>(norm_w)[min((int)threadIdx.x + kGemvThreads * i, vecs - 1)];
  }
  __builtin_amdgcn_sched_barrier(0);
  Regs ra, rb;
  int tile = blockIdx.x * 4 + wave;
  load(tile, ra);
  __builtin_amdgcn_sched_barrier(0);

  float ns = 1.f;
  if (NORM) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < XV; ++i)
      if ((int)threadIdx.x + kGemvThreads * i < vecs) ss = sum_squares8(raw[i], ss);
    ss = block_sum<kGemvThreads>(ss, scratch);
    ns = 1.0f / sqrtf(ss / (float)K + eps);
  }
#pragma unroll
  for (int i = 0; i < XV; ++i) {
    const int v = (int)threadIdx.x + kGemvThreads * i;
    uint32_t p[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
    if (NORM) {
      const uint32_t w[4] = {wraw[i].x, wraw[i].y, wraw[i].z, wraw[i].w};
#pragma unroll
      for (int k = 0; k < 4; ++k)
        p[k] = cvt_pk_bf16((ns * bf16_lo(p[k])) * bf16_lo(w[k]), (ns * bf16_hi(p[k])) * bf16_hi(w[k]));
    }
    float sum = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) sum = dot2_bf16(p[k], 0x43004300u, sum);  // 128 x, exact products
    sum += dpp_move<kDppXor1>(sum);
    if (v < vecs) {
      xs[v] = make_uint4(p[0], p[1], p[2], p[3]);
      if ((v & 1) == 0) csum[v >> 1] = sum;
    }
  }
  __syncthreads();
  uint4 xr[XREG ? CPL : 1][2];
  float cr[XREG ? CPL : 1];
  if (XREG) {
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      xr[j][0] = xs[2 * cidx[j]];
      xr[j][1] = xs[2 * cidx[j] + 1];
      cr[j] = csum[cidx[j]];
    }
  }

  auto consume = [&](int at, const Regs& r) {
    float total = 0.f, total_up = 0.f;
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      // a lane past the row's last chunk computes on the clamped one and weighs it zero
      const bool valid = li + LPR * j < nchunks;
      const uint4 xa = XREG ? xr[j][0] : xs[2 * cidx[j]], xb = XREG ? xr[j][1] : xs[2 * cidx[j] + 1];
      const float off = XREG ? cr[j] : csum[cidx[j]];
      total = fmaf(chunk_dot_w8_xs(r.q[j], xa, xb) - off, valid ? pair_half(r.s[j], shalf[j]) : 0.f, total);
      if (PAIRED)
        total_up = fmaf(chunk_dot_w8_xs(r.u[j], xa, xb) - off, valid ? pair_half(r.us[j], shalf[j]) : 0.f, total_up);
    }
    total = group_sum<LPR>(total);
    if (PAIRED) total_up = group_sum<LPR>(total_up);
    const int row = at * RPW + rsub;
    if (li == 0 && row < N) {
      float out = total;
      if (PAIRED) {
        const float g = round_bf16(total);
        out = total_up * (g / (1.0f + expf(-g)));
      } else if (BIAS) {
        out = beta * pair_half(r.b, row & 1) + alpha * total;
      }
      y[row] = (uint16_t)f32_to_bf16(out);
    }
  };
  // (as in the int4 form: a scheduling barrier after each prefetch, one exit, a wave's last tile prefetches
  // its clamped successor)
  while (tile < tiles) {
    load(tile + total_waves, rb);
    __builtin_amdgcn_sched_barrier(0);
    consume(tile, ra);
    tile += total_waves;
    if (tile >= tiles) break;
    load(tile + total_waves, ra);
    __builtin_amdgcn_sched_barrier(0);
    consume(tile, rb);
    tile += total_waves;
  }
}

}  // namespace aoto

#define AOTO_GEMV_W8_STREAM_INSTANCE(LPR, CPL, XV, NORM, PAIRED, BIAS)                                           \
  extern "C" __global__ __launch_bounds__(aoto::kGemvThreads) void                                             \
      aoto_w8_gemv_x##LPR##x##CPL##_n##NORM##_p##PAIRED##_b##BIAS(                                              \
          const uint4* words, const uint16_t* scales, const uint16_t* x, const uint16_t* norm_w, int K, int N,  \
          int group_shift, const uint16_t* bias, const uint4* up_words, const uint16_t* up_scales, float eps,   \
          float alpha, float beta, uint16_t* y) {                                                               \
    aoto::w8_gemv_stream_body<LPR, CPL, XV, NORM, PAIRED, BIAS>(words, scales, x, norm_w, K, N, group_shift,    \
                                                               bias, up_words, up_scales, eps, alpha, beta, y); \
  }
#define AOTO_GEMV_W8_STREAM_SINGLE(LPR, CPL, XV)          \
  AOTO_GEMV_W8_STREAM_INSTANCE(LPR, CPL, XV, 0, 0, 0)    \
  AOTO_GEMV_W8_STREAM_INSTANCE(LPR, CPL, XV, 0, 0, 1)    \
  AOTO_GEMV_W8_STREAM_INSTANCE(LPR, CPL, XV, 1, 0, 0)    \
  AOTO_GEMV_W8_STREAM_INSTANCE(LPR, CPL, XV, 1, 0, 1)
#define AOTO_GEMV_W8_STREAM_PAIRED(LPR, CPL, XV)          \
  AOTO_GEMV_W8_STREAM_INSTANCE(LPR, CPL, XV, 1, 1, 0)    \
  AOTO_GEMV_W8_STREAM_INSTANCE(LPR, CPL, XV, 0, 1, 0)
