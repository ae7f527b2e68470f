// Symmetric int4 group quantizer/packer and the bf16 unpack, on the GPU.
//
// Bit-exact restatement of quantize.py:95-152 and models/quantized.py:61-76,
// 133-163 of the reference:
//   scale = max|w| / 7 in f32 (an all-zero group takes 1/7);
//   code  = clip(rint(w / scale), -8, 7) with IEEE f32 division, half-to-even;
//   word j of a row holds codes 8j..8j+7, code 8j+k at bits 4k;
//   the stored scale is bf16(scale) (RNE) while the codes use the f32 scale.
// The unpack writes bf16(code * scale_bf16), the torch op's value in bf16.
#pragma once

#include "common.h"

// One thread per (row, group), for groups or bases the coalesced packer does not take.
// `src_f32` selects an f32 source, else bf16.
extern "C" __global__ __launch_bounds__(256) void aoto_w4_quantize(
    const void* __restrict__ src, int src_f32, int rows, int inner, int group,
    int32_t* __restrict__ packed, uint16_t* __restrict__ scales_bf16, float* __restrict__ scales_f32) {
  const int groups = inner / group;
  const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
  if (gid >= (long long)rows * groups) return;
  const int row = (int)(gid / groups);
  const int g = (int)(gid - (long long)row * groups);
  const size_t base = (size_t)row * inner + (size_t)g * group;
  auto load = [&](int i) -> float {
    if (src_f32) return reinterpret_cast<const float*>(src)[base + i];
    return bf16_to_f32(reinterpret_cast<const uint16_t*>(src)[base + i]);
  };
  float widest = 0.f;
  for (int i = 0; i < group; ++i) widest = fmaxf(widest, fabsf(load(i)));
  const float scale = (widest > 0.f ? widest : 1.0f) / 7.0f;
  int32_t* out = packed + (size_t)row * (inner >> 3) + (size_t)g * (group >> 3);
  for (int w = 0; w < (group >> 3); ++w) {
    uint32_t word = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      float code = rintf(load(w * 8 + k) / scale);
      code = fminf(fmaxf(code, -8.0f), 7.0f);
      word |= ((uint32_t)(int)code & 0xFu) << (4 * k);
    }
    out[w] = (int32_t)word;
  }
  scales_bf16[(size_t)row * groups + g] = (uint16_t)f32_to_bf16(scale);
  if (scales_f32) scales_f32[(size_t)row * groups + g] = scale;
}

namespace aoto {

// The coalesced packer, either width: a thread takes four units of 8 consecutive
// weights, 256 units apart (a wave's 16-byte loads are 1 KB of one row each), a
// group is 2^shift neighbouring lanes, whose maximum is a DPP / permlane reduction,
// and a unit's codes leave as one store of its one (two) whole words. Same f32
// arithmetic per weight as the kernels above, so the codes are the same bits: the
// maximum of a group does not depend on the order (fmaxf drops NaN in any order).
// Bound: HBM (2 or 4 bytes read per weight). One thread per group read 2 bytes per
// lane 128 bytes apart, twice: 14336 x 4096 bf16 to int4 2014 us there, 35.5 us (4.2
// TB/s of the 4.9 that a copy reaches) here.
template <int BITS>
__device__ __forceinline__ void quantize_units_body(const void* __restrict__ src, int src_f32, int shift,
                                                    long long units, int32_t* __restrict__ packed,
                                                    uint16_t* __restrict__ scales_bf16,
                                                    float* __restrict__ scales_f32) {
  constexpr int kUnits = 4;
  constexpr float kTop = BITS == 4 ? 7.0f : 127.0f;
  const long long first = (long long)blockIdx.x * (256 * kUnits) + threadIdx.x;
  float w[kUnits][8];
#pragma unroll
  for (int i = 0; i < kUnits; ++i) {
    // lanes past the end read the last unit and store nothing; units come in whole
    // groups, so such a lane never shares a group with a live one
    const long long u = min(first + i * 256, units - 1);
    if (src_f32) {
      const float4 a = reinterpret_cast<const float4*>(src)[2 * u], b = reinterpret_cast<const float4*>(src)[2 * u + 1];
      w[i][0] = a.x, w[i][1] = a.y, w[i][2] = a.z, w[i][3] = a.w;
      w[i][4] = b.x, w[i][5] = b.y, w[i][6] = b.z, w[i][7] = b.w;
    } else {
      const uint4 r = reinterpret_cast<const uint4*>(src)[u];
      const uint32_t raw[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        w[i][2 * j] = bf16_lo(raw[j]);
        w[i][2 * j + 1] = bf16_hi(raw[j]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < kUnits; ++i) {
    const long long u = first + i * 256;
    float widest = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) widest = fmaxf(widest, fabsf(w[i][k]));
    if (shift >= 1) widest = fmaxf(widest, dpp_move<kDppXor1>(widest));
    if (shift >= 2) widest = fmaxf(widest, dpp_move<kDppXor2>(widest));
    if (shift >= 3) widest = fmaxf(widest, dpp_move<kDppHalfMirror>(widest));
    if (shift >= 4) widest = fmaxf(widest, dpp_move<kDppMirror>(widest));
    if (shift >= 5) widest = xor16_max(widest);
    if (shift >= 6) widest = xor32_max(widest);
    const float scale = (widest > 0.f ? widest : 1.0f) / kTop;
    // The code is rint(w / scale), w / scale correctly rounded. A product with the reciprocal is within 3e-5 of
    // it (127 and a last place and a half), so it rounds to the same whole number unless it lies that close to a
    // half: there, for scales whose reciprocal is not a normal number, and for values that are not finite, the
    // division decides (the division everywhere took 40.6 us, VALU-bound).
    const float inverse = 1.0f / scale;
    const bool plain = scale > 1e-30f && scale < 1e30f;
    uint32_t word[2] = {0u, 0u};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float near = w[i][k] * inverse;
      float code = rintf(near);
      if (!(plain && fabsf(near - code) < 0.4999f)) code = rintf(w[i][k] / scale);
      code = fminf(fmaxf(code, -kTop - 1.0f), kTop);
      if (BITS == 4)
        word[0] |= ((uint32_t)(int)code & 0xFu) << (4 * k);
      else
        word[k >> 2] |= ((uint32_t)(int)code & 0xFFu) << (8 * (k & 3));
    }
    if (u < units) {
      if (BITS == 4)
        packed[u] = (int32_t)word[0];
      else
        reinterpret_cast<uint2*>(packed)[u] = make_uint2(word[0], word[1]);
      if ((u & ((1ll << shift) - 1)) == 0) {
        scales_bf16[u >> shift] = (uint16_t)f32_to_bf16(scale);
        if (scales_f32) scales_f32[u >> shift] = scale;
      }
    }
  }
}

}  // namespace aoto

extern "C" __global__ __launch_bounds__(256) void aoto_w4_quantize_units(
    const void* __restrict__ src, int src_f32, int shift, long long units, int32_t* __restrict__ packed,
    uint16_t* __restrict__ scales_bf16, float* __restrict__ scales_f32) {
  aoto::quantize_units_body<4>(src, src_f32, shift, units, packed, scales_bf16, scales_f32);
}

extern "C" __global__ __launch_bounds__(256) void aoto_w8_quantize_units(
    const void* __restrict__ src, int src_f32, int shift, long long units, int32_t* __restrict__ packed,
    uint16_t* __restrict__ scales_bf16, float* __restrict__ scales_f32) {
  aoto::quantize_units_body<8>(src, src_f32, shift, units, packed, scales_bf16, scales_f32);
}

// One thread per packed word: eight bf16(code * scale) values, one 16-byte store.
extern "C" __global__ __launch_bounds__(256) void aoto_w4_dequantize(
    const int32_t* __restrict__ packed, const uint16_t* __restrict__ scales, int rows, int inner,
    int group, uint16_t* __restrict__ out) {
  const int words = inner >> 3;
  const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
  if (gid >= (long long)rows * words) return;
  const int row = (int)(gid / words);
  const int w = (int)(gid - (long long)row * words);
  const uint32_t word = (uint32_t)packed[gid];
  const float s = bf16_to_f32(scales[(size_t)row * (inner / group) + (w * 8) / group]);
  uint32_t v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int code = (int)(word << (28 - 4 * k)) >> 28;
    v[k] = f32_to_bf16((float)code * s);
  }
  uint4 o;
  o.x = v[0] | (v[1] << 16);
  o.y = v[2] | (v[3] << 16);
  o.z = v[4] | (v[5] << 16);
  o.w = v[6] | (v[7] << 16);
  reinterpret_cast<uint4*>(out)[gid] = o;
}
