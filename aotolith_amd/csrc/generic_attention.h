// The graph plans' scaled-dot-product attention on the matrix cores.
//
// out[b][h][i] = softmax_j(scale * q_i . k_j + mask) v_j, f32 scores and softmax: a bool mask keeps
// True entries, a float mask is added, is_causal keeps j <= i (aligned to the top-left, as torch's), a
// row with every key masked gives zeros, and a key whose probability is zero contributes nothing,
// whatever its value holds - the semantics of aoto_generic_attention, which keeps head sizes over 128.
//
// A block owns 32 queries of one head; its four waves take the key tiles in turn, each with its own
// running softmax (no barrier inside the loop), and combine through LDS at the end. Per wave and tile:
//   S^T [keys x 32 queries] = K . Q^T    K straight from global memory in operand order, Q in registers
//   O^T [d x 32 queries] += V^T . P^T    P from S^T's accumulators, lane l holding query l % 32
// bf16 operands: 64-key tiles on v_mfma_f32_32x32x16_bf16, V staged row-major in the wave's LDS and read
// with the transposing LDS reads; P stays at f32 precision: it enters as three bf16 terms (8 + 8 + 8
// bits: p = hi + mid + lo exactly, short of the f32's underflow), three products into the one f32 sum.
// f32 (and mixed) operands: 32-key tiles on v_mfma_f32_32x32x2_f32, V read in operand order.
//
// Values that are not finite: 0 * inf would poison every query through the product, so they enter it as
// zeros, and a wave that met any goes over its keys once more (special_values) with the row's final
// maximum and gives +-inf / NaN to the queries whose probability of such a key is not zero. (Within the loop
// a key's probability is still relative to the maximum so far: one that ends as zero may not be zero yet.)
// A kept score that is NaN makes its query NaN: it stays in the running sum, which no rescale to zero drops.
//
// Bound: latency (two tiles a wave at 512 keys), then the MFMA pipe. 14 heads of 64, 512 tokens,
// causal, bf16: 881 us with one block per query row and scalar dots (every score a 64-step chain of
// typed loads) -> 14.8 us. The loads of V and of the mask are free of branches on types (one per tile) and edges
// (clamped, their weights zero): with a branch an element it was 16.9 us, 8 heads of f32 41.1 against 22.6, one query
// of 8 heads over 64 f32 keys 15.0 against 10.0 - and the masks of those branches and 460 registers made the compiler
// split live ranges across them, in one form of this source with a copy under the wrong lanes.
#pragma once

#include "aoto_hip.h"
#include "common.h"
#include "flash_attention.h"
#include "generic.h"
#include "generic_args.h"

namespace aoto {

constexpr int kGenAttnQueries = 32;
constexpr int kGenAttnWaves = 4;

// Order of one wave's own LDS writes and reads (the hardware keeps it; this keeps the compiler to it).
AOTO_DEVICE void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

AOTO_DEVICE bool not_finite_f32(float v) { return (__float_as_uint(v) & 0x7F800000u) == 0x7F800000u; }

// One 16-byte operand chunk (8 bf16 or 4 f32) at `off` along stride `step`, elements from `count` on zero.
template <bool F32, bool VEC>
AOTO_DEVICE uint4 attn_chunk(const void* p, int dtype, long long off, long long step, int count) {
  if (VEC) {
    // whole chunks only (the host checks the head sizes): past the row's end nothing is read
    if (count <= 0) return make_uint4(0u, 0u, 0u, 0u);
    return F32 ? *reinterpret_cast<const uint4*>(static_cast<const float*>(p) + off)
               : *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p) + off);
  }
  uint32_t w[4] = {0u, 0u, 0u, 0u};
  constexpr int E = F32 ? 4 : 8;
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (e < count) {
      if (F32)
        w[e & 3] = __float_as_uint(load_float(p, dtype, off + e * step));
      else
        w[e >> 1] |= (uint32_t) static_cast<const uint16_t*>(p)[off + e * step] << (16 * (e & 1));
    }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

template <bool F32, int D, bool VEC>
__device__ __forceinline__ void generic_attention_body(const AttnArgs& a) {
  constexpr int E = F32 ? 4 : 8;          // elements of a 16-byte chunk
  constexpr int KT = F32 ? 1 : 2;         // 32-key parts of a tile
  constexpr int BK = 32 * KT;
  constexpr int S = D / (2 * E);          // operand chunks of a row and half
  constexpr int DT = D / 32;
  constexpr int STRV = D + 32;            // bf16 of a staged V row (transpose reads touch all banks)
  constexpr int RC = D / E;               // chunks of a V row
  constexpr int VL = F32 ? 1 : BK * RC / 64;  // V chunks a lane stages
  constexpr int REC = 2 + 16 * DT;        // a lane's softmax state: max, sum, O
  constexpr int kWaveBytes = 64 * REC * 4 > (F32 ? 0 : BK * STRV * 2) ? 64 * REC * 4 : BK * STRV * 2;
  __shared__ __attribute__((aligned(16))) char lds[kGenAttnWaves][kWaveBytes];

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, half = lane >> 5;
  const int h = blockIdx.y % a.heads, b = blockIdx.y / a.heads;
  const int kvh = h / (a.heads / a.kv_heads);
  // the last query tile first: a causal one has the most keys
  const int q0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * kGenAttnQueries;
  const int qi = q0 + col, qrow = min(qi, a.lq - 1);
  const long long kbase = b * a.ks[0] + kvh * a.ks[1], vbase = b * a.vs[0] + kvh * a.vs[1];
  uint16_t* vs = reinterpret_cast<uint16_t*>(lds[wave]);

  uint4 qf[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int d0 = (2 * s + half) * E;
    qf[s] = attn_chunk<F32, VEC>(a.q, a.q_dtype,
                                 b * a.qs[0] + h * a.qs[1] + qrow * a.qs[2] + d0 * a.qs[3], a.qs[3], a.d - d0);
  }

  const int last_key = a.causal ? min(a.lk, q0 + kGenAttnQueries) : a.lk;
  const int tiles = (last_key + BK - 1) / BK;

  uint4 kf[KT][S], vf[VL];
  auto load_keys = [&](int j0) {
#pragma unroll
    for (int sub = 0; sub < KT; ++sub) {
      const long long off = kbase + (long long)min(j0 + 32 * sub + col, a.lk - 1) * a.ks[2];
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int d0 = (2 * s + half) * E;
        kf[sub][s] = attn_chunk<F32, VEC>(a.k, a.k_dtype, off + d0 * a.ks[3], a.ks[3], a.d - d0);
      }
    }
  };
  auto load_values = [&](int j0) {
    if constexpr (!F32) {
#pragma unroll
      for (int i = 0; i < VL; ++i) {
        const int c = lane + 64 * i, row = c / RC, d0 = (c % RC) * E;
        const long long off = vbase + (long long)min(j0 + row, a.lk - 1) * a.vs[2] + d0 * a.vs[3];
        vf[i] = attn_chunk<F32, VEC>(a.v, a.v_dtype, off, a.vs[3], a.dv - d0);
      }
    }
  };
  // f32 V in operand order: key (e, half) of a tile, column 32 t + col. One branch on the type and none on the
  // edges: a branch a load serialized the loads and spilled the scalar registers of their masks.
  float vf32[F32 ? 16 : 1][F32 ? DT : 1];
  auto load_values_f32 = [&](int j0) {
    if constexpr (F32) {
      auto at = [&](int e, int t) {
        const int j = min(j0 + 8 * (e >> 2) + 4 * half + (e & 3), a.lk - 1), d = min(32 * t + col, a.dv - 1);
        return vbase + (long long)j * a.vs[2] + (long long)d * a.vs[3];
      };
      if (a.v_dtype == AOTO_DT_F32) {
#pragma unroll
        for (int e = 0; e < 16; ++e)
#pragma unroll
          for (int t = 0; t < DT; ++t) vf32[e][t] = static_cast<const float*>(a.v)[at(e, t)];
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e)
#pragma unroll
          for (int t = 0; t < DT; ++t) vf32[e][t] = bf16_to_f32(static_cast<const uint16_t*>(a.v)[at(e, t)]);
      }
    }
  };

  const long long mrow = b * a.ms[0] + h * a.ms[1] + (long long)qrow * a.ms[2];
  f32x16_t o[DT] = {}, p[KT];
  float run_max = -INFINITY, run_sum = 0.f;

  // +-inf and NaN of the wave's keys, added to its recorded products for the queries whose probability of the key is
  // not zero. Key by key and column by column: the pass is as rare as such values, and its code is kept short.
  auto special_values = [&](float* products_record, float top) {
    const long long qbase = b * a.qs[0] + h * a.qs[1] + qrow * a.qs[2];
#pragma nounroll
    for (int tile = wave; tile < tiles; tile += kGenAttnWaves) {
#pragma nounroll
      for (int j = tile * BK; j < min(tile * BK + BK, a.lk); ++j) {
        const long long vrow = vbase + (long long)j * a.vs[2];
        bool any = false;
#pragma nounroll
        for (int d = lane; d < a.dv; d += 64)
          any = any || not_finite_f32(load_float(a.v, a.v_dtype, vrow + d * a.vs[3]));
        if (!__any(any)) continue;
        bool keep = !(a.causal && j > qi);
        float add = 0.f;
        if (a.mask != nullptr && keep) {
          const long long mo = mrow + (long long)j * a.ms[3];
          if (a.mask_dtype == AOTO_DT_BOOL)
            keep = static_cast<const uint8_t*>(a.mask)[mo] != 0;
          else
            add = load_float(a.mask, a.mask_dtype, mo);
        }
        float dot = 0.f;
#pragma nounroll
        for (int d = 0; d < a.d; ++d)
          dot = fmaf(load_float(a.q, a.q_dtype, qbase + d * a.qs[3]),
                     load_float(a.k, a.k_dtype, kbase + (long long)j * a.ks[2] + d * a.ks[3]), dot);
        const float score = keep ? dot * a.scale + add : -INFINITY;
        if (score == -INFINITY || expf(score - top) == 0.f) continue;
#pragma nounroll
        for (int r = 0; r < 16 * DT; ++r) {
          const int d = 8 * (r >> 2) + 4 * half + (r & 3);
          const float v = d < a.dv ? load_float(a.v, a.v_dtype, vrow + d * a.vs[3]) : 0.f;
          if (not_finite_f32(v)) products_record[r * 64 + lane] += v;
        }
      }
    }
  };

  if (wave < tiles) {
    load_keys(wave * BK);
    load_values(wave * BK);
  }
  bool odd = false;  // the lane has met a value that is not finite
  for (int tile = wave; tile < tiles; tile += kGenAttnWaves) {
    const int j0 = tile * BK;
    const int next = min(tile + kGenAttnWaves, tiles - 1) * BK;

    if constexpr (!F32) {
      wave_lds_order();
#pragma unroll
      for (int i = 0; i < VL; ++i) {
        const int c = lane + 64 * i, row = c / RC, cc = c % RC;
        uint32_t w[4] = {vf[i].x, vf[i].y, vf[i].z, vf[i].w};
        bool mine = false;
#pragma unroll
        for (int u = 0; u < 4; ++u)
          mine = mine || (w[u] & 0x7F80u) == 0x7F80u || (w[u] & 0x7F800000u) == 0x7F800000u;
        if (mine) {
          odd = true;
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if ((w[u] & 0x7F80u) == 0x7F80u) w[u] &= 0xFFFF0000u;
            if ((w[u] & 0x7F800000u) == 0x7F800000u) w[u] &= 0xFFFFu;
          }
        }
        *reinterpret_cast<uint4*>(vs + row * STRV + cc * E) = make_uint4(w[0], w[1], w[2], w[3]);
      }
      wave_lds_order();
    }

    f32x16_t sc[KT];
#pragma unroll
    for (int sub = 0; sub < KT; ++sub) {
      sc[sub] = f32x16_t{};
#pragma unroll
      for (int s = 0; s < S; ++s) {
        if constexpr (F32) {
          const uint32_t kw[4] = {kf[sub][s].x, kf[sub][s].y, kf[sub][s].z, kf[sub][s].w};
          const uint32_t qw[4] = {qf[s].x, qf[s].y, qf[s].z, qf[s].w};
#pragma unroll
          for (int e = 0; e < 4; ++e)
            sc[sub] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(kw[e]), __uint_as_float(qw[e]), sc[sub], 0,
                                                           0, 0);
        } else {
          sc[sub] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, kf[sub][s]),
                                                            __builtin_bit_cast(bf16x8_t, qf[s]), sc[sub], 0, 0, 0);
        }
      }
    }
    // the next tile's loads work under this one's softmax and products (the last trip reads its own again)
    load_values_f32(j0);
    load_keys(next);
    load_values(next);

    // Scaled and masked, with one branch on the mask's type and none on its edges (the mask of a key past the last
    // is read at the last).
    auto key_of = [&](int sub, int e) { return j0 + 32 * sub + 8 * (e >> 2) + 4 * half + (e & 3); };
#pragma unroll
    for (int sub = 0; sub < KT; ++sub)
#pragma unroll
      for (int e = 0; e < 16; ++e) p[sub][e] = sc[sub][e] * a.scale;
    if (a.mask != nullptr) {
      auto mask_at = [&](int sub, int e) { return mrow + (long long)min(key_of(sub, e), a.lk - 1) * a.ms[3]; };
      if (a.mask_dtype == AOTO_DT_BOOL) {
#pragma unroll
        for (int sub = 0; sub < KT; ++sub)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            p[sub][e] = static_cast<const uint8_t*>(a.mask)[mask_at(sub, e)] != 0 ? p[sub][e] : -INFINITY;
      } else if (a.mask_dtype == AOTO_DT_F32) {
#pragma unroll
        for (int sub = 0; sub < KT; ++sub)
#pragma unroll
          for (int e = 0; e < 16; ++e) p[sub][e] += static_cast<const float*>(a.mask)[mask_at(sub, e)];
      } else {
#pragma unroll
        for (int sub = 0; sub < KT; ++sub)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            p[sub][e] += bf16_to_f32(static_cast<const uint16_t*>(a.mask)[mask_at(sub, e)]);
      }
    }
    float tile_max = -INFINITY;
    const int keys_end = a.causal ? min(a.lk, qi + 1) : a.lk;
#pragma unroll
    for (int sub = 0; sub < KT; ++sub)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        p[sub][e] = key_of(sub, e) < keys_end ? p[sub][e] : -INFINITY;
        tile_max = fmaxf(tile_max, p[sub][e]);
      }
    tile_max = xor32_max(tile_max);
    const float moved = fmaxf(run_max, tile_max);
    // (a maximum of -inf has only zeros, or a NaN score's NaN, behind it: kept as they are)
    const float correction = run_max == moved || run_max == -INFINITY ? 1.f : expf(run_max - moved);
    run_max = moved;
    if (__any(correction != 1.f)) {
      // a correction of zero drops the products, overflowed ones too, and of the sum all but a NaN
      run_sum *= correction;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] = correction == 0.f ? 0.f : o[t][e] * correction;
    }
#pragma unroll
    for (int sub = 0; sub < KT; ++sub)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        p[sub][e] = p[sub][e] == -INFINITY ? 0.f : expf(p[sub][e] - moved);
        run_sum += p[sub][e];
      }

    if constexpr (F32) {
#pragma unroll
      for (int e = 0; e < 16; ++e)
#pragma unroll
        for (int t = 0; t < DT; ++t) {
          // (rows past the keys and columns past the head repeat the last: their weight is zero, or they are not
          // stored)
          const bool special = not_finite_f32(vf32[e][t]);
          odd = odd || special;
          const float v = special ? 0.f : vf32[e][t];
          o[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, p[0][e], o[t], 0, 0, 0);
        }
    } else {
#pragma unroll
      for (int kt = 0; kt < 2 * KT; ++kt) {
        uint32_t hi[4], mid[4], lo[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p0 = p[kt >> 1][8 * (kt & 1) + 2 * i], p1 = p[kt >> 1][8 * (kt & 1) + 2 * i + 1];
          hi[i] = cvt_pk_bf16(p0, p1);
          const float r0 = p0 - bf16_lo(hi[i]), r1 = p1 - bf16_hi(hi[i]);
          mid[i] = cvt_pk_bf16(r0, r1);
          lo[i] = cvt_pk_bf16(r0 - bf16_lo(mid[i]), r1 - bf16_hi(mid[i]));
        }
#pragma unroll
        for (int t = 0; t < DT; ++t) {
          const fa_bf16x8 va = flash_v_operand<STRV>(vs, kt, 32 * t, lane);
          o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, __builtin_bit_cast(fa_bf16x8, hi), o[t], 0, 0, 0);
          o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, __builtin_bit_cast(fa_bf16x8, mid), o[t], 0, 0, 0);
          o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, __builtin_bit_cast(fa_bf16x8, lo), o[t], 0, 0, 0);
        }
      }
    }
  }

  // The waves' states (the V stages are dead: a wave's records lie in its own), combined by all four: wave w
  // takes every fourth run of 4 output columns. A sum's sign bit says that its wave has met a value that is not
  // finite.
  const bool special = __any(odd);
  wave_lds_order();
  float* rec = reinterpret_cast<float*>(lds[wave]);
  rec[lane] = run_max;
  rec[64 + lane] = __uint_as_float((__float_as_uint(run_sum) & 0x7FFFFFFFu) | (special ? 0x80000000u : 0u));
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) rec[(2 + 16 * t + e) * 64 + lane] = o[t][e];
  __syncthreads();
  float big = -INFINITY, sum = 0.f, factor[kGenAttnWaves];
  uint32_t any_special = 0u;
#pragma unroll
  for (int w = 0; w < kGenAttnWaves; ++w) big = fmaxf(big, reinterpret_cast<const float*>(lds[w])[lane]);
#pragma unroll
  for (int w = 0; w < kGenAttnWaves; ++w) {
    const float* other = reinterpret_cast<const float*>(lds[w]);
    factor[w] = other[lane] == -INFINITY ? 1.f : expf(other[lane] - big);
    // both halves' keys
    any_special |= __float_as_uint(other[64 + col]);
    const float l = fabsf(other[64 + col]) + fabsf(other[64 + 32 + col]);
    sum += l * factor[w];
  }
  if (__builtin_expect(__builtin_amdgcn_readfirstlane(any_special) >> 31, 0)) {  // (uniform)
    if (special) special_values(rec + 128, big);
    __syncthreads();
  }
  if (qi >= a.lq) return;
  const float inv = sum > 0.f ? 1.0f / sum : 0.f;
  const long long ob = ((long long)(b * a.heads + h) * a.lq + qi) * a.dv;
#pragma unroll
  for (int g = wave; g < 4 * DT; g += kGenAttnWaves) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 8 * g + 4 * half + i;
      if (d >= a.dv) continue;
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < kGenAttnWaves; ++w) {
        const float x = reinterpret_cast<const float*>(lds[w])[(2 + 4 * g + i) * 64 + lane];
        if (factor[w] != 0.f) v += x * factor[w];
      }
      // a row with no kept key (and one whose kept scores are all NaN or -inf) gives zeros
      store_float_type(a.out, a.out_dtype, ob + d, big == -INFINITY ? 0.f : sum != sum ? sum : v * inv);
    }
  }
}

}  // namespace aoto

#define AOTO_GENERIC_ATTENTION(TYPE, F32, D, LETTER, VEC)                                             \
  extern "C" __global__ __launch_bounds__(64 * aoto::kGenAttnWaves) void                              \
      aoto_generic_attention_##TYPE##_d##D##_##LETTER(aoto::AttnArgs a) {                             \
    aoto::generic_attention_body<F32, D, VEC>(a);                                                     \
  }
