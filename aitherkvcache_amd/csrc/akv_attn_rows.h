// Rotations of many rows on the matrix cores: queries of the prologues, outputs of the reduce.
//
//   Y[n, row] = sum_k M[n, k] X[row, k]           v_mfma_f32_16x16x32_f16
//
// A wavefront keeps sixteen rows of the matrix (outputs) in registers, split into float16 terms at its start, and multiplies
// sixteen rows of X at a time, which lie in LDS as float16 terms.  Lane (row, g) ends up with four neighbouring outputs
// 4 g .. 4 g + 3 of its row: what is stored next is eight or sixteen bytes.
//
// Precision: a row is scaled by a power of two (the largest element to [2^5, 2^6)), the matrix by its prepared one, all terms are
// rounded to nearest, sums are float32.  Queries: three terms of the float32 matrix against one of float16 and bfloat16 queries, which
// hold them exactly (down to 2^-30 of the largest), or three of float32 ones, products down to 2^-24: at head_dim 64, 128 and 256
// the mean error of a float32 attention output of 300 tokens is 3.7, 4.4 and 5.4e-7; float32 multiply-adds gave 3.8, 4.8 and 5.7,
// three products of two terms each 4.2, 5.0 and 6.2.  (A step of 24 sequences, 16 heads on 4 of 256, takes 0.6 us longer than with
// those.)  The reduce at head_dim 256 keeps to two terms: outputs of a single token are at 2.1e-7, 2.2 with multiply-adds.
#pragma once
#include "akv_attn_common.h"

#define AR_M_SCALE 1024.f

typedef _Float16 ar_half8 __attribute__((ext_vector_type(8)));
typedef _Float16 ar_half4 __attribute__((ext_vector_type(4)));
typedef float ar_float4 __attribute__((ext_vector_type(4)));

template <int D, int TERMS> struct ar_rows {
  static constexpr int KS = D / 32, PITCH = D + 8;      // (sixteen bytes more: eight rows meet all banks)
  _Float16 term[TERMS][16][PITCH];
  float unscale[16];                                    // of a row
};

#define AR_THIRD 4096.f        // third terms are kept this much larger: they are no subnormals then
// sixteen rows of a matrix: lane (m, g) holds row m, elements 32 ks + 8 g + e
template <int D> struct ar_matrix {
  ar_half8 term[3][D / 32];
  __device__ __forceinline__ void load(const float* __restrict__ m, float scale) {
    const int lane = threadIdx.x & 63;
    const float4* p = (const float4*)(m + (size_t)(lane & 15) * D + 8 * (lane >> 4));
    float4 v[D / 16];
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) {
      v[2 * ks] = p[8 * ks];
      v[2 * ks + 1] = p[8 * ks + 1];
    }
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) {
      const float x[8] = {v[2 * ks].x, v[2 * ks].y, v[2 * ks].z, v[2 * ks].w, v[2 * ks + 1].x, v[2 * ks + 1].y, v[2 * ks + 1].z, v[2 * ks + 1].w};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float s = x[e] * scale;
        term[0][ks][e] = (_Float16)s;
        const float r = s - (float)term[0][ks][e];
        term[1][ks][e] = (_Float16)r;
        term[2][ks][e] = (_Float16)((r - (float)term[1][ks][e]) * AR_THIRD);
      }
    }
  }
  template <int TERMS> __device__ __forceinline__ ar_float4 times(const ar_rows<D, TERMS>& rows) const {
    const int lane = threadIdx.x & 63, row = lane & 15, g = lane >> 4;
    ar_float4 first = {0.f, 0.f, 0.f, 0.f}, second = first, third = first;
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) {
      ar_half8 x[TERMS];
#pragma unroll
      for (int i = 0; i < TERMS; ++i) x[i] = *(const ar_half8*)&rows.term[i][row][32 * ks + 8 * g];
      first = __builtin_amdgcn_mfma_f32_16x16x32_f16(term[0][ks], x[0], first, 0, 0, 0);
      second = __builtin_amdgcn_mfma_f32_16x16x32_f16(term[1][ks], x[0], second, 0, 0, 0);
      third = __builtin_amdgcn_mfma_f32_16x16x32_f16(term[2][ks], x[0], third, 0, 0, 0);
      if constexpr (TERMS == 3) {
        second = __builtin_amdgcn_mfma_f32_16x16x32_f16(term[0][ks], x[1], second, 0, 0, 0);
        second = __builtin_amdgcn_mfma_f32_16x16x32_f16(term[1][ks], x[1], second, 0, 0, 0);
        third = __builtin_amdgcn_mfma_f32_16x16x32_f16(term[0][ks], x[2], third, 0, 0, 0);
      }
    }
    return first + (second + third * (1.f / AR_THIRD));
  }
};
// scale of a row whose largest magnitude is m, and what undoes it (and AR_M_SCALE)
__device__ __forceinline__ float ar_scale(float m, float& unscale) {
  const uint32_t e = akv_row_exponent(m), up = min(254u - e + 5u, 253u);
  unscale = __uint_as_float((254u - up) << 23) * (1.f / AR_M_SCALE);
  return __uint_as_float(up << 23);
}

// ----------------------------------------------------------------------------------
// terms of a query: float16 and bfloat16 fit one
template <int QDT> constexpr int ar_terms() { return QDT == AKV_F32 ? 3 : 1; }
// Query rows into the operand of a main kernel, by workgroup b of nb (a multiple of D / 64) of 256 threads: b % (D / 64) is its
// slice of 64 outputs, b / (D / 64) its first tile of sixteen rows.  A tile holds 16 / `slots` (sequence, kv head) items of up to
// `slots` query heads (4 or 8; the rest of a tile's rows are zero: columns of the operand that no head has but a main kernel
// looks at).
//   FULL: [item][8 steps][64 lanes] uint4, each pair of coordinates twice (it faces both terms of the keys), the scale
//   `qscale` in it; else [item][D / 16 steps][64 lanes] uint2 and `fac` = the row's scale times qscale.
// Lane (column, quarter) of a step: column q the rounding of query head q's coordinates, 8 + q their remainder.
// ----------------------------------------------------------------------------------
template <int D, int QDT, bool FULL>
__device__ __forceinline__ void ar_rotate_queries(ar_rows<D, ar_terms<QDT>()>& rows, int b, int nb, const void* __restrict__ query, int64_t qs_seq, int64_t qs_head,
                                                  const float* __restrict__ Pi, const akv_prep_scale* __restrict__ scale, int S, int QH, int KVH,
                                                  int slots, void* __restrict__ qop, float* __restrict__ fac, float qscale, int bits) {
  constexpr int NS = D / 64, EPT = D / 16;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int gqa = QH / KVH, nq = S * KVH, per = 16 / slots, tiles = (nq + per - 1) / per;
  const int slice = b % NS, n0 = 64 * slice + 16 * wave;
  const int row = tid >> 4, part = tid & 15;
  float x[EPT];
  auto fetch = [&](int tile) {
    const int item = tile * per + row / slots, q = row % slots;
    const bool held = item < nq && q < gqa;
    const int64_t at = held ? (int64_t)(item / KVH) * qs_seq + (int64_t)(item % KVH * gqa + q) * qs_head : 0;
#pragma unroll
    for (int i = 0; i < EPT; ++i) x[i] = held ? akv_elem<QDT>::load(query, at + 64 * (i >> 2) + 4 * part + (i & 3)) : 0.f;
  };
  int tile = b / NS;
  if (tile >= tiles) return;
  fetch(tile);
  ar_matrix<D> m;
  m.load(Pi + (size_t)n0 * D, AR_M_SCALE * scale->down);
  const float up = scale->up;
  for (; tile < tiles; tile += nb / NS) {
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < EPT; ++i) mx = fmaxf(mx, fabsf(x[i]));
    mx = fmaxf(mx, akv_lane_xor<1>(mx)); mx = fmaxf(mx, akv_lane_xor<2>(mx));
    mx = fmaxf(mx, akv_lane_xor<4>(mx)); mx = fmaxf(mx, akv_lane_xor<8>(mx));
    float un;
    const float sc = ar_scale(mx, un);
    un *= up;
#pragma unroll
    for (int i = 0; i < EPT; i += 4) {
      constexpr int TERMS = ar_terms<QDT>();
      ar_half4 t[TERMS];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float s = x[i + e] * sc;
#pragma unroll
        for (int j = 0; j < TERMS; ++j) {
          t[j][e] = (_Float16)(j == 2 ? s * AR_THIRD : s);
          s -= (float)t[j][e];
        }
      }
#pragma unroll
      for (int j = 0; j < TERMS; ++j) *(ar_half4*)&rows.term[j][row][16 * i + 4 * part] = t[j];
    }
    const int item = tile * per + row / slots, q = row % slots;
    if (part == 0) {
      rows.unscale[row] = un;
      if (!FULL && slice == 0 && item < nq && q < gqa) fac[(size_t)(item / KVH) * QH + item % KVH * gqa + q] = un * AR_M_SCALE * qscale;
    }
    if (tile + nb / NS < tiles) fetch(tile + nb / NS);
    __syncthreads();
    const ar_float4 y = m.times(rows);
    {
      const int r = lane & 15, g = lane >> 4, it = tile * per + r / slots, col = r % slots;
      const float f = FULL ? rows.unscale[r] * qscale : 1.f / AR_M_SCALE;
      float v[4] = {y[0] * f, y[1] * f, y[2] * f, y[3] * f};
      // (one rounding for both terms: left to itself the compiler takes a term from the product before it is rounded, and where
      // that decides a tie the remainder belongs to another rounding)
#pragma unroll
      for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(v[e]));
      // (2-bit codes are looked up as (0, 2) and (1, 3) by the kernels of independent wavefronts)
      if (!FULL && bits == 2) { const float t = v[1]; v[1] = v[2]; v[2] = t; }
      union { ar_half4 h; uint2 u; } hi, lo;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        hi.h[e] = (_Float16)v[e];
        lo.h[e] = (_Float16)(v[e] - (float)hi.h[e]);
      }
      const int c0 = n0 + 4 * g, at = (c0 % (D / 4) / 4) * 64 + 16 * (c0 / (D / 4)) + col;
      if (it < nq) {
        if constexpr (FULL) {
          uint4* dst = (uint4*)qop + (size_t)it * (D / 16 * 64) + at;
          dst[0] = make_uint4(hi.u.x, hi.u.x, hi.u.y, hi.u.y);
          dst[8] = make_uint4(lo.u.x, lo.u.x, lo.u.y, lo.u.y);
        } else {
          uint2* dst = (uint2*)qop + (size_t)it * (D / 16 * 64) + at;
          dst[0] = hi.u;
          dst[8] = lo.u;
        }
      }
    }
    __syncthreads();      // (the next tile's rows go where these are)
  }
}
// workgroups for it: `most` at the same time at most
static inline int ar_query_blocks(int d, int S, int KVH, int slots, int most) {
  const int64_t per = 16 / slots, ns = d / 64, tiles = ((int64_t)S * KVH + per - 1) / per, cap = most / ns > 0 ? most / ns : 1;
  return (int)((tiles < cap ? tiles : cap) * ns);
}
