// MFMA encode (norm -> rotate -> codebook search -> pack -> store) at head_dim 64, 128 and 256 for float16, bfloat16
// and float32 input, flat rows or scattered through a slot mapping (K and V of a step in one launch).
//
//   Y^T[j, row] = sum_i Pi[j, i] X^T[i, row]            v_mfma_f32_32x32x16_f16, operands as described in akv_frag.h
//
// A workgroup takes 32 rows at a time (64 at head_dim 64).  Its threads load the rows -- sixteen neighbouring elements each, so a
// wavefront covers whole rows -- reduce the squared norm over the lanes of a row, and leave the rows in LDS in operand
// order; wavefront w, which keeps the 32 x D slice of Pi for coordinates 32 w .. 32 w + 31 in registers, multiplies them
// in.  float16 input is exact in the operand, so the vector is not normalised first: y = (Pi x) / (|x| + 1e-10).
// bfloat16 rows are scaled by the power of two of their largest element and converted (exact for elements within 2^14
// of the largest); float32 rows are scaled the same way and split into two float16 terms (three products instead of two).
// A lane ends up with sixteen neighbouring coordinates of one row: it searches the codebook and packs eight, six or
// four bytes on its own.  LDS tiles are double-buffered: one barrier per tile, the next rows already requested.
//
// What bounds it (1,048,576 bfloat16 rows of 128 scattered into a 4-bit cache, 110 us = 3.1 TB/s): the SIMDs' issue slots --
// 290 vector instructions per wavefront and tile (96 of them the search), vector unit 58 % and matrix cores 24 % of the
// cycles; the LDS index unit is 36 % active.  Calls of serving size are a start-up (rows and matrix on their way, the
// cell table built meanwhile) and one or two tiles: 8,192 rows take 5.6-8 us where the general kernel below takes 19 (head_dim 64)
// and 70 us (head_dim 256).  Rows of head_dim 256 need 128 registers of matrix per lane: two wavefronts a SIMD,
// 131,072 rows 45 us = 1.9 TB/s.
#include "akv_frag.h"

#define ER_PSCALE AKV_FRAG_SCALE
template <int D> struct er_cfg {
  static constexpr int NT = D / 32;                       // tiles of 32 coordinates
  static constexpr int KS = D / 16;                       // k-steps
  static constexpr int RG = D == 64 ? 2 : 1;              // row groups of 32 a workgroup works on side by side
  static constexpr int WAVES = NT * RG;                   // 4, 4, 8
  static constexpr int THREADS = WAVES * 64;
  static constexpr int ROWS = 32 * RG;
  static constexpr int TPR = D / 16;                      // threads per row while loading
  static constexpr int PITCH = D * 2 + 16;                // bytes of a row in LDS (16 more: eight rows meet all banks)
  static_assert(THREADS / TPR == ROWS, "every thread loads sixteen elements of one row");
};
// LDS: cell table | per-wavefront flags | per parity: squared norms and scales | destinations of three tiles | per parity:
// packed pieces | rows (hi, and lo for float32)
#define ER_TAB 0
#define ER_FLAG (AKV_CELLS * 8)
#define ER_NORM (ER_FLAG + 64)
template <int D> constexpr int er_dst_off() { return ER_NORM + 2 * er_cfg<D>::ROWS * 8; }
template <int D> constexpr int er_out_off() { return er_dst_off<D>() + 3 * er_cfg<D>::ROWS * 8; }
template <int D> constexpr int er_row_off() { return er_out_off<D>() + 2 * er_cfg<D>::ROWS * er_cfg<D>::TPR * 8; }
template <int D, int XDT> constexpr int er_lds_bytes() {
  return er_row_off<D>() + 2 * (XDT == AKV_F32 ? 2 : 1) * er_cfg<D>::ROWS * er_cfg<D>::PITCH;
}

// ----------------------------------------------------------------------------------
// fragment tables of the prepared-rotation buffer
// ----------------------------------------------------------------------------------
// one thread per (tile, k-step, lane): eight entries of Pi (fwd) and of Pi^T (inv), hi and lo
__global__ __launch_bounds__(256) void akv_frag_prepare_kernel(const float* __restrict__ Pi, int D, uint4* __restrict__ fwd, uint4* __restrict__ inv) {
  const int t = blockIdx.x * 256 + threadIdx.x;          // D/32 * D/16 * 64 threads
  const int ksn = D / 16;
  const int lane = t & 63, ks = (t >> 6) % ksn, tile = (t >> 6) / ksn;
  const int row = 32 * tile + akv_frag_coord(lane & 31), k0 = 16 * ks + 8 * (lane >> 5);
  const int half = D * D / 8;                            // uint4 entries of the hi table
#pragma unroll
  for (int which = 0; which < 2; ++which) {
    uint32_t hi[4] = {0, 0, 0, 0}, lo[4] = {0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float v = (which == 0 ? Pi[(size_t)row * D + k0 + e] : Pi[(size_t)(k0 + e) * D + row]) * ER_PSCALE;
      const __half h = __float2half_rn(v);
      const __half l = __float2half_rn(v - __half2float(h));
      hi[e >> 1] |= (uint32_t)__half_as_ushort(h) << (16 * (e & 1));
      lo[e >> 1] |= (uint32_t)__half_as_ushort(l) << (16 * (e & 1));
    }
    uint4* dst = which == 0 ? fwd : inv;
    dst[t] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    dst[half + t] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
  }
}

// flag word: 1 when some row of the matrix is longer than AKV_MAX_ROW_NORM (then a rotated unit vector may leave the
// range of the cell table and the kernel counts boundaries)
__global__ __launch_bounds__(256) void akv_frag_rownorm_kernel(const float* __restrict__ Pi, int D, uint32_t* __restrict__ flag) {
  __shared__ uint32_t bad;
  if (threadIdx.x == 0) bad = 0u;
  __syncthreads();
  if ((int)threadIdx.x < D) {
    float ss = 0.f;
    for (int i = 0; i < D; ++i) {
      const float v = Pi[(size_t)threadIdx.x * D + i];
      ss = fmaf(v, v, ss);
    }
    if (!(sqrtf(ss) <= AKV_MAX_ROW_NORM)) atomicOr(&bad, 1u);
  }
  __syncthreads();
  if (threadIdx.x == 0) flag[0] = bad;
}

int akv_prepare_frags(const float* rotation, int d, void* prep, hipStream_t stream) {
  if (!akv_frag_dim(d)) return AKV_OK;
  char* base = (char*)prep;
  akv_frag_prepare_kernel<<<d * d / 8 / 256, 256, 0, stream>>>(rotation, d, (uint4*)(base + akv_frag_fwd_offset(d)), (uint4*)(base + akv_frag_inv_offset(d)));
  AKV_LAUNCH_CHECK("akv_frag_prepare_kernel");
  akv_frag_rownorm_kernel<<<1, 256, 0, stream>>>(rotation, d, (uint32_t*)(base + akv_frag_flag_offset(d)));
  AKV_LAUNCH_CHECK("akv_frag_rownorm_kernel");
  return AKV_OK;
}

// ----------------------------------------------------------------------------------
// encode kernel
// ----------------------------------------------------------------------------------
typedef _Float16 er_half2 __attribute__((ext_vector_type(2)));
typedef unsigned short er_us2 __attribute__((ext_vector_type(2)));
typedef uint32_t er_u32x2 __attribute__((ext_vector_type(2)));

// maximum / sum over the N neighbouring lanes (a power of two up to sixteen) that hold one row
template <int N> __device__ __forceinline__ float er_row_sum(float v) {
  v += akv_lane_xor<1>(v);
  v += akv_lane_xor<2>(v);
  if constexpr (N >= 8) v += akv_lane_xor<4>(v);
  if constexpr (N >= 16) v += akv_lane_xor<8>(v);
  return v;
}
template <int N> __device__ __forceinline__ uint32_t er_row_max(uint32_t v) {
  v = max(v, akv_lane_xor_u32<1>(v));
  v = max(v, akv_lane_xor_u32<2>(v));
  if constexpr (N >= 8) v = max(v, akv_lane_xor_u32<4>(v));
  if constexpr (N >= 16) v = max(v, akv_lane_xor_u32<8>(v));
  return v;
}
// orders LDS traffic only: rows requested ahead keep flying
__device__ __forceinline__ void er_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int D, int BITS, int XDT, bool PAGED>
__global__ __launch_bounds__(er_cfg<D>::THREADS, D == 256 ? 2 : D == 128 ? 3 : 4) void akv_encode_rows_kernel(
    akv_gen_args a, const uint4* __restrict__ frag, const uint32_t* __restrict__ flag, uint32_t heads_rcp, uint32_t block_rcp) {
  typedef er_cfg<D> cfg;
  constexpr int KS = cfg::KS, ROWS = cfg::ROWS, TPR = cfg::TPR, PITCH = cfg::PITCH;
  constexpr int NA = XDT == AKV_F32 ? 2 : 1;              // float16 terms of the rows
  constexpr int NP = 2 * NA;                              // 16-byte pieces a thread loads
  constexpr int XB = XDT == AKV_F32 ? 4 : 2;
  constexpr int NB = (1 << BITS) - 1;
  constexpr int TILE_BYTES = ROWS * PITCH;
  extern __shared__ __align__(16) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile32 = wave % cfg::NT, rgroup = wave / cfg::NT;
  float2* norm2 = (float2*)(lds + ER_NORM);               // [parity][ROWS] squared norm (NaN: a row that is not finite), power of two taken out
  int64_t* dst = (int64_t*)(lds + er_dst_off<D>());       // [tile % 3][ROWS] address of the packed row, 0 = skip

  // a second tensor's rows follow the first's in tiles of their own: which tensor a tile belongs to is uniform
  const uint32_t n = (uint32_t)a.n;
  const uint32_t tiles_one = (n + ROWS - 1) / ROWS;
  const uint32_t ntiles = (PAGED && a.x2) ? 2u * tiles_one : tiles_one;

  // quotient by a divisor whose reciprocal ceil(2^32 / d) is at hand: at most one too large (d = 1: no reciprocal)
  auto divide = [](uint32_t v, uint32_t d, uint32_t rcp, uint32_t& rest) {
    uint32_t q = d == 1u ? v : __umulhi(v, rcp);
    rest = v - q * d;
    if ((int32_t)rest < 0) { rest += d; --q; }
    return q;
  };

  // ---- a thread's part of the rows: 16 elements.  Which rows go where is one wavefront's job per tile, in turn: its
  // lane l resolves row l (the other wavefronts skip the code), and stores the row's norm.
  const int lrow = tid / TPR, part = tid % TPR;
  typedef uint4 rows_t[NP];
  int64_t slot = -1;
  float* norm_at = nullptr;
  auto fetch = [&](rows_t& R, uint32_t tile, bool on_duty) __attribute__((always_inline)) {
    // (tiles and rows past the end repeat the last one, so that the loads are issued on every path)
    tile = min(tile, ntiles - 1);
    const bool second = PAGED && tile >= tiles_one;
    const uint32_t row0 = (second ? tile - tiles_one : tile) * ROWS;
    const char* xb = (const char*)(second ? a.x2 : a.x);
    const uint32_t m = min(row0 + lrow, n - 1);
    uint64_t off;
    if constexpr (PAGED) {
      uint32_t head;
      const uint32_t tok = divide(m, (uint32_t)a.heads, heads_rcp, head);
      off = (uint64_t)tok * (uint32_t)a.xs0 + (uint64_t)head * (uint32_t)a.xs1;
    } else {
      off = (uint64_t)m * (uint32_t)a.xs0;
    }
    const uint4* p = (const uint4*)(xb + XB * (off + 16 * part));
#pragma unroll
    for (int i = 0; i < NP; ++i) R[i] = p[i];
    if constexpr (PAGED) {
      if (on_duty) {
        uint32_t head;
        const uint32_t tok = divide(min(row0 + lane, n - 1), (uint32_t)a.heads, heads_rcp, head);
        slot = akv_load_index(a.slots, a.slot_itype, tok);
      }
    }
  };
  // address of row `lane` of the tile and of its norm
  auto resolve = [&](uint32_t tile, int third) {
    const bool second = PAGED && tile >= tiles_one;
    const uint32_t m = (second ? tile - tiles_one : tile) * ROWS + lane;
    uint8_t* pb = second ? a.packed2 : a.packed;
    float* nb = second ? a.norms2 : a.norms;
    int64_t dp = 0;
    norm_at = nullptr;
    if (lane < ROWS && m < n) {
      if constexpr (PAGED) {
        if (slot >= 0) {
          uint32_t head, pos;
          divide(m, (uint32_t)a.heads, heads_rcp, head);
          int64_t blk;
          if (slot < ((int64_t)1 << 31)) {      // (a 64-bit division is a hundred instructions)
            blk = divide((uint32_t)slot, (uint32_t)a.block_size, block_rcp, pos);
          } else {
            blk = slot / a.block_size;
            pos = (uint32_t)(slot - blk * a.block_size);
          }
          if (blk < a.max_blocks) {
            dp = (int64_t)(uintptr_t)(pb + blk * a.ps0 + (uint64_t)pos * (uint32_t)a.ps1 + (uint64_t)head * (uint32_t)a.ps2);
            norm_at = nb + blk * a.ns0 + (uint64_t)pos * (uint32_t)a.ns1 + (uint64_t)head * (uint32_t)a.ns2;
          }
        }
      } else {
        dp = (int64_t)(uintptr_t)(pb + (uint64_t)m * (uint32_t)a.ps0);
        norm_at = nb + m;
      }
    }
    if (lane < ROWS) dst[third * ROWS + lane] = dp;
  };

  // ---- cell table: its boundaries are requested before anything else, so that it is built while the rows and the
  // matrix are on their way
  float bnd[NB];
#pragma unroll
  for (int k = 0; k < NB; ++k) bnd[k] = a.table[k];
  const bool long_rows = flag[0] != 0u;
  // rows are requested two tiles ahead: a tile takes a workgroup less time than a trip to memory
  rows_t Ra, Rb;
  fetch(Ra, blockIdx.x, wave == 0);
  fetch(Rb, blockIdx.x + gridDim.x, wave == 1);
  // ---- the wavefront's slice of Pi
  akv_h8 Ah[KS], Al[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    Ah[ks] = akv_as_h8(frag[(tile32 * KS + ks) * 64 + lane]);
    Al[ks] = akv_as_h8(frag[D * D / 8 + (tile32 * KS + ks) * 64 + lane]);
  }
  __builtin_amdgcn_sched_barrier(0);
  {
    // the table serves finite, strictly increasing boundaries inside (-1, 1), at most one to a cell
    bool bad = long_rows || !(fabsf(bnd[0]) < 1.f && fabsf(bnd[NB - 1]) < 1.f);
#pragma unroll
    for (int k = 1; k < NB; ++k) bad = bad || !(bnd[k] > bnd[k - 1]);
    for (int c = tid; c < AKV_CELLS; c += cfg::THREADS) {
      uint32_t base = 0, cnt = 0;
      float inside = INFINITY;
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        const uint32_t cb = akv_cell(bnd[k]);
        base += cb < 8u * c ? 1u : 0u;
        if (cb == 8u * c) { ++cnt; inside = bnd[k]; }
      }
      uint32_t* lut = (uint32_t*)(lds + ER_TAB);
      lut[2 * c] = base;
      lut[2 * c + 1] = __float_as_uint(inside);
      bad = bad || cnt > 1;
    }
    if (lane == 0) ((uint32_t*)(lds + ER_FLAG))[wave] = 0u;
    if (bad) ((uint32_t*)(lds + ER_FLAG))[wave] = 1u;
  }
  er_barrier();
  bool linear = false;
#pragma unroll
  for (int w = 0; w < cfg::WAVES; ++w) linear = linear || ((const uint32_t*)(lds + ER_FLAG))[w] != 0u;
  linear = __builtin_amdgcn_readfirstlane(linear ? 1 : 0) != 0;
  // The matrix has arrived HERE: left open, the wait for it would sit in the loop, in front of the first product, as a
  // wait for every load in flight -- the rows requested for the next tile included.
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    asm volatile("" : "+v"(Ah[ks]));
    asm volatile("" : "+v"(Al[ks]));
  }

  // ---- norm, conversion, rows into LDS
  auto stage = [&](rows_t& R, uint32_t tile, int p, int third, bool on_duty) __attribute__((always_inline)) {
    float ss = 0.f;
    uint32_t unscale = 0x3f800000u;     // float bits of the power of two taken out of the row
    bool nonfinite = false;
    uint4 hi[2], lo[2];
    if constexpr (XDT == AKV_F16) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        union { uint4 u; er_half2 h2[4]; } cv;
        cv.u = R[i];
        hi[i] = R[i];
#pragma unroll
        for (int q = 0; q < 4; ++q) ss = __builtin_amdgcn_fdot2(cv.h2[q], cv.h2[q], ss, false);
      }
    } else if constexpr (XDT == AKV_BF16) {
      er_us2 mx2 = {0, 0};
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t w[4] = {R[i].x, R[i].y, R[i].z, R[i].w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          union { uint32_t u; er_us2 v; } mm;
          mm.u = w[q] & 0x7fff7fffu;
          mx2 = __builtin_elementwise_max(mx2, mm.v);
          const float l = __uint_as_float(w[q] << 16), h = __uint_as_float(w[q] & 0xffff0000u);
          ss = fmaf(l, l, ss);
          ss = fmaf(h, h, ss);
        }
      }
      uint32_t ef = er_row_max<TPR>(max((uint32_t)mx2[0], (uint32_t)mx2[1])) >> 7;      // exponent field of the largest element
      nonfinite = ef == 255u;
      if (ef == 0u || ef == 255u) ef = 127u;       // all (sub)zero, or not finite (flagged)
      if (ef == 254u) ef = 253u;                   // keep the scale a normal number
      const float sc = __uint_as_float((254u - ef) << 23);      // 2^(127 - ef)
      unscale = ef << 23;                                        // 2^(ef - 127)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t w[4] = {R[i].x, R[i].y, R[i].z, R[i].w};
        union { uint4 u; uint32_t w[4]; } cv;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          union { decltype(__builtin_amdgcn_cvt_pkrtz(0.f, 0.f)) h; uint32_t u; } pk;
          pk.h = __builtin_amdgcn_cvt_pkrtz(__uint_as_float(w[q] << 16) * sc, __uint_as_float(w[q] & 0xffff0000u) * sc);
          cv.w[q] = pk.u;
        }
        hi[i] = cv.u;
      }
    } else {
      // float32: the norm from the values themselves; hi keeps 11 bits, x - hi is exact in float32, so lo is off by at
      // most half a float32 ulp of the element (2^-25 of the largest element once lo is a float16 subnormal)
      uint32_t mx = 0u;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const uint32_t w[4] = {R[i].x, R[i].y, R[i].z, R[i].w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          mx = max(mx, w[q] & 0x7fffffffu);
          const float v = __uint_as_float(w[q]);
          ss = fmaf(v, v, ss);
        }
      }
      uint32_t ef = er_row_max<TPR>(mx) >> 23;
      nonfinite = ef == 255u;
      if (ef == 0u || ef == 255u) ef = 127u;
      if (ef == 254u) ef = 253u;
      const float sc = __uint_as_float((254u - ef) << 23);
      unscale = ef << 23;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        union { uint4 u; er_half2 h2[4]; } ch, cl;
        const uint32_t w[8] = {R[2 * i].x, R[2 * i].y, R[2 * i].z, R[2 * i].w, R[2 * i + NA - 1].x, R[2 * i + NA - 1].y, R[2 * i + NA - 1].z, R[2 * i + NA - 1].w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float x0 = __uint_as_float(w[2 * q]) * sc, x1 = __uint_as_float(w[2 * q + 1]) * sc;
          const _Float16 h0 = (_Float16)x0, h1 = (_Float16)x1;
          ch.h2[q] = (er_half2){h0, h1};
          cl.h2[q] = (er_half2){(_Float16)(x0 - (float)h0), (_Float16)(x1 - (float)h1)};
        }
        hi[i] = ch.u;
        lo[i] = cl.u;
      }
    }
    unsigned char* xr = lds + er_row_off<D>() + (p * NA) * TILE_BYTES + lrow * PITCH + 32 * part;
    *(uint4*)xr = hi[0];
    *(uint4*)(xr + 16) = hi[1];
    if constexpr (NA == 2) {
      *(uint4*)(xr + TILE_BYTES) = lo[0];
      *(uint4*)(xr + TILE_BYTES + 16) = lo[1];
    }
    ss = er_row_sum<TPR>(ss);
    // A vector with a NaN or an infinity rotates to NaN everywhere: every code is the last level.  (float16 squares
    // cannot overflow, so there an infinite sum means an infinite element; a finite bfloat16 or float32 row whose
    // squares overflow has norm inf, unit vector 0 and y = 0: its reciprocal is 0 and the scaled products are finite.)
    // The sign of the scale tells such a row apart (its squared norm is stored as it is: inf or NaN).
    const bool nan_row = XDT == AKV_F16 ? !(ss < INFINITY) : (nonfinite || ss != ss);
    if (part == 0) norm2[p * ROWS + lrow] = make_float2(ss, __uint_as_float(unscale | (nan_row ? 0x80000000u : 0u)));
    if (on_duty) resolve(tile, third);
  };

  // ---- rotate, search, pack, store: the lane's row, coordinates 32 tile32 + 16 (lane / 32) + 0..15
  const int crow = 32 * rgroup + (lane & 31), half = lane >> 5;
  auto compute = [&](int p, bool on_duty) __attribute__((always_inline)) {
    const unsigned char* xr = lds + er_row_off<D>() + (p * NA) * TILE_BYTES + crow * PITCH + 16 * half;
    const float2 nm = norm2[p * ROWS + crow];
    akv_f16v acc = akv_zero16();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const akv_h8 b = akv_as_h8(*(const uint4*)(xr + 32 * ks));
      acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(Ah[ks], b, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(Al[ks], b, acc, 0, 0, 0);
      if constexpr (NA == 2) {
        const akv_h8 bl = akv_as_h8(*(const uint4*)(xr + TILE_BYTES + 32 * ks));
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(Ah[ks], bl, acc, 0, 0, 0);
      }
    }
    if (on_duty) {
      const float ns = norm2[p * ROWS + (lane < ROWS ? lane : 0)].x;
      if (norm_at != nullptr) *norm_at = sqrtf(ns);
    }
    // 1 / (|x| + 1e-10) by the hardware's square root and reciprocal (one unit in the last place each, the same for
    // all coordinates of the row), the scales of the row and of the matrix put back
    const float r = __builtin_amdgcn_rcpf(__builtin_amdgcn_sqrtf(nm.x) + 1e-10f) * (1.f / ER_PSCALE) * fabsf(nm.y);
    // words of eight codes; a word is built by shift-and-add from its top code down (4-bit: bytes of two codes, first
    // byte lowest; 3-bit: a big-endian 24-bit word; 2-bit: sixteen codes are one dword of bytes of four codes)
    uint32_t w[2] = {0u, 0u};
    auto place = [&](int q, int kk) { return 8 * q + (BITS == 4 ? 6 - (kk & ~1) + (kk & 1) : BITS == 3 ? kk : 4 - (kk & 4) + (kk & 3)); };
    if (__builtin_expect(linear, 0)) {
      uint32_t code[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) { acc[k] *= r; code[k] = 0u; }
#pragma unroll 1
      for (int b = 0; b < NB; ++b) {
        const float bv = a.table[b];
#pragma unroll
        for (int k = 0; k < 16; ++k) code[k] += bv < acc[k] ? 1u : 0u;
      }
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) w[q] = (w[q] << BITS) + code[place(q, kk)];
    } else {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        er_u32x2 e[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          acc[8 * q + k] *= r;
          e[k] = *(const er_u32x2*)(lds + ER_TAB + akv_cell(acc[8 * q + k]));
        }
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
          const int k = place(q, kk);
          w[q] = (w[q] << BITS) + (e[k & 7].x + (__uint_as_float(e[k & 7].y) < acc[k] ? 1u : 0u));
        }
      }
    }
    if (nm.y < 0.f) { w[0] = 0xffffffffu; w[1] = 0xffffffffu; }      // a row that is not finite: last level everywhere
    *(er_u32x2*)(lds + er_out_off<D>() + ((p * ROWS + crow) * TPR + 2 * tile32 + half) * 8) = (er_u32x2){w[0], w[1]};
  };

  // ---- store a tile's packed rows, a tile late and in the order of the loads: the threads of a row write it whole
  // (straight from the lanes that pack them, a wavefront would write sixteen bytes of each of 32 rows)
  auto flush = [&](int p, int third) {
    const er_u32x2 w = *(const er_u32x2*)(lds + er_out_off<D>() + (p * ROWS * TPR + tid) * 8);
    const int64_t dp = dst[third * ROWS + lrow];
    if (dp != 0) {
      uint8_t* prow = (uint8_t*)(uintptr_t)dp + 2 * part * BITS;
      if constexpr (BITS == 4) {
        *(er_u32x2*)prow = w;
      } else if constexpr (BITS == 3) {
        // six bytes: the two big-endian 24-bit words one after the other
        *(uint16_t*)prow = (uint16_t)__builtin_amdgcn_perm(0u, w.x, 0x0c0c0102u);
        *(uint16_t*)(prow + 2) = (uint16_t)__builtin_amdgcn_perm(w.y, w.x, 0x0c0c0600u);
        *(uint16_t*)(prow + 4) = (uint16_t)__builtin_amdgcn_perm(0u, w.y, 0x0c0c0001u);
      } else {
        *(uint32_t*)prow = (w.x & 0xffffu) | (w.y << 16);
      }
    }
  };

  int duty = 0, third = 0, last = -1;      // last: the destinations of the tile before this one
  auto step = [&](rows_t& R, uint32_t t, const int p) __attribute__((always_inline)) {
    stage(R, t, p, third, wave == duty);
    fetch(R, t + 2 * gridDim.x, wave == (duty + 2) % cfg::WAVES);
    // One barrier per tile.  A wavefront that is ahead writes rows, norms and pieces of the other parity, and the third
    // set of destinations: every wavefront has passed the barrier after its last reads of those.
    er_barrier();
    if (last >= 0) flush(p ^ 1, last);
    compute(p, wave == duty);
    duty = (duty + 1) % cfg::WAVES;
    last = third;
    third = third == 2 ? 0 : third + 1;
  };
  int p = 0;
  for (uint32_t t = blockIdx.x;;) {
    step(Ra, t, 0);
    p = 0;
    t += gridDim.x;
    if (t >= ntiles) break;
    step(Rb, t, 1);
    p = 1;
    t += gridDim.x;
    if (t >= ntiles) break;
  }
  er_barrier();
  flush(p, last);
}

static bool er_disabled() {
  static int v = -1;
  if (v < 0) {
    const char* e = getenv("AKV_DISABLE_MFMA");
    v = (e && e[0] == '1') ? 1 : 0;
  }
  return v == 1;
}

template <int D, int BITS, int XDT, bool PAGED>
static int er_launch(const akv_gen_args& a, const uint4* frag, const uint32_t* flag, hipStream_t stream) {
  constexpr int LDS = er_lds_bytes<D, XDT>();
  const int cus = akv_cached_cu_count();
  const int64_t tiles = (a.n + er_cfg<D>::ROWS - 1) / er_cfg<D>::ROWS * (PAGED && a.x2 ? 2 : 1);
  const int64_t most = (int64_t)(cus > 0 ? cus : 256) * (D == 256 ? 1 : D == 128 ? 3 : 4);
  const int grid = (int)(tiles < most ? tiles : most);
  static bool configured = false;
  if (!configured) {
    AKV_HIP(hipFuncSetAttribute((const void*)akv_encode_rows_kernel<D, BITS, XDT, PAGED>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
    configured = true;
  }
  auto rcp = [](int d) { return d <= 1 ? 0u : (uint32_t)((((uint64_t)1 << 32) + d - 1) / (uint64_t)d); };
  AKV_LAUNCH_TIMED((akv_encode_rows_kernel<D, BITS, XDT, PAGED>), grid, er_cfg<D>::THREADS, LDS, stream, a, frag, flag, rcp(a.heads), rcp(a.block_size));
  AKV_LAUNCH_CHECK("akv_encode_rows_kernel");
  return AKV_OK;
}

template <int D, int BITS, int XDT>
static int er_launch_paged(bool paged, const akv_gen_args& a, const uint4* frag, const uint32_t* flag, hipStream_t stream) {
  return paged ? er_launch<D, BITS, XDT, true>(a, frag, flag, stream) : er_launch<D, BITS, XDT, false>(a, frag, flag, stream);
}
template <int D, int BITS>
static int er_launch_dt(int x_dtype, bool paged, const akv_gen_args& a, const uint4* frag, const uint32_t* flag, hipStream_t stream) {
  if (x_dtype == AKV_F16) return er_launch_paged<D, BITS, AKV_F16>(paged, a, frag, flag, stream);
  if (x_dtype == AKV_BF16) return er_launch_paged<D, BITS, AKV_BF16>(paged, a, frag, flag, stream);
  return er_launch_paged<D, BITS, AKV_F32>(paged, a, frag, flag, stream);
}

// returns AKV_ERR_UNSUPPORTED for head sizes and layouts the kernel does not take (the caller then uses the general kernel)
int akv_encode_rows_try(const akv_gen_args& a, bool paged, int x_dtype, int d, int bits, const void* rot_prep, hipStream_t stream) {
  if (er_disabled() || !akv_frag_dim(d) || bits < 2 || bits > 4) return AKV_ERR_UNSUPPORTED;
  // 16-byte loads of the input rows; stores of 8 / 2 x 3 / 4 bytes into the packed rows
  const int64_t xmask = x_dtype == AKV_F32 ? 3 : 7;        // elements per 16 bytes, minus one
  if (((uintptr_t)a.x & 15) || ((uintptr_t)a.x2 & 15) || (a.xs0 & xmask) || (paged && (a.xs1 & xmask))) return AKV_ERR_UNSUPPORTED;
  const uintptr_t pmask = bits == 3 ? 1 : 3;
  if (((uintptr_t)a.packed | (uintptr_t)a.packed2 | (uintptr_t)a.ps0 | (uintptr_t)a.ps1 | (uintptr_t)a.ps2) & pmask) return AKV_ERR_UNSUPPORTED;
  // row numbers are 32-bit, steps past the end included (and what the reciprocals divide stays below 2^31); so are the
  // strides inside a block and of the input
  if (a.n >= ((int64_t)1 << 29)) return AKV_ERR_UNSUPPORTED;
  const int64_t strides[7] = {a.xs0, paged ? a.xs1 : 0, paged ? 0 : a.ps0, a.ps1, a.ps2, a.ns1, a.ns2};
  for (int i = 0; i < 7; ++i)
    if (strides[i] < 0 || strides[i] >= ((int64_t)1 << 31)) return AKV_ERR_UNSUPPORTED;
  const uint4* frag = (const uint4*)((const char*)rot_prep + akv_frag_fwd_offset(d));
  const uint32_t* flag = (const uint32_t*)((const char*)rot_prep + akv_frag_flag_offset(d));
#define ER_CASE(DD, BB) if (d == DD && bits == BB) return er_launch_dt<DD, BB>(x_dtype, paged, a, frag, flag, stream);
  ER_CASE(64, 2) ER_CASE(64, 3) ER_CASE(64, 4)
  ER_CASE(128, 2) ER_CASE(128, 3) ER_CASE(128, 4)
  ER_CASE(256, 2) ER_CASE(256, 3) ER_CASE(256, 4)
#undef ER_CASE
  return AKV_ERR_UNSUPPORTED;
}
