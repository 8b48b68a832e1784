// MFMA encode (norm -> rotate -> codebook search -> pack -> store) for float16, bfloat16 and float32
// input at head_dim 128.
//
// The rotation is the only heavy arithmetic of the encode path (128 x 128 multiply-adds per
// vector), so it runs on the matrix cores; everything else is arranged so that the matrix-core
// register layouts are also the memory layouts:
//
//   Y[v, j] = sum_i X[v, i] * Pi[j, i]                     v_mfma_f32_16x16x32_f16
//     A = X: lane (row = l%16, g = l/16) holds, for k-step ks, elements i = 32g + 8ks + e (e<8)
//         of vector `row` -- 64 contiguous bytes of the input row, loaded by four 16-byte loads
//         that ARE the four A operands (measured faster than the layout in which the four lanes
//         of a row share each load).  float16 input is exact in the operand, so the vector is
//         not normalised before the product: y = (sum_i Pi[j,i] x_i) * 1/(|x| + 1e-10), with one
//         correctly rounded reciprocal per vector.  float32 input is scaled by the power of two of the
//         row's largest element and split into two float16 terms (hi + lo: every element to half a
//         float32 ulp of itself, or to 2^-25 of the largest element where lo is subnormal); the product
//         takes three MFMAs per tile (x_hi Pi_hi + x_hi Pi_lo + x_lo Pi_hi) and a wavefront step
//         holds one M-tile instead of two, so that both terms of the rows fit the registers.
//     B = Pi: float32 entries split into two float16 terms (hi + lo, scaled by 64 to stay clear
//         of float16 subnormals), i.e. two MFMAs per tile and ~22 bits of the matrix.  N-tile nt,
//         column col is output coordinate j = 8 col + nt.
//     D: lane (col, g) holds rows 4g..4g+3; over the eight N-tiles it collects outputs
//         8col..8col+7 of a vector: one dword of a 4-bit row, three bytes of a 3-bit row, one
//         halfword of a 2-bit row -- sixteen lanes write one packed row contiguously.
//
// Codebook search: code = #{b < y}.  A table of EM_CELLS uniform cells over y in (-1.004, 1.004)
// maps cell -> (number of boundaries in lower cells, the one boundary inside the cell or +inf);
// the cell index is a monotone function of y evaluated by the same instructions for y and, when
// the table is built, for the boundaries, so base + (boundary < y) is exact for every float in
// range.  |y| <= (longest row of Pi) x |unit vector|, and the prepare step records whether every
// row is short enough; if not, or if two boundaries share a cell or lie outside (-1, 1) (no such
// codebook is produced by the library), the kernel counts all boundaries instead.
//
// (Above: the kernel of the larger calls.  Calls of one or two steps a CU keep the matrix in registers: akv_encode_rows_kernel.)
//
// A wavefront encodes EM_ROWS vectors per step (its M-tiles share every B operand read from LDS);
// a workgroup is EM_WAVES independent wavefronts plus the B operand (64 KB) and the cell table.
// Vector-unit and matrix-core time add up on a SIMD here (measured), so the search is kept to six
// vector instructions per value: multiply, fma, mask, compare, add-with-carry, shift-or.
#include "akv_common.h"
#include <type_traits>

typedef _Float16 em_half8 __attribute__((ext_vector_type(8)));
typedef _Float16 em_half2 __attribute__((ext_vector_type(2)));
typedef float em_float4 __attribute__((ext_vector_type(4)));
typedef unsigned short em_us2 __attribute__((ext_vector_type(2)));

#ifndef EM_MT
#define EM_MT 2                    // M-tiles (16 vectors each) per wavefront step
#endif
#define EM_WAVES (32 / EM_MT)      // EM_MT 2: sixteen wavefronts under 128 registers; 4: eight under 256
#define EM_THREADS (EM_WAVES * 64)
#define EM_ROWS (16 * EM_MT)       // vectors per wavefront step
#define EM_CELLS 512               // uniform cells over y in [-1.0039, 1.0039)
#define EM_CELL_S 2040.f           // 8 x cells per unit of y: the cell table is addressed in bytes
#define EM_CELL_C (8388608.f + 2048.f)   // 2^23 + centre: the sum's mantissa is 8 x the cell coordinate
#define EM_CELL_MASK 0xff8u
#define EM_MAX_ROW_NORM 1.0015f    // |y| <= |row of Pi| <= this keeps y inside the table
#define EM_PSCALE 64.f             // scale of the matrix operand
#define EM_B_BYTES 65536           // [hi/lo][8 nt][4 ks][64 lanes] x 16 B
#define EM_LUT_OFF 0               // EM_CELLS x {uint32 base, float boundary}: LDS address = cell byte offset
#define EM_B_OFF (EM_CELLS * 8)
#define EM_PAR_OFF (EM_B_OFF + EM_B_BYTES)       // uint32 bad, pad
#define EM_BND_OFF (EM_PAR_OFF + 16)              // 16 floats: boundaries (fallback search)
#define EM_WAVE_OFF (EM_BND_OFF + 64)
#define EM_WAVE_BYTES (EM_ROWS * (8 + 8 + 8 + 4))  // src offset, packed offset, norm offset, 1/(|x|+eps)
#define EM_LDS_BYTES (EM_WAVE_OFF + EM_WAVES * EM_WAVE_BYTES)

// ----------------------------------------------------------------------------------
// B operand: prep + 2*d*d floats (the reserved half of the prepared-rotation buffer)
// ----------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void akv_em_prepare_kernel(const float* __restrict__ Pi, uint4* __restrict__ bop) {
  // one thread per (nt, ks, lane): 8 entries, hi and lo
  const int t = blockIdx.x * 256 + threadIdx.x;      // 8*4*64 = 2048 threads
  const int lane = t & 63, ks = (t >> 6) & 3, nt = t >> 8;
  const int col = lane & 15, g = lane >> 4;
  const int j = 8 * col + nt;
  uint32_t hi[4], lo[4];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float v = Pi[(size_t)j * 128 + 32 * g + 8 * ks + e] * EM_PSCALE;
    const __half h = __float2half_rn(v);
    const __half l = __float2half_rn(v - __half2float(h));
    if (e & 1) {
      hi[e >> 1] |= (uint32_t)__half_as_ushort(h) << 16;
      lo[e >> 1] |= (uint32_t)__half_as_ushort(l) << 16;
    } else {
      hi[e >> 1] = __half_as_ushort(h);
      lo[e >> 1] = __half_as_ushort(l);
    }
  }
  bop[t] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
  bop[2048 + t] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
}

// flag word after the B operand: 1 when some row of the matrix is longer than EM_MAX_ROW_NORM (then
// a rotated unit vector may leave the range of the cell table and the kernel counts boundaries)
__global__ __launch_bounds__(128) void akv_em_rownorm_kernel(const float* __restrict__ Pi, uint32_t* __restrict__ flag) {
  __shared__ uint32_t bad;
  if (threadIdx.x == 0) bad = 0u;
  __syncthreads();
  float ss = 0.f;
  for (int i = 0; i < 128; ++i) {
    const float v = Pi[(size_t)threadIdx.x * 128 + i];
    ss = fmaf(v, v, ss);
  }
  if (!(sqrtf(ss) <= EM_MAX_ROW_NORM)) atomicOr(&bad, 1u);
  __syncthreads();
  if (threadIdx.x == 0) flag[0] = bad;
}

int akv_prepare_rotation_mfma(const float* rotation, int d, void* prep, hipStream_t stream) {
  if (d != 128) return AKV_OK;
  uint4* bop = (uint4*)((float*)prep + (size_t)2 * d * d);
  akv_em_prepare_kernel<<<8, 256, 0, stream>>>(rotation, bop);
  AKV_LAUNCH_CHECK("akv_em_prepare_kernel");
  akv_em_rownorm_kernel<<<1, 128, 0, stream>>>(rotation, (uint32_t*)(bop + EM_B_BYTES / 16));
  AKV_LAUNCH_CHECK("akv_em_rownorm_kernel");
  return AKV_OK;
}

// ----------------------------------------------------------------------------------
// encode kernel
// ----------------------------------------------------------------------------------
typedef uint32_t em_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t em_u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) em_u32x4 em_lds_u128;
typedef __attribute__((address_space(3))) em_u32x2 em_lds_u64;

// Byte offset of the cell of y in the table: y * S + (2^23 + centre) has the cell coordinate (x 8)
// in its mantissa, so one fused multiply-add and one mask replace scale, clamp, convert and shift.
// Monotone non-decreasing for |y| < 1.0039; NaN lands inside the table like any other pattern.
__device__ __forceinline__ uint32_t em_cell(float y) {
  return __float_as_uint(fmaf(y, EM_CELL_S, EM_CELL_C)) & EM_CELL_MASK;
}

// MT: M-tiles (16 vectors each) per wavefront step -- MT, or 1 for float32 input
// SPLIT (calls of some thousand vectors, e.g. one serving step): a workgroup is eight wavefronts that share ONE
// step of 16 vectors, wavefront w computes N-tile w with its eighth of the B operand straight from memory in
// registers -- no 64 KB fill, no cell table, one barrier; the codes meet in LDS and 256 threads pack and store
// them.  Same products, same reciprocal, same comparison against the boundaries: the same codes.
#define EM_SPLIT_WAVES 8
#define EM_SPLIT_CODES 0           // [16 vectors][128 coordinates] code bytes
#define EM_SPLIT_WAVE_OFF 2048
#define EM_SPLIT_LDS_BYTES (EM_SPLIT_WAVE_OFF + EM_SPLIT_WAVES * EM_WAVE_BYTES)
template <int BITS, bool PAGED, int XDT, bool DIRECT, int MT, bool SPLIT = false>
__global__ __launch_bounds__(EM_THREADS) void akv_encode_mfma_kernel(akv_gen_args a, const uint4* __restrict__ bop) {
  extern __shared__ __align__(16) unsigned char lds[];
  static_assert(MT <= MT && (XDT != AKV_F32 || MT == 1), "the LDS regions are sized for MT tiles");
  static_assert(!SPLIT || (MT == 1 && XDT != AKV_F32 && !DIRECT), "the split form: one M-tile of 16-bit rows");
  constexpr uint32_t WAVE_OFF = SPLIT ? EM_SPLIT_WAVE_OFF : EM_WAVE_OFF;
  constexpr int ROWS = 16 * MT;                       // vectors per wavefront step
  constexpr int XB = XDT == AKV_F32 ? 4 : 2;          // bytes per input element
  constexpr int NA = XDT == AKV_F32 ? 2 : 1;          // float16 terms of the input operand
  constexpr int NB = (1 << BITS) - 1;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;

  // ---- workgroup set-up: B operand, boundaries, cell table (called after the wavefront has requested the rows
  // of its first step, so that their trip to memory runs beside the fill: a call of one serving step is a single
  // step per wavefront and nothing else)
  auto setup = [&]() {
    uint4* b_lds = (uint4*)(lds + EM_B_OFF);
    for (int i = threadIdx.x; i < EM_B_BYTES / 16; i += EM_THREADS) b_lds[i] = bop[i];
    float* bnd = (float*)(lds + EM_BND_OFF);
    uint32_t* par = (uint32_t*)(lds + EM_PAR_OFF);
    if (threadIdx.x < 16) bnd[threadIdx.x] = threadIdx.x < NB ? a.table[threadIdx.x] : INFINITY;
    if (threadIdx.x == 0) par[0] = ((const uint32_t*)(bop + EM_B_BYTES / 16))[0];   // rows of Pi too long for the table
    __syncthreads();
    if (threadIdx.x == 0) {
      // the table serves finite, strictly increasing boundaries inside (-1, 1)
      bool ok = fabsf(bnd[0]) < 1.f && fabsf(bnd[NB - 1]) < 1.f;
      for (int k = 1; k < NB; ++k) ok = ok && (bnd[k] > bnd[k - 1]);
      if (!ok) par[0] = 1u;
    }
    __syncthreads();
    for (int c = threadIdx.x; c < EM_CELLS; c += EM_THREADS) {
      uint32_t base = 0, cnt = 0;
      float inside = INFINITY;
      for (int k = 0; k < NB; ++k) {
        const uint32_t cb = em_cell(bnd[k]) >> 3;
        if (cb < (uint32_t)c) ++base;
        if (cb == (uint32_t)c) { ++cnt; inside = bnd[k]; }
      }
      uint32_t* lut = (uint32_t*)(lds + EM_LUT_OFF);
      lut[2 * c] = base;
      lut[2 * c + 1] = __float_as_uint(inside);
      if (cnt > 1) atomicOr(par, 1u);
    }
    __syncthreads();
  };
  const float* bnd = (const float*)(lds + EM_BND_OFF);

  unsigned char* wl = lds + WAVE_OFF + wave * EM_WAVE_BYTES;
  int64_t* src_off = (int64_t*)wl;                    // address of the vector, or 0
  int64_t* dst_p = (int64_t*)(wl + ROWS * 8);      // address of the packed row, or 0
  int64_t* dst_n = (int64_t*)(wl + ROWS * 16);     // address of the norm
  float* rinv = (float*)(wl + ROWS * 24);          // 1/(|x| + 1e-10), scaled back by 1/EM_PSCALE; NaN rows flagged

  const int64_t n_total = (PAGED && a.x2) ? 2 * a.n : a.n;      // a second tensor rides along (K and V of a step)
  const int64_t steps = (n_total + ROWS - 1) / ROWS;
  const int64_t stride = SPLIT ? (int64_t)gridDim.x : (int64_t)gridDim.x * EM_WAVES;
  // SPLIT: the wavefront's N-tile of the B operand, both terms, four k-steps
  em_half8 Bh[4], Bl[4];
  if constexpr (SPLIT) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      union { uint4 u; em_half8 h; } ch, cl;
      ch.u = bop[(wave * 4 + ks) * 64 + lane];
      cl.u = bop[2048 + (wave * 4 + ks) * 64 + lane];
      Bh[ks] = ch.h;
      Bl[ks] = cl.h;
    }
  }

  // A operands of one step straight from memory (zeros past the end): lane l resolves the source
  // row of vector base + l, the lanes of an M-tile pick the rows up through LDS
  // (a row's 32 elements of the lane as 16-byte pieces: four for 16-bit input -- the A operands themselves --
  // eight for float32 input)
  constexpr int NP = 4 * NA;
  auto fetch = [&](uint4 (&R)[MT][NP], int64_t step) {
    if constexpr (DIRECT) {
      // contiguous rows whose byte offsets fit 31 bits: every lane forms its rows' addresses itself
      // (scalar base + 32-bit lane offset), no exchange through LDS
      if ((uint32_t)step * ROWS + ROWS <= (uint32_t)a.n) {      // a whole step (all but the last): nothing to check
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const uint32_t n = (uint32_t)step * ROWS + 16 * mt + (lane & 15);
          const uint4* p = (const uint4*)((const char*)a.x + (n * (uint32_t)a.xs0 + 32u * g) * (uint32_t)XB);
#pragma unroll
          for (int ks = 0; ks < NP; ++ks) R[mt][ks] = p[ks];
        }
        return;
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const uint32_t n = (uint32_t)step * ROWS + 16 * mt + (lane & 15);
        if (n < (uint32_t)a.n) {
          const uint4* p = (const uint4*)((const char*)a.x + (n * (uint32_t)a.xs0 + 32u * g) * (uint32_t)XB);
#pragma unroll
          for (int ks = 0; ks < NP; ++ks) R[mt][ks] = p[ks];
        } else {
#pragma unroll
          for (int ks = 0; ks < NP; ++ks) R[mt][ks] = make_uint4(0u, 0u, 0u, 0u);
        }
      }
      return;
    }
    int64_t n = step * ROWS + lane;
    int64_t so = 0;      // byte address of the vector, 0 = none
    if (step < steps && n < n_total && lane < ROWS) {
      const bool second = PAGED && n >= a.n;
      if (second) n -= a.n;
      const char* xb = (const char*)(second ? a.x2 : a.x);
      if (PAGED) {
        const int64_t tok = n / a.heads, head = n - tok * a.heads;
        so = (int64_t)(uintptr_t)(xb + XB * (tok * a.xs0 + head * a.xs1));
      } else {
        so = (int64_t)(uintptr_t)(xb + XB * n * a.xs0);
      }
    }
    if (lane < ROWS) src_off[lane] = so;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int64_t ro = src_off[16 * mt + (lane & 15)];
      if (ro != 0) {
        const uint4* p = (const uint4*)(uintptr_t)(ro + 32 * XB * g);
#pragma unroll
        for (int ks = 0; ks < NP; ++ks) R[mt][ks] = p[ks];
      } else {
#pragma unroll
        for (int ks = 0; ks < NP; ++ks) R[mt][ks] = make_uint4(0u, 0u, 0u, 0u);
      }
    }
  };

  auto encode_step = [&](auto linear_tag, int64_t step, uint4 (&R)[MT][NP]) {
    constexpr bool LINEAR = decltype(linear_tag)::value;
    em_half8 A[MT][4];          // the operand (16-bit input), or its float16 hi term (float32 input)
    em_half8 Alo[MT][4];        // float32 input: the lo term
    if constexpr (XDT != AKV_F32) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          union { uint4 u; em_half8 h; } cv;
          cv.u = R[mt][ks];
          A[mt][ks] = cv.h;
        }
    }
    const int64_t base = step * ROWS;
    // ---- lane l resolves the destination of vector base + l
    if constexpr (!DIRECT) {
      int64_t n = base + lane;
      int64_t dp = 0, dn = 0;      // byte addresses of the packed row and of the norm, 0 = skip
      if (n < n_total && lane < ROWS) {
        const bool second = PAGED && n >= a.n;
        if (second) n -= a.n;
        uint8_t* pb = second ? a.packed2 : a.packed;
        float* nb = second ? a.norms2 : a.norms;
        if (PAGED) {
          const int64_t tok = n / a.heads, head = n - tok * a.heads;
          const int64_t slot = akv_load_index(a.slots, a.slot_itype, tok);
          if (slot >= 0) {
            const int64_t blk = slot / a.block_size, pos = slot - blk * a.block_size;
            if (blk < a.max_blocks) {
              dp = (int64_t)(uintptr_t)(pb + blk * a.ps0 + pos * a.ps1 + head * a.ps2);
              dn = (int64_t)(uintptr_t)(nb + blk * a.ns0 + pos * a.ns1 + head * a.ns2);
            }
          }
        } else {
          dp = (int64_t)(uintptr_t)(pb + n * a.ps0);
          dn = (int64_t)(uintptr_t)(nb + n);
        }
      }
      if (lane < ROWS) {
        dst_p[lane] = dp;
        dst_n[lane] = dn;
      }
    }
    float ss[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) ss[mt] = 0.f;
    uint32_t unscale[MT];     // float bits of the power of two taken out of each M-tile's rows
    bool nonfinite[MT];       // bfloat16 only: the row holds an infinity or a NaN
    if constexpr (XDT == AKV_F16) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        unscale[mt] = 0x3f800000u;
        nonfinite[mt] = false;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          union { em_half8 h; em_half2 h2[4]; } cv;
          cv.h = A[mt][ks];
#pragma unroll
          for (int q = 0; q < 4; ++q) ss[mt] = __builtin_amdgcn_fdot2(cv.h2[q], cv.h2[q], ss[mt], false);
        }
      }
    } else if constexpr (XDT == AKV_F32) {
      // float32 rows: squared norm from the values themselves; then each row is scaled by the power of two
      // that brings its largest element into [1, 2) and split into two float16 terms, both rounded to
      // nearest: hi keeps 11 bits, x - hi is exact in float32 and has at most 12 significant bits and a sign,
      // so lo is off by at most half a float32 ulp of the element (2^-25 of the largest element once lo is a
      // float16 subnormal)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        uint32_t mx = 0u;
#pragma unroll
        for (int pc = 0; pc < NP; ++pc) {
          const uint32_t w[4] = {R[mt][pc].x, R[mt][pc].y, R[mt][pc].z, R[mt][pc].w};
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            mx = max(mx, w[q] & 0x7fffffffu);
            const float v = __uint_as_float(w[q]);
            ss[mt] = fmaf(v, v, ss[mt]);
          }
        }
        {   // largest magnitude of the row over its four lanes
          auto r1 = __builtin_amdgcn_permlane32_swap(mx, mx, false, false);
          mx = max(r1[0], r1[1]);
          auto r2 = __builtin_amdgcn_permlane16_swap(mx, mx, false, false);
          mx = max(r2[0], r2[1]);
        }
        uint32_t ef = mx >> 23;                      // exponent field of the largest element
        nonfinite[mt] = ef == 255u;
        if (ef == 0u || ef == 255u) ef = 127u;       // all (sub)zero, or not finite (flagged)
        if (ef == 254u) ef = 253u;                   // keep the scale a normal number
        const float sc = __uint_as_float((254u - ef) << 23);     // 2^(127 - ef)
        unscale[mt] = ef << 23;                                   // 2^(ef - 127)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          const float v[8] = {__uint_as_float(R[mt][2 * ks].x), __uint_as_float(R[mt][2 * ks].y),
                              __uint_as_float(R[mt][2 * ks].z), __uint_as_float(R[mt][2 * ks].w),
                              __uint_as_float(R[mt][2 * ks + 1].x), __uint_as_float(R[mt][2 * ks + 1].y),
                              __uint_as_float(R[mt][2 * ks + 1].z), __uint_as_float(R[mt][2 * ks + 1].w)};
          union { em_half8 h; em_half2 h2[4]; } hi, lo;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float x0 = v[2 * q] * sc, x1 = v[2 * q + 1] * sc;
            const _Float16 h0 = (_Float16)x0, h1 = (_Float16)x1;
            hi.h2[q] = (em_half2){h0, h1};
            lo.h2[q] = (em_half2){(_Float16)(x0 - (float)h0), (_Float16)(x1 - (float)h1)};
          }
          A[mt][ks] = hi.h;
          Alo[mt][ks] = lo.h;
        }
      }
    } else {
      // bfloat16 rows: squared norm from the exact float32 values; then each row is scaled by the
      // power of two that brings its largest element into [1, 2) and converted to float16 -- exact
      // for every element within 2^14 of the largest (8 significant bits fit in 11), and off by at
      // most 2^-25 of the largest otherwise, far below the resolution of the codebook search
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        em_us2 mx2 = {0, 0};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          union { em_half8 h; uint32_t w[4]; } cv;
          cv.h = A[mt][ks];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            union { uint32_t u; em_us2 v; } mm;
            mm.u = cv.w[q] & 0x7fff7fffu;
            mx2 = __builtin_elementwise_max(mx2, mm.v);
            const float lo = __uint_as_float(cv.w[q] << 16), hi = __uint_as_float(cv.w[q] & 0xffff0000u);
            ss[mt] = fmaf(lo, lo, ss[mt]);
            ss[mt] = fmaf(hi, hi, ss[mt]);
          }
        }
        uint32_t mx = max((uint32_t)mx2[0], (uint32_t)mx2[1]);
        {   // largest magnitude of the row over its four lanes
          auto r1 = __builtin_amdgcn_permlane32_swap(mx, mx, false, false);
          mx = max(r1[0], r1[1]);
          auto r2 = __builtin_amdgcn_permlane16_swap(mx, mx, false, false);
          mx = max(r2[0], r2[1]);
        }
        uint32_t ef = mx >> 7;                       // exponent field of the largest element
        nonfinite[mt] = ef == 255u;
        if (ef == 0u || ef == 255u) ef = 127u;       // all (sub)zero, or not finite (flagged)
        if (ef == 254u) ef = 253u;                   // keep the scale a normal number
        const float sc = __uint_as_float((254u - ef) << 23);     // 2^(127 - ef)
        unscale[mt] = ef << 23;                                   // 2^(ef - 127)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          union { em_half8 h; uint32_t w[4]; em_half2 h2[4]; } cv;
          cv.h = A[mt][ks];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float lo = __uint_as_float(cv.w[q] << 16) * sc, hi = __uint_as_float(cv.w[q] & 0xffff0000u) * sc;
            auto pk = __builtin_amdgcn_cvt_pkrtz(lo, hi);
            cv.h2[q] = (em_half2){(_Float16)pk[0], (_Float16)pk[1]};
          }
          A[mt][ks] = cv.h;
        }
      }
    }
    // lane l < ROWS finishes vector l = 16 mt + row: transpose-reduce the partial sums over the
    // four lanes of a row
    bool any_nan;       // some vector of the step holds a NaN or an infinity (the same in every lane)
    {
      const bool g1 = (g & 1) != 0;
      float mine;
      if constexpr (MT == 1) {
        const float a01 = ss[0] + akv_lane_xor<16>(ss[0]);     // (row swaps, not shuffles: the step waits for this chain)
        mine = a01 + akv_lane_xor<32>(a01);                   // all four lanes of a row hold its sum
      } else {
        static_assert(MT <= 2, "two M-tiles at most");
        const float a01 = (g1 ? ss[MT - 1] : ss[0]) + akv_lane_xor<16>(g1 ? ss[0] : ss[MT - 1]);
        mine = a01 + akv_lane_xor<32>(a01);                   // lanes g and g + 2 both hold M-tile g & 1
      }
      const float nrm = sqrtf(mine);
      const uint32_t my_unscale = (MT > 1 && g1) ? unscale[MT - 1] : unscale[0];
      const float r = (1.f / (nrm + 1e-10f)) * (1.f / EM_PSCALE) * __uint_as_float(my_unscale);
      // a vector with a NaN or an infinity rotates to NaN everywhere: every code is the last level.
      // (float16 squares cannot overflow, so there an infinite norm means an infinite element; a
      // finite bfloat16 row whose squares overflow has norm inf, unit vector 0 and y = 0 like the
      // reference: r is 0 and the scaled products are finite.)
      const bool my_nonfinite = (MT > 1 && g1) ? nonfinite[MT - 1] : nonfinite[0];
      const bool nan_row = XDT == AKV_F16 ? !(nrm < INFINITY) : (my_nonfinite || nrm != nrm);   // (float32 as bfloat16)
      any_nan = __ballot(nan_row && lane < ROWS) != 0;
      if (lane < ROWS) {
        rinv[lane] = nan_row ? __uint_as_float(0x7fc00000u) : r;
        if constexpr (DIRECT) {
          if ((uint32_t)base + lane < (uint32_t)a.n) a.norms[(uint32_t)base + lane] = nrm;
        } else {
          if (dst_p[lane] != 0 && (!SPLIT || wave == 0)) *(float*)(uintptr_t)dst_n[lane] = nrm;
        }
      }
    }
    if constexpr (SPLIT) {
      // ---- the wavefront's tile: products, reciprocal, comparison with every boundary, code bytes to LDS
      union { em_u32x4 u; em_float4 f; } rc;
      rc.u = *(em_lds_u128*)(uintptr_t)(uint32_t)(WAVE_OFF + wave * EM_WAVE_BYTES + ROWS * 24 + (4 * g) * 4);
      em_float4 acc = (em_float4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[0][ks], Bh[ks], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[0][ks], Bl[ks], acc, 0, 0, 0);
      }
      uint8_t* codes = lds + EM_SPLIT_CODES;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float y = acc[i] * rc.f[i];
        uint32_t code = 0;
#pragma unroll
        for (int k = 0; k < NB; ++k) code += (a.table[k] < y) ? 1u : 0u;
        if (!(rc.f[i] == rc.f[i])) code = (uint32_t)NB;            // NaN vector: last level everywhere
        codes[(4 * g + i) * 128 + 8 * col + wave] = (uint8_t)code;
      }
      __syncthreads();
      if (threadIdx.x < 256) {
        const int row = threadIdx.x >> 4, grp = threadIdx.x & 15;
        const int64_t dp = dst_p[row];
        if (dp != 0) {
          const uint2 c8 = *(const uint2*)(codes + row * 128 + 8 * grp);
          auto code_of = [&](int t) { return ((t < 4 ? c8.x : c8.y) >> (8 * (t & 3))) & 0xffu; };
          uint32_t v = 0;
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const int t = BITS == 4 ? 6 - (k & ~1) + (k & 1) : BITS == 3 ? k : ((k + 4) & 7);
            v = (v << BITS) + code_of(t);
          }
          uint8_t* prow = (uint8_t*)(uintptr_t)dp;
          if (BITS == 4) {
            *(uint32_t*)(prow + 4 * grp) = v;
          } else if (BITS == 3) {
            prow[3 * grp] = (uint8_t)(v >> 16);
            prow[3 * grp + 1] = (uint8_t)(v >> 8);
            prow[3 * grp + 2] = (uint8_t)v;
          } else {
            *(uint16_t*)(prow + 2 * grp) = (uint16_t)v;
          }
        }
      }
      __syncthreads();      // the code bytes are rewritten by the next step
      return;
    }
    // ---- rotate, search, pack
    uint32_t packed[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) packed[mt][i] = 0u;
    em_float4 rv[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      union { em_u32x4 u; em_float4 f; } cv;
      cv.u = *(em_lds_u128*)(uintptr_t)(uint32_t)(WAVE_OFF + wave * EM_WAVE_BYTES + ROWS * 24 + (16 * mt + 4 * g) * 4);
      rv[mt] = cv.f;
    }
    // N-tiles are software-pipelined: the matrix-core work of tile nt + 1 is issued together with
    // the search of tile nt (independent instruction streams in one basic block), so the vector
    // unit works in the shadow of the MFMAs.  The loop stays rolled (two tiles per pass): unrolled,
    // the scheduler would want every B operand in registers at once.
    auto mfma_tile = [&](int nt, em_float4 (&acc)[MT]) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = (em_float4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        union { em_u32x4 u; em_half8 h; } bh, bl;
        bh.u = *(em_lds_u128*)(uintptr_t)(uint32_t)(EM_B_OFF + ((nt * 4 + ks) * 64 + lane) * 16);
        bl.u = *(em_lds_u128*)(uintptr_t)(uint32_t)(EM_B_OFF + 32768 + ((nt * 4 + ks) * 64 + lane) * 16);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[mt][ks], bh.h, acc[mt], 0, 0, 0);
          acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[mt][ks], bl.h, acc[mt], 0, 0, 0);
          if constexpr (XDT == AKV_F32)
            acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Alo[mt][ks], bh.h, acc[mt], 0, 0, 0);
        }
      }
    };
    // A lane's packed group is built by shift-and-add, one instruction per code: the N-tiles are visited
    // in the order in which their codes enter the group from the top (4-bit: 6 7 4 5 2 3 0 1 -- a dword
    // is four little-endian bytes of two nibbles; 3-bit: 0 .. 7; 2-bit: 4 5 6 7 0 1 2 3).
    auto tile_at = [&](int k) -> int {
      return BITS == 4 ? 6 - (k & ~1) + (k & 1) : BITS == 3 ? k : ((k + 4) & 7);
    };
    auto search_tile = [&](const em_float4 (&acc)[MT]) {
      float y[MT][4];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) y[mt][i] = acc[mt][i] * rv[mt][i];
      if constexpr (!LINEAR) {
        em_u32x2 e[MT][4];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            e[mt][i] = *(em_lds_u64*)(uintptr_t)em_cell(y[mt][i]);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint32_t code = e[mt][i].x + ((__uint_as_float(e[mt][i].y) < y[mt][i]) ? 1u : 0u);
            packed[mt][i] = (packed[mt][i] << BITS) + code;
          }
      } else {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            uint32_t code = 0;
#pragma unroll 1
            for (int k = 0; k < NB; ++k) code += (bnd[k] < y[mt][i]) ? 1u : 0u;
            packed[mt][i] = (packed[mt][i] << BITS) + code;
          }
      }
    };
    em_float4 accA[MT], accB[MT];
    mfma_tile(tile_at(0), accA);
#pragma unroll 1
    for (int k = 0; k < 6; k += 2) {
      mfma_tile(tile_at(k + 1), accB);
      search_tile(accA);
      mfma_tile(tile_at(k + 2), accA);
      search_tile(accB);
      // issue order of the pass: one MFMA, then the vector and LDS work that fits in its shadow
#pragma unroll
      for (int q = 0; q < 8 * (NA + 1) * MT; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);   // VALU
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // LDS read
      }
    }
    mfma_tile(tile_at(7), accB);
    search_tile(accA);
#pragma unroll
    for (int q = 0; q < 4 * (NA + 1) * MT; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    search_tile(accB);
    // ---- store: lane (col, g) writes group col of rows 4g + i
    auto put = [&](uint8_t* prow, uint32_t v) {
      if (BITS == 4) {
        *(uint32_t*)(prow + 4 * col) = v;
      } else if (BITS == 3) {
        prow[3 * col] = (uint8_t)(v >> 16);
        prow[3 * col + 1] = (uint8_t)(v >> 8);
        prow[3 * col + 2] = (uint8_t)v;
      } else {
        *(uint16_t*)(prow + 2 * col) = (uint16_t)v;
      }
    };
    if (DIRECT && !any_nan && (uint32_t)base + ROWS <= (uint32_t)a.n) {
      // a whole step of finite vectors (all but a few): the row's address is a scalar (step and row number)
      // plus the lane's own offset (its row quarter and group), nothing is checked
      const uint32_t lane_off = (uint32_t)(4 * g) * (uint32_t)a.ps0;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          put(a.packed + (uint64_t)((uint32_t)base + 16 * mt + i) * (uint32_t)a.ps0 + lane_off, packed[mt][i]);
      return;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * mt + 4 * g + i;
        uint8_t* prow;
        if constexpr (DIRECT) {
          const uint32_t n = (uint32_t)base + row;
          if (n >= (uint32_t)a.n) continue;
          prow = a.packed + n * (uint32_t)a.ps0;
        } else {
          const int64_t dp = dst_p[row];
          if (dp == 0) continue;
          prow = (uint8_t*)(uintptr_t)dp;
        }
        uint32_t v = packed[mt][i];
        if (!(rv[mt][i] == rv[mt][i])) v = 0xffffffffu;     // NaN vector: last level everywhere
        put(prow, v);
      }
  };

  // the rows of a step are requested at the end of the step before it (the first: before the set-up)
  const int64_t first = SPLIT ? (int64_t)blockIdx.x : (int64_t)wave * gridDim.x + blockIdx.x;
  uint4 R[MT][NP];
  fetch(R, first);
  if constexpr (SPLIT) {
    for (int64_t step = first; step < steps; step += stride) {      // (the same steps in every wavefront)
      encode_step(std::true_type{}, step, R);
      fetch(R, step + stride);
    }
    return;
  }
  setup();
  const bool linear_search = ((const uint32_t*)(lds + EM_PAR_OFF))[0] != 0;   // uniform
  if (__builtin_expect(!linear_search, 1)) {
    for (int64_t step = first; step < steps; step += stride) {
      encode_step(std::false_type{}, step, R);
      fetch(R, step + stride);
    }
  } else {
    for (int64_t step = first; step < steps; step += stride) {
      encode_step(std::true_type{}, step, R);
      fetch(R, step + stride);
    }
  }
}

// ----------------------------------------------------------------------------------
// encode with the matrix in registers: a workgroup is four wavefronts that share a step of 16 MT rows, wavefront w owns output
// coordinates 32 w .. 32 w + 31 (two tiles of 16, both terms, 64 registers) and multiplies them into all rows.  The threads
// load the rows (16 / MT lanes a row), take their norms and leave them in LDS as float16 terms, once for all wavefronts:
//
//   Y[j, v] = sum_i Pi[j, i] X[v, i]              v_mfma_f32_16x16x32_f16, Pi the first operand
//
// Row m of tile t is coordinate 32 w + 8 (m / 4) + 4 t + m % 4, so lane (v, g) ends up with coordinates 32 w + 8 g .. + 7 of row v:
// one group of the packed row, stored from where it is.  The terms, their products and the order of the sums are those of the
// kernel above.
// ----------------------------------------------------------------------------------
template <int XDT, int MT> struct er_cfg {
  static constexpr int ROWS = 16 * MT, LPR = 16 / MT;             // rows of a step, lanes of a row while loading
  static constexpr int NA = XDT == AKV_F32 ? 2 : 1, NP = MT * NA; // float16 terms of a row, 16-byte pieces of a thread
  static constexpr int PITCH = 128 * 2 + 16;                      // bytes of a row in LDS (sixteen rows meet all banks)
  static constexpr int BND = EM_CELLS * 8, DST = BND + 64, INFO = DST + ROWS * 8, DATA = INFO + ROWS * 4;
  static constexpr int LDS = DATA + NA * ROWS * PITCH;
};
// floor((2^32 - 1) / heads) and / block size; slots of the cache.  (Products in 32 and 24 bits: er_fits.  In 64 bits they were a quarter
// of a step's vector cycles.)
struct er_div { uint32_t heads_r, block_r, slots; };

template <int BITS, bool PAGED, int XDT, int MT>
__global__ __launch_bounds__(256, 3) void akv_encode_rows_kernel(akv_gen_args a, const uint4* __restrict__ bop, er_div dv) {
  extern __shared__ __align__(16) unsigned char lds[];            // the kernel's only LDS object: the cell table lies at address 0
  typedef er_cfg<XDT, MT> cfg;
  constexpr int ROWS = cfg::ROWS, LPR = cfg::LPR, NA = cfg::NA, NP = cfg::NP, PITCH = cfg::PITCH;
  constexpr int XB = XDT == AKV_F32 ? 4 : 2, NB = (1 << BITS) - 1;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, g = lane >> 4;
  const int row = tid / LPR, part = tid % LPR;
  const uint32_t n_one = (uint32_t)a.n, n_total = PAGED && a.x2 ? 2u * n_one : n_one;

  // ---- the rows: thread (row, part) takes elements 8 MT part .. + 8 MT - 1
  uint4 R[NP];
  uint32_t tok = 0, head = 0;
  bool second = false, held = false;
  int64_t slot = 0;
  {
    uint32_t n = blockIdx.x * ROWS + row;
    held = n < n_total;                                          // (past the end: the last row, not stored)
    n = min(n, n_total - 1);
    second = PAGED && n >= n_one;
    if (second) n -= n_one;
    tok = n;
    if constexpr (PAGED) tok = akv_div32(n, (uint32_t)a.heads, dv.heads_r, head);
    const uint64_t off = (uint64_t)tok * (uint32_t)a.xs0 + (PAGED ? __umul24(head, (uint32_t)a.xs1) : 0u);
    const char* p = (const char*)(second ? a.x2 : a.x) + XB * off;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int h = 0; h < NA; ++h) R[i * NA + h] = *(const uint4*)(p + (part * MT + i) * 8 * XB + 16 * h);
    if constexpr (PAGED) slot = akv_load_index(a.slots, a.slot_itype, tok);
  }

  // ---- the wavefront's tiles of the matrix
  em_half8 Ph[2][4], Pl[2][4];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      union { uint4 u; em_half8 h; } ch, cl;
      const int at = ((4 * t + (col & 3)) * 4 + ks) * 64 + 16 * g + 4 * wave + (col >> 2);
      ch.u = bop[at];
      cl.u = bop[2048 + at];
      Ph[t][ks] = ch.h;
      Pl[t][ks] = cl.h;
    }

  // ---- cell table (as above; every thread judges the boundaries for itself)
  bool linear;
  {
    float b[NB];
    uint32_t cell[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) b[k] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(a.table[k])));
    bool ok = fabsf(b[0]) < 1.f && fabsf(b[NB - 1]) < 1.f;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      cell[k] = __builtin_amdgcn_readfirstlane(em_cell(b[k]) >> 3);
      if (k > 0) ok = ok && b[k] > b[k - 1] && cell[k] != cell[k - 1];
    }
    linear = !ok || ((const uint32_t*)(bop + EM_B_BYTES / 16))[0] != 0u;
    if (tid == 0) {
#pragma unroll
      for (int k = 0; k < NB; ++k) ((float*)(lds + cfg::BND))[k] = b[k];
    }
#pragma unroll
    for (int c = tid; c < EM_CELLS; c += 256) {
      uint32_t base = 0;
      float inside = INFINITY;
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        base += cell[k] < (uint32_t)c ? 1u : 0u;
        inside = cell[k] == (uint32_t)c ? b[k] : inside;
      }
      *(uint2*)(lds + 8 * c) = make_uint2(base, __float_as_uint(inside));
    }
  }

  // ---- norms, float16 terms into LDS, where the packed rows go
  {
    // squared norm: a quarter of the row is one chain of sums, as above, which its 4 / MT lanes walk one after another
    float ss = 0.f;
#pragma unroll
    for (int stage = 0; stage < 4 / MT; ++stage) {
      if (stage > 0) ss = __uint_as_float(akv_dpp_u32<(MT == 1 ? 0x90 : 0xA0) /*the lane before: quad_perm 0,0,1,2 or 0,0,2,2*/>(__float_as_uint(ss)));
      if (stage > 0 && part % (4 / MT) == 0) ss = 0.f;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const uint32_t w[4] = {R[i].x, R[i].y, R[i].z, R[i].w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if constexpr (XDT == AKV_F16) {
            union { uint32_t u; em_half2 h; } cv;
            cv.u = w[q];
            ss = __builtin_amdgcn_fdot2(cv.h, cv.h, ss, false);
          } else if constexpr (XDT == AKV_BF16) {
            const float e0 = __uint_as_float(w[q] << 16), e1 = __uint_as_float(w[q] & 0xffff0000u);
            ss = fmaf(e0, e0, ss);
            ss = fmaf(e1, e1, ss);
          } else {
            ss = fmaf(__uint_as_float(w[q]), __uint_as_float(w[q]), ss);
          }
        }
      }
    }
    constexpr int LAST = 4 / MT - 1;                 // lanes part % (4 / MT) == LAST hold the sum of their quarter
    ss += akv_lane_xor<4 / MT>(ss);
    ss += akv_lane_xor<8 / MT>(ss);
    uint32_t unscale = 0x3f800000u;
    bool nonfinite = false;
    uint4 hi[MT], lo[MT];
    if constexpr (XDT == AKV_F16) {
#pragma unroll
      for (int i = 0; i < MT; ++i) hi[i] = R[i];
    } else {
      // scaled by the power of two of the largest element, as above
      uint32_t ef;
      if constexpr (XDT == AKV_BF16) {
        em_us2 mx2 = {0, 0};
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const uint32_t w[4] = {R[i].x, R[i].y, R[i].z, R[i].w};
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            union { uint32_t u; em_us2 v; } mm;
            mm.u = w[q] & 0x7fff7fffu;
            mx2 = __builtin_elementwise_max(mx2, mm.v);
          }
        }
        ef = max((uint32_t)mx2[0], (uint32_t)mx2[1]) >> 7;
      } else {
        uint32_t mx = 0u;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
          const uint32_t w[4] = {R[i].x, R[i].y, R[i].z, R[i].w};
#pragma unroll
          for (int q = 0; q < 4; ++q) mx = max(mx, w[q] & 0x7fffffffu);
        }
        ef = mx >> 23;
      }
      ef = max(ef, akv_lane_xor_u32<1>(ef));
      ef = max(ef, akv_lane_xor_u32<2>(ef));
      if constexpr (LPR >= 8) ef = max(ef, akv_lane_xor_u32<4>(ef));
      if constexpr (LPR >= 16) ef = max(ef, akv_lane_xor_u32<8>(ef));
      nonfinite = ef == 255u;
      if (ef == 0u || ef == 255u) ef = 127u;       // all (sub)zero, or not finite (flagged)
      if (ef == 254u) ef = 253u;                   // keep the scale a normal number
      const float sc = __uint_as_float((254u - ef) << 23);
      unscale = ef << 23;
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        union { uint4 u; uint32_t w[4]; em_half2 h2[4]; } ph, pl;
        if constexpr (XDT == AKV_BF16) {
          const uint32_t w[4] = {R[i].x, R[i].y, R[i].z, R[i].w};
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            auto pk = __builtin_amdgcn_cvt_pkrtz(__uint_as_float(w[q] << 16) * sc, __uint_as_float(w[q] & 0xffff0000u) * sc);
            ph.h2[q] = (em_half2){(_Float16)pk[0], (_Float16)pk[1]};
          }
        } else {
          const uint32_t w[8] = {R[2 * i].x, R[2 * i].y, R[2 * i].z, R[2 * i].w, R[2 * i + NA - 1].x, R[2 * i + NA - 1].y, R[2 * i + NA - 1].z, R[2 * i + NA - 1].w};
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float x0 = __uint_as_float(w[2 * q]) * sc, x1 = __uint_as_float(w[2 * q + 1]) * sc;
            const _Float16 h0 = (_Float16)x0, h1 = (_Float16)x1;
            ph.h2[q] = (em_half2){h0, h1};
            pl.h2[q] = (em_half2){(_Float16)(x0 - (float)h0), (_Float16)(x1 - (float)h1)};
          }
          lo[i] = pl.u;
        }
        hi[i] = ph.u;
      }
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      unsigned char* p = lds + cfg::DATA + row * PITCH + (part * MT + i) * 16;
      *(uint4*)p = hi[i];
      if constexpr (NA == 2) *(uint4*)(p + ROWS * PITCH) = lo[i];
    }
    const float nrm = sqrtf(ss);
    const float r = (1.f / (nrm + 1e-10f)) * (1.f / EM_PSCALE) * __uint_as_float(unscale);
    const bool nan_row = XDT == AKV_F16 ? !(nrm < INFINITY) : (nonfinite || nrm != nrm);
    // ---- where the row goes
    uint8_t* pb = second ? a.packed2 : a.packed;
    float* nb = second ? a.norms2 : a.norms;
    bool stored = held;
    if constexpr (PAGED) {
      stored = held && (uint64_t)slot < dv.slots;
      uint32_t pos;
      const uint32_t blk = akv_div32((uint32_t)slot, (uint32_t)a.block_size, dv.block_r, pos);
      pb += (uint64_t)blk * (uint32_t)a.ps0 + (__umul24(pos, (uint32_t)a.ps1) + __umul24(head, (uint32_t)a.ps2));
      nb += (uint64_t)blk * (uint32_t)a.ns0 + (__umul24(pos, (uint32_t)a.ns1) + __umul24(head, (uint32_t)a.ns2));
    } else {
      pb += (uint64_t)tok * (uint32_t)a.ps0;
      nb += tok;
    }
    if (part == LAST) {
      ((uint64_t*)(lds + cfg::DST))[row] = stored ? (uint64_t)(uintptr_t)pb : 0u;
      ((float*)(lds + cfg::INFO))[row] = nan_row ? __uint_as_float(0x7fc00000u) : r;
      if (stored) *nb = nrm;
    }
  }
  __syncthreads();

  // ---- rotate, search, pack, store
  auto encode = [&](auto linear_tag) __attribute__((always_inline)) {
    constexpr bool LINEAR = decltype(linear_tag)::value;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int v = 16 * mt + col;
      em_float4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      const unsigned char* p = lds + cfg::DATA + v * PITCH + 64 * g;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const em_half8 x = *(const em_half8*)(p + 16 * ks);
        em_half8 xl;
        if constexpr (NA == 2) xl = *(const em_half8*)(p + ROWS * PITCH + 16 * ks);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ph[t][ks], x, acc[t], 0, 0, 0);
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Pl[t][ks], x, acc[t], 0, 0, 0);
          if constexpr (NA == 2) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Ph[t][ks], xl, acc[t], 0, 0, 0);
        }
      }
      const float r = ((const float*)(lds + cfg::INFO))[v];
      const uint64_t dp = ((const uint64_t*)(lds + cfg::DST))[v];
      float y[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) y[k] = acc[k >> 2][k & 3] * r;
      uint32_t code[8];
      if constexpr (!LINEAR) {
        em_u32x2 e[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) e[k] = *(em_lds_u64*)(uintptr_t)em_cell(y[k]);
#pragma unroll
        for (int k = 0; k < 8; ++k) code[k] = e[k].x + (__uint_as_float(e[k].y) < y[k] ? 1u : 0u);
      } else {
        const float* bnd = (const float*)(lds + cfg::BND);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          code[k] = 0;
#pragma unroll 1
          for (int b = 0; b < NB; ++b) code[k] += bnd[b] < y[k] ? 1u : 0u;
        }
      }
      // the group by shift and add, its codes in the order in which they enter it from the top
      uint32_t w = 0;
#pragma unroll
      for (int k = 0; k < 8; ++k) w = (w << BITS) + code[BITS == 4 ? 6 - (k & ~1) + (k & 1) : BITS == 3 ? k : ((k + 4) & 7)];
      if (!(r == r)) w = 0xffffffffu;                // NaN vector: last level everywhere
      if (dp != 0) {
        uint8_t* q = (uint8_t*)(uintptr_t)dp + BITS * (4 * wave + g);
        if constexpr (BITS == 4) {
          *(uint32_t*)q = w;
        } else if constexpr (BITS == 3) {
          q[0] = (uint8_t)(w >> 16);
          q[1] = (uint8_t)(w >> 8);
          q[2] = (uint8_t)w;
        } else {
          *(uint16_t*)q = (uint16_t)w;
        }
      }
    }
  };

  if (__builtin_expect(!linear, 1)) encode(std::false_type{});
  else encode(std::true_type{});
}

// rows a CU up to which a call of 16-bit rows shares each step of 16 among eight wavefronts (akv_encode_mfma_try)
static constexpr int em_split_rows(int bits, bool paged) { return paged && bits != 4 ? 8 : 16; }

// what the kernel's 32- and 24-bit products take
static bool er_fits(const akv_gen_args& a, bool paged, int64_t n_total) {
  auto below = [](int64_t v, int bits) { return v >= 0 && v < ((int64_t)1 << bits); };
  if (!below(n_total, 31) || !below(a.xs0, 32) || !below(a.ps0, 32)) return false;
  if (!paged) return true;
  return below(a.max_blocks, 31) && below(a.block_size, 24) && a.max_blocks * a.block_size < ((int64_t)1 << 31) && below(a.heads, 24) && below(a.ns0, 32) &&
         below(a.xs1, 24) && below(a.ps1, 24) && below(a.ps2, 24) && below(a.ns1, 24) && below(a.ns2, 24) && below(a.heads * a.xs1, 32) &&
         below(a.block_size * a.ps1 + a.heads * a.ps2, 32) && below(a.block_size * a.ns1 + a.heads * a.ns2, 32);
}

template <int BITS, bool PAGED, int XDT, int MT>
static int er_launch(const akv_gen_args& a, const uint4* bop, const er_div& dv, int64_t n, hipStream_t stream) {
  AKV_LAUNCH_TIMED((akv_encode_rows_kernel<BITS, PAGED, XDT, MT>), (int)((n + 16 * MT - 1) / (16 * MT)), 256, (er_cfg<XDT, MT>::LDS), stream, a, bop, dv);
  AKV_LAUNCH_CHECK("akv_encode_rows_kernel");
  return AKV_OK;
}
// steps of 16, 32 or 64 rows (float32: of 32 at most), so that a call that gives a CU one step has it on every CU
template <int BITS, bool PAGED, int XDT>
static int er_run_rows(const akv_gen_args& a, const uint4* bop, int64_t n, int cus, hipStream_t stream) {
  er_div dv = {0u, 0u, 0u};
  if constexpr (PAGED) dv = {0xffffffffu / (uint32_t)a.heads, 0xffffffffu / (uint32_t)a.block_size, (uint32_t)(a.max_blocks * a.block_size)};
  if constexpr (XDT == AKV_F32 || em_split_rows(BITS, PAGED) < 16)
    if (n <= 16 * (int64_t)cus) return er_launch<BITS, PAGED, XDT, 1>(a, bop, dv, n, stream);
  if constexpr (XDT != AKV_F32)
    if (n > 32 * (int64_t)cus) return er_launch<BITS, PAGED, XDT, 4>(a, bop, dv, n, stream);
  return er_launch<BITS, PAGED, XDT, 2>(a, bop, dv, n, stream);
}
static int er_run(const akv_gen_args& a, bool paged, int x_dtype, int bits, const uint4* bop, int64_t n, int cus, hipStream_t stream) {
#define ER_DT(BB, PG) (x_dtype == AKV_F16 ? er_run_rows<BB, PG, AKV_F16>(a, bop, n, cus, stream) : x_dtype == AKV_BF16 ? er_run_rows<BB, PG, AKV_BF16>(a, bop, n, cus, stream) \
                                                                                                : er_run_rows<BB, PG, AKV_F32>(a, bop, n, cus, stream))
  if (bits == 4) return paged ? ER_DT(4, true) : ER_DT(4, false);
  if (bits == 3) return paged ? ER_DT(3, true) : ER_DT(3, false);
  return paged ? ER_DT(2, true) : ER_DT(2, false);
#undef ER_DT
}

// the split form exists for 16-bit rows addressed row by row; returns false where it does not
template <int BB, bool PG, int DT, bool DR>
static bool em_launch_split(int grid, hipStream_t stream, const akv_gen_args& a, const uint4* bop) {
  if constexpr (DT != AKV_F32 && !DR) {
    AKV_LAUNCH_TIMED((akv_encode_mfma_kernel<BB, PG, DT, false, 1, true>), grid, EM_SPLIT_WAVES * 64, EM_SPLIT_LDS_BYTES,
                     stream, a, bop);
    return true;
  } else {
    return false;
  }
}

static bool em_disabled() {
  static int v = -1;
  if (v < 0) {
    const char* e = getenv("AKV_DISABLE_MFMA");
    v = (e && e[0] == '1') ? 1 : 0;
  }
  return v == 1;
}

int akv_encode_mfma_try(const akv_gen_args& a, bool paged, int x_dtype, int d, int bits,
                        const void* rot_prep, hipStream_t stream) {
  if (em_disabled() || d != 128 || (x_dtype != AKV_F16 && x_dtype != AKV_BF16 && x_dtype != AKV_F32)) return AKV_ERR_UNSUPPORTED;
  // 16-byte loads of the input rows; aligned stores of the packed groups
  const int64_t xmask = x_dtype == AKV_F32 ? 3 : 7;        // elements per 16 bytes, minus one
  if (((uintptr_t)a.x & 15) || ((uintptr_t)a.x2 & 15) || (a.xs0 & xmask) || (paged && (a.xs1 & xmask))) return AKV_ERR_UNSUPPORTED;
  const int64_t amask = bits == 4 ? 3 : bits == 2 ? 1 : 0;
  if (((uintptr_t)a.packed | (uintptr_t)a.packed2 | (uintptr_t)a.ps0 | (uintptr_t)a.ps1 | (uintptr_t)a.ps2) & amask) return AKV_ERR_UNSUPPORTED;
  const uint4* bop = (const uint4*)((const float*)rot_prep + (size_t)2 * d * d);
  const int64_t n_total = (paged && a.x2) ? 2 * a.n : a.n;
  const int cus = akv_cached_cu_count() > 0 ? akv_cached_cu_count() : 256;
  // Calls that give a CU at most one step of 64 rows (float32: 32), or two where the rows are checked slot by slot or have 3 bits,
  // take the kernel with the matrix in registers: no 64 KB fill, and a wavefront's chain is a quarter of a row's tiles.  A second
  // or third step a CU brings the matrix in again, so the kernel above takes over at once.  A call among others, inputs in
  // turn, us, the kernel above | that one, at the last size of the rule and the next above it:
  //   paged bf16 4 bits 64 rows a CU 9.4 | 6.8, 128 10.6 | 9.7, 136 11.8 | 11.8, 192 12.3 | 12.4, 352 16.0 | 16.9
  //               3 bits 128 10.2 | 9.7, 136 11.3 | 12.0; 2 bits 128 9.7 | 9.3, 136 10.8 | 11.3
  //         f16  4 bits 128 10.1 | 9.6, 160 11.2 | 12.0; 3 bits 9.6 | 9.4, 10.7 | 11.9; 2 bits 9.3 | 9.0, 10.3 | 11.3
  //         f32  4 bits 64 9.6 | 9.0, 80 10.7 | 11.1; 3 bits 9.1 | 8.6, 10.1 | 10.8; 2 bits 8.7 | 8.2, 9.6 | 10.3
  //   flat  f16  4 bits 64 7.7 | 6.3, 68 7.7 | 8.3; 2 bits 6.9 | 5.7, 6.9 | 7.5; 3 bits 128 9.2 | 8.8, 160 10.2 | 11.2
  //         bf16 4 bits 64 8.1 | 6.5, 80 8.5 | 8.9; 2 bits 7.2 | 5.8, 7.7 | 7.9; 3 bits 128 9.7 | 9.1, 160 11.1 | 11.4
  //         f32  4 bits 32 7.3 | 5.8, 48 8.1 | 8.5; 3 bits 6.8 | 5.4, 7.7 | 8.1; 2 bits 6.3 | 5.2, 7.1 | 7.8
  // (Beyond, several steps a workgroup with rows of the next on their way were faster here and there, paged bf16 4 bits 512 rows a CU 20.2 | 19.0,
  // and slower as often, 384 16.5 | 17.0, 2 bits 15.3 | 16.5, 768 26.6 | 28.1: nothing to go by.)
  // The fewest share each step of 16 rows among eight wavefronts, that | this form: 16 rows a CU paged f16 4 bits 4.9 | 4.7, bf16
  // 5.1 | 5.1 (12 rows 5.1 | 5.0), but 3 bits 4.4 | 4.5, 4.5 | 4.9, 2 bits 4.1 | 4.3, 4.2 | 4.7; flat f16 4.8 | 4.2, bf16 4.9 | 4.5, 3 bits
  // 4.2 | 4.0, 2 bits 4.1 | 3.9; 24 rows flat f16 4 bits 7.9 | 8.8.
  const bool plain = getenv("AKV_ENCODE_NO_SPLIT") != nullptr;
  const bool split = x_dtype != AKV_F32 && n_total <= em_split_rows(bits, paged) * (int64_t)cus && !plain;
  const int64_t most = (x_dtype == AKV_F32 ? 32 : 64) * (int64_t)cus * (paged || (bits == 3 && x_dtype != AKV_F32) ? 2 : 1);
  if (n_total <= most && !split && !plain && er_fits(a, paged, n_total)) return er_run(a, paged, x_dtype, bits, bop, n_total, cus, stream);
  const int rows_per_step = (x_dtype == AKV_F32 || split) ? 16 : EM_ROWS;
  const int64_t steps = (n_total + rows_per_step - 1) / rows_per_step;
  // steps are dealt round-robin over workgroups first, so a small call (one serving step) spreads
  // over as many CUs as it has steps instead of filling the wavefronts of a few
  const int grid = (int)(steps < cus ? steps : cus);
#define EM_LAUNCH_MT(BB, PG, DT, DR, MM)                                                              \
  do {                                                                                               \
    static bool configured = false;                                                                  \
    if (!configured) {                                                                               \
      AKV_HIP(hipFuncSetAttribute((const void*)akv_encode_mfma_kernel<BB, PG, DT, DR, MM>,            \
                                  hipFuncAttributeMaxDynamicSharedMemorySize, EM_LDS_BYTES));        \
      configured = true;                                                                             \
    }                                                                                                \
    AKV_LAUNCH_TIMED((akv_encode_mfma_kernel<BB, PG, DT, DR, MM>), grid, EM_THREADS, EM_LDS_BYTES, stream, a, bop); \
  } while (0)
#define EM_LAUNCH(BB, PG, DT, DR)                                                                     \
  do {                                                                                               \
    if (split && em_launch_split<BB, PG, DT, DR>(grid, stream, a, bop)) break;                       \
    EM_LAUNCH_MT(BB, PG, DT, DR, (DT == AKV_F32 ? 1 : EM_MT));                                        \
  } while (0)
#define EM_LAUNCH_DT(BB, PG, DR) do { if (x_dtype == AKV_F16) EM_LAUNCH(BB, PG, AKV_F16, DR); else if (x_dtype == AKV_BF16) EM_LAUNCH(BB, PG, AKV_BF16, DR); else EM_LAUNCH(BB, PG, AKV_F32, DR); } while (0)
  // flat rows whose byte offsets stay below 2^31 take the variant with 32-bit lane offsets
  const int64_t xbytes = x_dtype == AKV_F32 ? 4 : 2;
  const bool direct = !paged && a.n < ((int64_t)1 << 31) / (xbytes * a.xs0 > a.ps0 ? xbytes * a.xs0 : a.ps0);
  if (paged) {
    if (bits == 4) EM_LAUNCH_DT(4, true, false); else if (bits == 3) EM_LAUNCH_DT(3, true, false); else EM_LAUNCH_DT(2, true, false);
  } else if (direct && !split) {
    if (bits == 4) EM_LAUNCH_DT(4, false, true); else if (bits == 3) EM_LAUNCH_DT(3, false, true); else EM_LAUNCH_DT(2, false, true);
  } else {
    if (bits == 4) EM_LAUNCH_DT(4, false, false); else if (bits == 3) EM_LAUNCH_DT(3, false, false); else EM_LAUNCH_DT(2, false, false);
  }
#undef EM_LAUNCH_DT
#undef EM_LAUNCH
#undef EM_LAUNCH_MT
  AKV_LAUNCH_CHECK("akv_encode_mfma_kernel");
  return AKV_OK;
}
