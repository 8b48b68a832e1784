// MFMA encode (norm -> rotate -> codebook search -> pack -> store) at head_dim 64 and 256 for float16, bfloat16 and float32
// input, flat rows or scattered through a slot mapping (K and V of a step in one launch).
//
//   Y[row, j] = sum_i X[row, i] Pi[j, i]              v_mfma_f32_16x16x32_f16, Pi the first operand
//
// Wavefront w of a workgroup owns NT times 16 output coordinates and keeps these rows of Pi in registers, split into two float16
// terms from the float32 matrix at its start.  A workgroup takes 16 MT rows at a time: its threads
// load them (four neighbouring elements each), reduce the squared norms over the lanes of a row and leave the rows in LDS;
// every wavefront multiplies all of them by its slice.  A lane then holds four neighbouring coordinates of one row: their
// codes, found by halving, are one halfword for LDS, and pairs of halfwords are stored.  Two barriers a step, the next rows
// requested before the first.  PARTS workgroups share the coordinates of a row where there are few rows: each loads and splits
// only its part of the matrix (and all of the rows).
//
// Precision: float16 rows are exact in the operand.  bfloat16 and float32 rows are scaled by the power of two that
// brings the largest element to [2^10, 2^11): bfloat16 is then exact (down to 2^-27 of the largest element), float32 is
// split into two terms like the matrix (2^-23 of the element, the product of two remainders left out).  The general
// kernel's chain of float32 sums is no closer to 64 bits.
//
// What bounds it: a decode step (192 to 768 rows) is one step per workgroup, a chain of trips to memory: matrix and rows,
// slots, stores: 11.4 us before the coordinates were shared out, 6.4 now (head_dim 256, up to 1,024 rows).  Large calls are bound
// by the search, 23 instructions a value in 4 bits.  K and V of 8,192 tokens of 8 heads in 4 bits: 82.0 us at
// head_dim 256 and 17.6 at 64, where counting with two instructions a boundary and a byte per code through LDS took 98.0 and 22.5.
#include "akv_common.h"

typedef _Float16 ew_half8 __attribute__((ext_vector_type(8)));
typedef _Float16 ew_half4 __attribute__((ext_vector_type(4)));
typedef float ew_float4 __attribute__((ext_vector_type(4)));

#define EW_PI_SCALE 1024.f
#define EW_PI_EXP 10

template <int D, int MT, int XDT, int PARTS, int NT> struct ew_cfg {
  static constexpr int DP = D / PARTS;                     // output coordinates of a workgroup
  static constexpr int WAVES = DP / (16 * NT), THREADS = WAVES * 64, ROWS = 16 * MT;
  static constexpr int TPR = D / 4;                        // threads of a row while loading
  static constexpr int PIECES = ROWS * TPR / THREADS;      // pieces of four elements a thread loads
  static constexpr int CPITCH = DP / 4 + 2;                // halfwords of codes per row in LDS
  static constexpr int KS = D / 32;
  static constexpr int PITCH = D + 8;                      // float16 per row in LDS (16 bytes more: eight rows meet all banks)
  static constexpr int NA = XDT == AKV_F32 ? 2 : 1;        // float16 terms of a row
};

// four elements of a row as they lie in memory
template <int XDT> struct ew_piece { typedef uint2 type; };
template <> struct ew_piece<AKV_F32> { typedef uint4 type; };
template <int XDT> __device__ __forceinline__ void ew_floats(const typename ew_piece<XDT>::type& r, float (&x)[4]) {
  if constexpr (XDT == AKV_F32) {
    x[0] = __uint_as_float(r.x); x[1] = __uint_as_float(r.y); x[2] = __uint_as_float(r.z); x[3] = __uint_as_float(r.w);
  } else if constexpr (XDT == AKV_BF16) {
    x[0] = __uint_as_float(r.x << 16); x[1] = __uint_as_float(r.x & 0xffff0000u);
    x[2] = __uint_as_float(r.y << 16); x[3] = __uint_as_float(r.y & 0xffff0000u);
  } else {
    union { uint2 u; ew_half4 h; } cv;
    cv.u = r;
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = (float)cv.h[i];
  }
}

template <int D, int BITS, int XDT, bool PAGED, int MT, int PARTS, int NT>
__global__ __launch_bounds__((ew_cfg<D, MT, XDT, PARTS, NT>::THREADS)) void akv_encode_wide_kernel(akv_gen_args a, const float* __restrict__ Pi, const akv_prep_scale* __restrict__ scale) {
  typedef ew_cfg<D, MT, XDT, PARTS, NT> cfg;
  typedef typename ew_piece<XDT>::type piece_t;
  constexpr int ROWS = cfg::ROWS, TPR = cfg::TPR, KS = cfg::KS, PITCH = cfg::PITCH, NA = cfg::NA, THREADS = cfg::THREADS, PIECES = cfg::PIECES, DP = cfg::DP;
  constexpr int NB = (1 << BITS) - 1;
  constexpr int XB = XDT == AKV_F32 ? 4 : 2;
  __shared__ __align__(16) _Float16 rows[NA][ROWS][PITCH];
  __shared__ __align__(16) unsigned short codes[ROWS][cfg::CPITCH];
  __shared__ float4 info[ROWS];                            // reciprocal of the norm (NaN: not finite), exponent to put back, norm
  __shared__ int64_t dst[2][ROWS];                         // [parity of the step] address of the packed row, 0 = skip
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 15, g = lane >> 4;
  const int64_t n_total = (PAGED && a.x2) ? 2 * a.n : a.n;
  const int64_t steps = (n_total + ROWS - 1) / ROWS, first = blockIdx.x / PARTS, stride = gridDim.x / PARTS;
  const int part = PARTS > 1 ? (int)(blockIdx.x % PARTS) : 0;

  // ---- rows: thread (row, part) of piece i
  piece_t R[PIECES];
  auto fetch = [&](int64_t step) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int u = tid + i * THREADS;
      int64_t n = step * ROWS + u / TPR;
      if (n >= n_total) n = n_total - 1;                   // past the end: loaded, not stored
      const bool second = PAGED && n >= a.n;
      if (second) n -= a.n;
      int64_t off;
      if constexpr (PAGED) {
        const uint32_t tok = (uint32_t)n / (uint32_t)a.heads, head = (uint32_t)n - tok * (uint32_t)a.heads;
        off = (int64_t)tok * a.xs0 + (int64_t)head * a.xs1;
      } else {
        off = n * a.xs0;
      }
      R[i] = *(const piece_t*)((const char*)(second ? a.x2 : a.x) + XB * (off + 4 * (u % TPR)));
    }
  };
  fetch(first);

  const float pi_scale = EW_PI_SCALE * scale->down;
  const int pi_exp = scale->k - EW_PI_EXP;
  // ---- the wavefront's NT slices of Pi: lane (col, g) holds row DP part + 16 (NT wave + nt) + col, elements 32 ks + 8 g + e
  ew_half8 Bh[NT][KS], Bl[NT][KS];
#pragma unroll
  for (int k = 0; k < NT * KS; ++k) {
    const int nt = k / KS, ks = k % KS;
    const float4* p = (const float4*)(Pi + (size_t)(DP * part + 16 * (NT * wave + nt) + col) * D + 32 * ks + 8 * g);
    const float4 p0 = p[0], p1 = p[1];
    const float v[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float s = v[e] * pi_scale;
      const _Float16 h = (_Float16)s;
      Bh[nt][ks][e] = h;
      Bl[nt][ks][e] = (_Float16)(s - (float)h);
    }
  }
  float bnd[NB];
#pragma unroll
  for (int k = 0; k < NB; ++k) bnd[k] = a.table[k];
  akv_sort_boundaries(bnd);

  int par = 0;
  for (int64_t step = first; step < steps; step += stride, par ^= 1) {
    // ---- norm, conversion, rows into LDS
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int u = tid + i * THREADS, row = u / TPR, at = u % TPR;
      float x[4];
      ew_floats<XDT>(R[i], x);
      float ss = 0.f, mx = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        ss = fmaf(x[e], x[e], ss);
        mx = fmaxf(mx, fabsf(x[e]));
      }
      ss += akv_lane_xor<1>(ss); ss += akv_lane_xor<2>(ss); ss += akv_lane_xor<4>(ss); ss += akv_lane_xor<8>(ss);
      mx = fmaxf(mx, akv_lane_xor<1>(mx)); mx = fmaxf(mx, akv_lane_xor<2>(mx));
      mx = fmaxf(mx, akv_lane_xor<4>(mx)); mx = fmaxf(mx, akv_lane_xor<8>(mx));
      if constexpr (TPR == 64) {
        ss += akv_lane_xor<16>(ss); ss += akv_lane_xor<32>(ss);
        mx = fmaxf(mx, akv_lane_xor<16>(mx)); mx = fmaxf(mx, akv_lane_xor<32>(mx));
      }
      // a row with a NaN (its sum is NaN) or an infinity rotates to NaN everywhere; a finite row whose squares overflow
      // has norm inf and rotates to zero
      const bool bad = ss != ss || !(mx < INFINITY);
      int put_back = pi_exp;
      union { ew_half4 h; uint2 u; } hi, lo;
      if constexpr (XDT == AKV_F16) {
        hi.u = R[i];
      } else {
        const int ef = bad ? 127 : (int)(__float_as_uint(mx) >> 23);
        const int sef = min(254, 264 - ef);
        const float sc = __uint_as_float((uint32_t)sef << 23);         // 2^(sef - 127)
        put_back += 127 - sef;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float s = x[e] * sc;
          hi.h[e] = (_Float16)s;
          lo.h[e] = (_Float16)(s - (float)hi.h[e]);
        }
      }
      *(uint2*)&rows[0][row][4 * at] = hi.u;
      if constexpr (NA == 2) *(uint2*)&rows[NA - 1][row][4 * at] = lo.u;
      if (at == 0) {
        const float nrm = sqrtf(ss);
        info[row] = make_float4(bad ? NAN : 1.f / (nrm + 1e-10f), __int_as_float(put_back), nrm, 0.f);
      }
    }
    // ---- thread r resolves row r of the step
    float* norm_at = nullptr;
    if (tid < ROWS) {
      int64_t n = step * ROWS + tid, dp = 0;
      if (n < n_total) {
        const bool second = PAGED && n >= a.n;
        if (second) n -= a.n;
        uint8_t* pb = second ? a.packed2 : a.packed;
        float* nb = second ? a.norms2 : a.norms;
        if constexpr (PAGED) {
          const uint32_t tok = (uint32_t)n / (uint32_t)a.heads, head = (uint32_t)n - tok * (uint32_t)a.heads;
          const int64_t slot = akv_load_index(a.slots, a.slot_itype, tok);
          if (slot >= 0) {
            const int64_t blk = slot / a.block_size, pos = slot - blk * a.block_size;
            if (blk < a.max_blocks) {
              dp = (int64_t)(uintptr_t)(pb + blk * a.ps0 + pos * a.ps1 + (int64_t)head * a.ps2);
              norm_at = nb + blk * a.ns0 + pos * a.ns1 + (int64_t)head * a.ns2;
            }
          }
        } else {
          dp = (int64_t)(uintptr_t)(pb + n * a.ps0);
          norm_at = nb + n;
        }
      }
      dst[par][tid] = dp;
    }
    if (step + stride < steps) fetch(step + stride);
    __syncthreads();
    if (norm_at != nullptr && part == 0) *norm_at = info[tid].z;

    // ---- rotate and search: lane (col, g) ends up with coordinates 16 (NT wave + nt) + 4 g + i of row 16 mt + col
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      ew_float4 acc[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt] = ew_float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const ew_half8 x = *(const ew_half8*)&rows[0][16 * mt + col][32 * ks + 8 * g];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Bh[nt][ks], x, acc[nt], 0, 0, 0);
          acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Bl[nt][ks], x, acc[nt], 0, 0, 0);
        }
        if constexpr (NA == 2) {
          const ew_half8 xl = *(const ew_half8*)&rows[NA - 1][16 * mt + col][32 * ks + 8 * g];
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Bh[nt][ks], xl, acc[nt], 0, 0, 0);
        }
      }
      const float2 f = *(const float2*)&info[16 * mt + col];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        uint32_t c[2] = {0, 0};                            // first code in the top bits; NaN lies past every boundary
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = ldexpf(acc[nt][i] * f.x, __float_as_int(f.y));
        akv_append_codes<BITS>(c[0], y[0], c[1], y[2], bnd);
        akv_append_codes<BITS>(c[0], y[1], c[1], y[3], bnd);
        codes[16 * mt + col][4 * (NT * wave + nt) + g] = (unsigned short)((c[0] << (2 * BITS)) | c[1]);
      }
    }
    __syncthreads();

    // ---- store: eight codes are BITS bytes
    for (int u = tid; u < ROWS * (DP / 8); u += THREADS) {
      const int row = u / (DP / 8), at = u % (DP / 8);
      const int64_t dp = dst[par][row];
      if (dp == 0) continue;
      const uint32_t c = *(const uint32_t*)&codes[row][2 * at];
      uint8_t* p = (uint8_t*)(uintptr_t)dp + BITS * (DP / 8 * part + at);
      const uint32_t w = ((c & 0xffffu) << (4 * BITS)) | (c >> 16);
      if constexpr (BITS == 4) {
        *(uint32_t*)p = __builtin_bswap32(w);
      } else if constexpr (BITS == 2) {
        *(uint16_t*)p = (uint16_t)((w >> 8) | (w << 8));
      } else {
        p[0] = (uint8_t)(w >> 16);
        p[1] = (uint8_t)(w >> 8);
        p[2] = (uint8_t)w;
      }
    }
    // (the rows of the next step go where this one's were: read before the second barrier.  Its codes are written behind
    // its first barrier, its destinations to the other parity.)
  }
}

template <int D, int BITS, int XDT, bool PAGED, int MT, int PARTS, int NT>
static int ew_launch(const akv_gen_args& a, const float* Pi, hipStream_t stream) {
  const akv_prep_scale* scale = (const akv_prep_scale*)((const char*)Pi + AKV_PREP_SCALE_OFFSET(D));
  typedef ew_cfg<D, MT, XDT, PARTS, NT> cfg;
  const int cus = akv_cached_cu_count();
  const int64_t n_total = (PAGED && a.x2) ? 2 * a.n : a.n, steps = (n_total + cfg::ROWS - 1) / cfg::ROWS;
  const int64_t most = (int64_t)(cus > 0 ? cus : 256) * (D == 256 && PARTS == 1 ? 1 : 4) / PARTS;
  AKV_LAUNCH_TIMED((akv_encode_wide_kernel<D, BITS, XDT, PAGED, MT, PARTS, NT>), (int)(steps < most ? steps : most) * PARTS, cfg::THREADS, 0, stream, a, Pi, scale);
  AKV_LAUNCH_CHECK("akv_encode_wide_kernel");
  return AKV_OK;
}
// head_dim 256: a quarter of the coordinates per workgroup while all of these fit the chip at once (three a CU): 6.4 us up to
// 1,024 rows, 8.5 for 2,048 and 10.5 for 3,072, where one workgroup for all coordinates takes 11.2; at 4,096 rows it is
// 15.1 against 11.4.  More rows a step once every workgroup has several steps: a barrier is then shared by more products.
template <int D, int BITS, int XDT, bool PAGED>
static int ew_launch_rows(const akv_gen_args& a, const float* Pi, hipStream_t stream) {
  const int64_t n_total = (PAGED && a.x2) ? 2 * a.n : a.n;
  if constexpr (D == 256) {
    const int cus = akv_cached_cu_count();
    if (n_total <= 12 * (cus > 0 ? cus : 256)) return ew_launch<D, BITS, XDT, PAGED, 1, 4, 1>(a, Pi, stream);
    return n_total > 16384 ? ew_launch<D, BITS, XDT, PAGED, 2, 1, 2>(a, Pi, stream) : ew_launch<D, BITS, XDT, PAGED, 1, 1, 2>(a, Pi, stream);
  } else {
    return n_total > 16384 ? ew_launch<D, BITS, XDT, PAGED, 4, 1, 1>(a, Pi, stream) : ew_launch<D, BITS, XDT, PAGED, 1, 1, 1>(a, Pi, stream);
  }
}
template <int D, int BITS>
static int ew_launch_dt(int x_dtype, bool paged, const akv_gen_args& a, const float* Pi, hipStream_t stream) {
  if (x_dtype == AKV_F16) return paged ? ew_launch_rows<D, BITS, AKV_F16, true>(a, Pi, stream) : ew_launch_rows<D, BITS, AKV_F16, false>(a, Pi, stream);
  if (x_dtype == AKV_BF16) return paged ? ew_launch_rows<D, BITS, AKV_BF16, true>(a, Pi, stream) : ew_launch_rows<D, BITS, AKV_BF16, false>(a, Pi, stream);
  return paged ? ew_launch_rows<D, BITS, AKV_F32, true>(a, Pi, stream) : ew_launch_rows<D, BITS, AKV_F32, false>(a, Pi, stream);
}

// AKV_ERR_UNSUPPORTED: a shape or an alignment the general kernel takes
int akv_encode_wide_try(const akv_gen_args& a, bool paged, int x_dtype, int d, int bits, const void* rot_prep, hipStream_t stream) {
  static const bool disabled = [] { const char* e = getenv("AKV_DISABLE_MFMA"); return e && e[0] == '1'; }();
  if ((d != 64 && d != 256) || disabled) return AKV_ERR_UNSUPPORTED;
  if (paged && a.n >= ((int64_t)1 << 31)) return AKV_ERR_UNSUPPORTED;         // rows are divided by the heads in 32 bits
  // rows are read four elements at a time and written four (4-bit) or two (2-bit) bytes at a time
  const uintptr_t xa = x_dtype == AKV_F32 ? 15 : 7, pa = bits == 4 ? 3 : bits == 2 ? 1 : 0;
  const uintptr_t xb = x_dtype == AKV_F32 ? 4 : 2;
  if ((((uintptr_t)a.x | (uintptr_t)a.x2 | (uintptr_t)a.xs0 * xb | (uintptr_t)(paged ? a.xs1 : 0) * xb) & xa) != 0) return AKV_ERR_UNSUPPORTED;
  if ((((uintptr_t)a.packed | (uintptr_t)a.packed2 | (uintptr_t)a.ps0 | (uintptr_t)(paged ? a.ps1 | a.ps2 : 0)) & pa) != 0) return AKV_ERR_UNSUPPORTED;
  const float* Pi = (const float*)rot_prep;
#define EW_CASE(DD, BB) if (d == DD && bits == BB) return ew_launch_dt<DD, BB>(x_dtype, paged, a, Pi, stream)
  EW_CASE(64, 2); EW_CASE(64, 3); EW_CASE(64, 4);
  EW_CASE(256, 2); EW_CASE(256, 3); EW_CASE(256, 4);
#undef EW_CASE
  return AKV_ERR_UNSUPPORTED;
}
