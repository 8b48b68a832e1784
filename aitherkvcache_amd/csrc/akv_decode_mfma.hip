// MFMA decode (unpack -> centroid lookup -> inverse rotation -> x norm -> cast) for the 4-, 3- and 2-bit codecs at
// head_dim 64, 128 and 256: TurboQuant.decode, aither_kvcache/quantizer.py:168-197.
//
//   X^T[i, v] = n_v * sum_j Pi[j, i] c[code[v, j]]              v_mfma_f32_16x16x32_f16
//     A = Pi^T: a wavefront keeps the C x D slice of its C output coordinates in registers, two float16 terms (hi + lo,
//         scaled by 64), in the order its lanes take them from the prepared-rotation buffer (akv_dm_slices_kernel).  D / C
//         wavefronts share a row.
//     B = centroids of the codes: lane (v = l % 16, g = l / 16) loads quarter g of the packed row of vector v.  A code
//         BYTE (two codes) indexes a table in LDS whose entry is the float16 pair (c[a], c[b]), 32 times, and the pair of
//         remainders (c = hi + lo to ~22 bits), 32 times (address = byte * 256 + (lane & 31) * 4, built by one byte permute, and
//         128 bytes on), so look-ups do not conflict on a bank.  Both by one request of eight bytes, they landed side by side and were
//         moved to their operands, some 50 of 510 vector instructions of a step of 32 rows (K and V of 20k tokens x 8 heads to
//         bfloat16 blocks at head_dim 128: 41.2 -> 40.4 us, 3 bits 43.1 -> 42.1, head_dim 256 145.8 -> 142.0; look-ups a piece ahead of the
//         products were no faster).
//     Three products per tile: Pi_hi c_hi + Pi_hi c_lo + Pi_lo c_hi.
//   The rows of an A tile are permuted so that a lane ends up with eight neighbouring coordinates of ONE row from two tiles:
//   it needs one norm and one address per vector, and the four lanes of a vector write 64 neighbouring bytes per store.
//
// 3-bit and 2-bit rows are spread to one code per nibble in registers (akv_nibble.h) and take the same table; the
// coordinate order that the spreading leaves is matched when the matrix is loaded.
//
// What bounds it: the loop, 48 products of 16 cycles and some 210 vector instructions of four per 16 rows of head_dim 128
// and wavefront at two wavefronts a SIMD, and the trips to memory around it.
// Flat rows at head_dim 128 (us; the matrix in LDS, 64 KB read per 32 rows | split from the float32 matrix in every launch |
// as it is now): 4-bit to float16, 4,096 rows 10.2 | 9.5 | 5.9, 65,536 rows 14.6 | 16.9 | 13.1, 2^20 rows 110 | 110 | 105; 3-bit
// 2^20 115 | 115 | 109; 4-bit to float32 2^20 156 | 183 | 126.  2^20 rows at head_dim 64, 3 bits: 511 on the vector kernel, 35.
// K and V of 17k tokens x 8 heads at head_dim 128: 72 to 75 us as two launches with the matrix in LDS, 42 with the slice split
// in the launch (53 with block ids widened to 64 bits where they are loaded, a wait per load), 40 as it is now.  6,290 tokens x
// 8 heads at head_dim 256 784 us on the vector kernel, 53; 20,936 tokens x 16 heads at head_dim 64, 3 bits, 385 and 34 us.
// No barrier after the set-up: the wavefronts of a row only share cache lines.
#include "akv_common.h"
#include "akv_nibble.h"

typedef _Float16 dm_half8 __attribute__((ext_vector_type(8)));
typedef float dm_float4 __attribute__((ext_vector_type(4)));
typedef float dm_float2 __attribute__((ext_vector_type(2)));
typedef _Float16 dm_half2 __attribute__((ext_vector_type(2)));
typedef __bf16 dm_bf162 __attribute__((ext_vector_type(2)));
typedef uint32_t dm_u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) const uint32_t dm_lds_cu32;
typedef __attribute__((address_space(3))) dm_u32x4 dm_lds_u128;

#define DM_WAVES 8
#define DM_THREADS (DM_WAVES * 64)
#define DM_MT 2
#define DM_ROWS (16 * DM_MT)
#define DM_PSCALE 64.f
#define DM_LDS_BYTES 65536           // 256 entries x 32 copies x {hi pair, lo pair}

template <int D, int BITS> struct dm_cfg {
  static constexpr int C = D == 256 ? 32 : 64;              // output coordinates of a wavefront (its matrix slice: 64 to 128 registers)
  static constexpr int CW = D / C;                          // wavefronts of a row
  static constexpr int RG = DM_WAVES / CW;                  // row groups of a workgroup
  static constexpr int NT = C / 16, KS = D / 32;
  static constexpr int QB = D * BITS / 32;                  // bytes of a quarter row
  static constexpr int RAW = BITS == 3 && D == 64 ? 2 : QB / 4;   // dwords a lane loads of it
};

// Operand of the inverse rotation in the attention kernels (head_dim 128), stored after the encode operand in the
// prepared-rotation buffer
__global__ __launch_bounds__(256) void akv_dm_prepare_kernel(const float* __restrict__ Pi, uint4* __restrict__ bop) {
  const int t = blockIdx.x * 256 + threadIdx.x;      // (nt, ks, lane): 2048 threads
  const int lane = t & 63, ks = (t >> 6) & 3, nt = t >> 8;
  const int col = lane & 15, g = lane >> 4;
  const int i = 8 * col + nt;
  uint32_t hi[4], lo[4];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float v = Pi[(size_t)(32 * g + 8 * ks + e) * 128 + i] * DM_PSCALE;
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

int akv_prepare_decode_mfma(const float* rotation, int d, void* prep, hipStream_t stream) {
  if (d != 128) return AKV_OK;
  uint4* bop = (uint4*)((char*)prep + AKV_PREP_DECODE_OFFSET(d));
  akv_dm_prepare_kernel<<<8, 256, 0, stream>>>(rotation, bop);
  AKV_LAUNCH_CHECK("akv_dm_prepare_kernel");
  return AKV_OK;
}

// Operand of the decode kernel: Pi^T in tiles of 16 output coordinates, [hi | lo][tile][piece][lane] x 16 bytes.  Lane (m, g)
// of piece h holds contracted coordinates (D / 4) g + 8 h + 0 .. 7 of the tile's row m, output coordinate dm_coordinate.
__host__ __device__ constexpr int dm_coordinate(int tile, int m) {
  return 32 * (tile >> 1) + 8 * (m >> 2) + 4 * (tile & 1) + (m & 3);   // a lane's rows 4 g + i of two tiles are eight neighbours
}
__global__ __launch_bounds__(256) void akv_dm_slices_kernel(const float* __restrict__ Pi, int d, const akv_prep_scale* __restrict__ scale, uint4* __restrict__ slices) {
  const int pieces = d / 32, n = d * d / 8, t = blockIdx.x * 256 + threadIdx.x;      // (tile, piece, lane)
  if (t >= n) return;
  const int lane = t & 63, h = (t >> 6) % pieces, tile = (t >> 6) / pieces;
  const int i = dm_coordinate(tile, lane & 15), k0 = (d / 4) * (lane >> 4) + 8 * h;
  uint32_t hi[4] = {0u, 0u, 0u, 0u}, lo[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float v = Pi[(size_t)(k0 + e) * d + i] * scale->down * DM_PSCALE;
    const __half hh = __float2half_rn(v);
    hi[e >> 1] |= (uint32_t)__half_as_ushort(hh) << (16 * (e & 1));
    lo[e >> 1] |= (uint32_t)__half_as_ushort(__float2half_rn(v - __half2float(hh))) << (16 * (e & 1));
  }
  slices[t] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
  slices[n + t] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
}
int akv_prepare_decode_slices(const float* rotation, int d, void* prep, hipStream_t stream) {
  if (!(d == 64 || d == 128 || d == 256)) return AKV_OK;
  akv_dm_slices_kernel<<<(d * d / 8 + 255) / 256, 256, 0, stream>>>(rotation, d, (const akv_prep_scale*)((char*)prep + AKV_PREP_SCALE_OFFSET(d)), (uint4*)((char*)prep + AKV_PREP_SLICES_OFFSET(d)));
  AKV_LAUNCH_CHECK("akv_dm_slices_kernel");
  return AKV_OK;
}

// quarter g of a packed row.  (3-bit, head_dim 64: six bytes, read as the two dwords of the row that hold them)
template <int D, int BITS>
__device__ __forceinline__ void dm_load_quarter(const uint8_t* row, int g, uint32_t (&w)[dm_cfg<D, BITS>::RAW]) {
  constexpr int RAW = dm_cfg<D, BITS>::RAW, QB = dm_cfg<D, BITS>::QB;
  const uint32_t* p = (const uint32_t*)(row + (QB % 4 ? (QB * g & ~3) : QB * g));
  if constexpr (RAW == 1) {
    w[0] = p[0];
  } else if constexpr (RAW == 2) {
    const uint2 t = *(const uint2*)p;
    w[0] = t.x; w[1] = t.y;
  } else if constexpr (RAW % 4 == 0) {
#pragma unroll
    for (int i = 0; i < RAW; i += 4) {
      const uint4 t = *(const uint4*)(p + i);
      w[i] = t.x; w[i + 1] = t.y; w[i + 2] = t.z; w[i + 3] = t.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < RAW; ++i) w[i] = p[i];
  }
}
// one code per nibble: dword st, byte b, nibble lo holds coordinate mf_kcoord<BITS>(st, b, lo) of the quarter
template <int D, int BITS>
__device__ __forceinline__ void dm_spread(const uint32_t (&w)[dm_cfg<D, BITS>::RAW], int g, uint32_t (&kw)[dm_cfg<D, BITS>::KS]) {
  constexpr int KS = dm_cfg<D, BITS>::KS;
  if constexpr (BITS == 4) {
#pragma unroll
    for (int i = 0; i < KS; ++i) kw[i] = w[i];
  } else if constexpr (BITS == 2) {
#pragma unroll
    for (int i = 0; i < KS / 2; ++i) { kw[2 * i] = w[i] & 0x33333333u; kw[2 * i + 1] = (w[i] >> 2) & 0x33333333u; }
  } else if constexpr (D == 64) {
    // bytes 2 (g % 2) .. + 5 of the eight
    const uint32_t lo = (g & 1) ? (w[0] >> 16) | (w[1] << 16) : w[0], hi = (g & 1) ? w[1] >> 16 : w[1];
    kw[0] = mf_spread3(__builtin_amdgcn_perm(lo, lo, 0x0c000102u));
    kw[1] = mf_spread3(__builtin_amdgcn_perm(hi, lo, 0x0c030405u));
  } else {
#pragma unroll
    for (int i = 0; i < KS / 4; ++i) {
      const uint32_t part[4] = {w[3 * i], w[3 * i + 1], w[3 * i + 2], 0u};
      uint32_t out[4];
      mf_spread_row<3>(part, out);
#pragma unroll
      for (int q = 0; q < 4; ++q) kw[4 * i + q] = out[q];
    }
  }
}

// BLOCKS = false: n contiguous rows (TurboQuant.decode).  BLOCKS = true: the rows are the (position, head) entries of the
// cache blocks listed in a.slots; every listed block that exists is decoded into the block of the same index of the
// output buffer (the batch decompress of aither_kvcache/vllm/backend.py:1040-1091 without its gather / unique / scatter
// passes).  An entry equal to the one before it is not decoded again: the padding of a block table is such a run.
// With a.packed2 the rows of a second tensor (V) follow those of the first.  WIDE: strides of a block beyond 32 bits or inside a
// block beyond 24 (a cache whose heads or blocks lie further apart than its rows), all offsets in 64.
template <int D, int BITS, int ODT, bool BLOCKS, bool WIDE>
__global__ __launch_bounds__(DM_THREADS) void akv_decode_mfma_kernel(akv_gen_args a, const uint4* __restrict__ slices) {
  typedef dm_cfg<D, BITS> cfg;
  constexpr int C = cfg::C, CW = cfg::CW, RG = cfg::RG, NT = cfg::NT, KS = cfg::KS, RAW = cfg::RAW;
  typedef typename akv_elem<ODT>::type out_t;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  const int cw = wave % CW, rg = wave / CW;
  const uint32_t n_one = (uint32_t)a.n, n_total = BLOCKS && a.packed2 ? 2u * n_one : n_one;
  const uint32_t steps = (n_total + DM_ROWS - 1) / DM_ROWS, stride = gridDim.x * RG;
  const uint32_t per_blk = BLOCKS ? (uint32_t)a.block_size * (uint32_t)a.heads : 1u, heads = BLOCKS ? (uint32_t)a.heads : 1u;
  const uint32_t most_blocks = (uint32_t)a.max_blocks;
  const uint32_t per_r = 0xffffffffu / per_blk, heads_r = 0xffffffffu / heads;

  // ---- rows: block ids two steps ahead, codes and norms one step ahead
  uint32_t id[DM_MT][2], before[DM_MT][2];    // of a block and of the one listed before it: low and high word, or the same word twice
  uint32_t place[DM_MT];                      // position and head inside the block
  uint32_t raw[DM_MT][RAW];
  float nrm[DM_MT];
  out_t* dst[DM_MT];                          // null: nothing to write
  const uint32_t* ids = (const uint32_t*)a.slots;
  const uint32_t wide = a.slot_itype == AKV_I64 ? 1u : 0u;
  auto fetch_ids = [&](uint32_t step) {
    if constexpr (BLOCKS) {
#pragma unroll
      for (int mt = 0; mt < DM_MT; ++mt) {
        uint32_t n = min(step * DM_ROWS + 16 * mt + col, n_total - 1);
        if (n >= n_one) n -= n_one;
        const uint32_t li = akv_div32(n, per_blk, per_r, place[mt]);
        // (words as they lie: widened to 64 bits here, each of the loads was waited for on its own)
        const uint32_t at = li << wide, prev = (li - min(li, 1u)) << wide;
        id[mt][0] = ids[at]; id[mt][1] = ids[at + wide];
        before[mt][0] = ids[prev]; before[mt][1] = ids[prev + wide];
      }
    }
  };
  auto fetch_rows = [&](uint32_t step) {
#pragma unroll
    for (int mt = 0; mt < DM_MT; ++mt) {
      const uint32_t at = step * DM_ROWS + 16 * mt + col, n = min(at, n_total - 1);
      const bool second = BLOCKS && n >= n_one;
      uint64_t po, no, oo;
      bool live = true;          // (flat: a row past the end is the last one, stored once more)
      if constexpr (BLOCKS) {
        live = at < n_total;
        uint32_t head;
        const uint32_t pos = akv_div32(place[mt], heads, heads_r, head);
        const bool first = n - (second ? n_one : 0u) < per_blk;
        live = live && (wide ? id[mt][1] == 0u : (int32_t)id[mt][0] >= 0) && id[mt][0] < most_blocks;
        live = live && (first || id[mt][0] != before[mt][0] || id[mt][1] != before[mt][1]);
        const uint32_t blk = live ? id[mt][0] : 0u;                 // (a row of block 0 is read and dropped)
        if constexpr (WIDE) {
          po = (uint64_t)blk * (uint64_t)a.ps0 + (uint64_t)pos * (uint64_t)a.ps1 + (uint64_t)head * (uint64_t)a.ps2;
          no = (uint64_t)blk * (uint64_t)a.ns0 + (uint64_t)pos * (uint64_t)a.ns1 + (uint64_t)head * (uint64_t)a.ns2;
          oo = (uint64_t)blk * (uint64_t)a.os0 + (uint64_t)pos * (uint64_t)a.os1 + (uint64_t)head * (uint64_t)a.os2;
        } else {
          po = (uint64_t)blk * (uint32_t)a.ps0 + (__umul24(pos, (uint32_t)a.ps1) + __umul24(head, (uint32_t)a.ps2));
          no = (uint64_t)blk * (uint32_t)a.ns0 + (__umul24(pos, (uint32_t)a.ns1) + __umul24(head, (uint32_t)a.ns2));
          oo = (uint64_t)blk * (uint32_t)a.os0 + (__umul24(pos, (uint32_t)a.os1) + __umul24(head, (uint32_t)a.os2));
        }
      } else {
        po = (uint64_t)n * (uint32_t)a.ps0; no = n; oo = (uint64_t)n * (uint32_t)a.os0;
      }
      dm_load_quarter<D, BITS>((second ? a.packed2 : a.packed) + po, g, raw[mt]);
      nrm[mt] = (second ? a.norms2 : a.norms)[no];
      dst[mt] = live ? (out_t*)(second ? a.out2 : a.out) + oo : nullptr;
    }
  };
  uint32_t step = (uint32_t)rg * gridDim.x + blockIdx.x;
  fetch_ids(step);

  // ---- matrix slice, as prepared; float32 rows are stored four neighbouring coordinates a lane and tile, so there row m of
  // tile nt is coordinate 16 nt + m, wherever the operand has it
  dm_half8 Ah[NT][KS], Al[NT][KS];
  {
    const uint4* hi = slices + (size_t)(C / 16 * cw) * (KS * 64);
    const uint4* lo = hi + (D / 16) * (KS * 64);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int at = ODT == AKV_F32 ? (2 * (nt >> 1) + ((col >> 2) & 1)) * (KS * 64) + 16 * g + 4 * (2 * (nt & 1) + (col >> 3)) + (col & 3)
                                    : nt * (KS * 64) + lane;
#pragma unroll
      for (int ks = 0; ks < KS; ks += 2) {            // 16 neighbouring coordinates, in the order a row's codes are spread
        union { uint4 u[2]; _Float16 h[16]; } ph, pl;
        ph.u[0] = hi[at + ks * 64]; ph.u[1] = hi[at + (ks + 1) * 64];
        pl.u[0] = lo[at + ks * 64]; pl.u[1] = lo[at + (ks + 1) * 64];
#pragma unroll
        for (int k1 = 0; k1 < 2; ++k1)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            Ah[nt][ks + k1][e] = ph.h[mf_kcoord<BITS>(k1, e >> 1, e & 1)];
            Al[nt][ks + k1][e] = pl.h[mf_kcoord<BITS>(k1, e >> 1, e & 1)];
          }
      }
    }
  }

  // ---- table; the scale brings the largest level to [2^9, 2^10): no remainder that matters is a float16 subnormal
  float inv_cs;
  {
    constexpr int LM = (1 << BITS) - 1;                // nibble values above the top level do not occur
    const int e = threadIdx.x >> 1, half = threadIdx.x & 1;
    const float r0 = a.table[(e >> 4) & LM], r1 = a.table[e & LM];
    float mx = 0.f;
    for (int v = 0; v <= LM; ++v) mx = fmaxf(mx, fabsf(a.table[v]));
    const uint32_t ex = min(max((__float_as_uint(mx) >> 23) & 0xffu, 12u), 250u);
    const float cs = __uint_as_float((254u - ex) << 23) * 512.f;
    inv_cs = __uint_as_float(ex << 23) * (1.f / 512.f / DM_PSCALE) * ((const akv_prep_scale*)((const char*)slices + (size_t)4 * D * D))->up;
    // the code of the even coordinate is the high nibble (packing.py:13-23) and goes to the low half of the pair
    const float c0 = r0 * cs, c1 = r1 * cs;
    const __half h0 = __float2half_rn(c0), h1 = __float2half_rn(c1);
    const __half l0 = __float2half_rn(c0 - __half2float(h0)), l1 = __float2half_rn(c1 - __half2float(h1));
    const uint32_t hi = (uint32_t)__half_as_ushort(h0) | ((uint32_t)__half_as_ushort(h1) << 16);
    const uint32_t lo = (uint32_t)__half_as_ushort(l0) | ((uint32_t)__half_as_ushort(l1) << 16);
    // (the dynamic LDS block is the kernel's only LDS object: its offsets are LDS addresses)
#pragma unroll
    for (int i = 0; i < 8; ++i)      // (each entry starts with another of its pieces: sixteen lanes then write to all banks, not to two
      // groups: K and V of 4 x 500 tokens of 8 heads 10.5 -> 9.2 us)
      *(dm_lds_u128*)(uintptr_t)(uint32_t)(e * 256 + half * 128 + ((i + e) & 7) * 16) = half ? (dm_u32x4){lo, lo, lo, lo} : (dm_u32x4){hi, hi, hi, hi};
  }

  __syncthreads();
  const uint32_t copy = (uint32_t)(lane & 31) * 4u;

  if (step >= steps) return;
  uint32_t kw[DM_MT][KS];
  float nv[DM_MT];
  out_t* orow[DM_MT];
  auto take = [&]() {
#pragma unroll
    for (int mt = 0; mt < DM_MT; ++mt) {
      dm_spread<D, BITS>(raw[mt], g, kw[mt]);
      nv[mt] = nrm[mt];
      orow[mt] = dst[mt];
    }
  };
  auto ahead = [&](uint32_t k) { return min(step + k * stride, steps - 1); };      // (past the end: the last step once more)
  fetch_rows(step);
  fetch_ids(ahead(1));
  take();
  fetch_rows(ahead(1));
  fetch_ids(ahead(2));
  // (the slice is waited for here: left to its first use, in the loop, the wait would be for the stores of the step before too)
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(Ah[nt][ks]), "+v"(Al[nt][ks]));
  auto one_step = [&]() __attribute__((always_inline)) {
    dm_float4 acc[DM_MT][NT];
    if (!BLOCKS || __builtin_amdgcn_ballot_w64(orow[0] != nullptr || orow[DM_MT - 1] != nullptr) != 0) {
#pragma unroll
      for (int mt = 0; mt < DM_MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = (dm_float4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        union { uint32_t u[4]; dm_half8 h; } ch[DM_MT], cl[DM_MT];
#pragma unroll
        for (int mt = 0; mt < DM_MT; ++mt)
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            uint32_t at = __builtin_amdgcn_perm(kw[mt][ks], copy, 0x0c020400u + ((uint32_t)b << 8));
            ch[mt].u[b] = *(dm_lds_cu32*)(uintptr_t)at;
            asm("" : "+v"(at));       // (seen as one place and another, the two would be read by one request into neighbouring registers)
            cl[mt].u[b] = *(dm_lds_cu32*)(uintptr_t)(at + 128u);
          }
        // (term by term: products in a row do not wait for each other's sum)
#pragma unroll
        for (int term = 0; term < 3; ++term)
#pragma unroll
          for (int mt = 0; mt < DM_MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
              acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(term == 2 ? Al[nt][ks] : Ah[nt][ks], term == 1 ? cl[mt].h : ch[mt].h, acc[mt][nt], 0, 0, 0);
      }
    }
    // The next rows are taken, and those after them requested, before this step's stores: loads and stores complete in one
    // order, and the stores depend on a condition, so a wait behind them is a wait for the stores themselves.
    __builtin_amdgcn_sched_barrier(0);
    out_t* now[DM_MT];
    float nvn[DM_MT];
#pragma unroll
    for (int mt = 0; mt < DM_MT; ++mt) { now[mt] = orow[mt]; nvn[mt] = nv[mt]; }
    take();
    fetch_rows(ahead(2));
    fetch_ids(ahead(3));
    __builtin_amdgcn_sched_barrier(0);
    // ---- x norm, cast (the reference multiplies the float32 rotated vector by the norm and then casts): lane (v, g)
    // holds rows 4 g + i of every tile
#pragma unroll
    for (int mt = 0; mt < DM_MT; ++mt) {
      if (BLOCKS && now[mt] == nullptr) continue;
      if constexpr (ODT == AKV_F32 && !BLOCKS) {
        // Neighbouring lanes exchange half of what they hold: eight lanes then write 128 bytes of one row, a whole cache line
        // that need not stay in the L2 cache.  (2^20 rows of 128: 124 us; 139 without the hint, 177 as 64-byte pieces, 158 so
        // with the hint.  A block-wise row may have nothing to write beside one that has: there the pieces stay.)
        const bool odd = col & 1;
        const uint64_t mine = (uint64_t)(uintptr_t)now[mt];
        const uint64_t theirs = (uint64_t)akv_dpp_u32<0xB1>((uint32_t)mine) | ((uint64_t)akv_dpp_u32<0xB1>((uint32_t)(mine >> 32)) << 32);
        float* const r0 = (float*)(uintptr_t)(odd ? theirs : mine) + C * cw + 4 * g + (odd ? 16 : 0);      // the even lane's row, then the odd one's
        float* const r1 = (float*)(uintptr_t)(odd ? mine : theirs) + C * cw + 4 * g + (odd ? 16 : 0);
#pragma unroll
        for (int nt = 0; nt < NT; nt += 2) {
          const dm_float4 y0 = acc[mt][nt] * inv_cs * nvn[mt], y1 = acc[mt][nt + 1] * inv_cs * nvn[mt];
          dm_float4 w0, w1;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float give = odd ? y0[i] : y1[i];
            const float got = __uint_as_float(akv_dpp_u32<0xB1>(__float_as_uint(give)));
            w0[i] = odd ? got : y0[i];
            w1[i] = odd ? y1[i] : got;
          }
          __builtin_nontemporal_store(w0, (dm_float4*)(r0 + 16 * nt));
          __builtin_nontemporal_store(w1, (dm_float4*)(r1 + 16 * nt));
        }
      } else if constexpr (ODT == AKV_F32) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const dm_float4 y = acc[mt][nt] * inv_cs;
          *(float4*)(now[mt] + C * cw + 16 * nt + 4 * g) = make_float4(y.x * nvn[mt], y.y * nvn[mt], y.z * nvn[mt], y.w * nvn[mt]);
        }
      } else {
#pragma unroll
        for (int nt = 0; nt < NT; nt += 2) {
          uint32_t w[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const dm_float2 v = {acc[mt][nt + (q >> 1)][2 * (q & 1)] * inv_cs * nvn[mt], acc[mt][nt + (q >> 1)][2 * (q & 1) + 1] * inv_cs * nvn[mt]};
            // (one conversion instruction per pair, to nearest even; element by element the bfloat16 one was six and a branch)
            if constexpr (ODT == AKV_F16) w[q] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, dm_half2));
            else w[q] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, dm_bf162));
          }
          *(uint4*)(now[mt] + C * cw + 16 * nt + 8 * g) = make_uint4(w[0], w[1], w[2], w[3]);
        }
      }
    }
  };
  // (flat: the first step stands before the loop, so that the stores of the step before are outstanding on every way into it; else
  // the wait for a step's rows, which are older, is one for those stores too)
  if constexpr (!BLOCKS) {
    one_step();
    step += stride;
  }
  for (; step < steps; step += stride) one_step();
}

static bool dm_disabled() {
  static const bool off = [] { const char* e = getenv("AKV_DISABLE_MFMA"); return e && e[0] == '1'; }();
  return off;
}

template <int D, int BITS, int ODT, bool BLOCKS, bool WIDE>
static int dm_launch(const akv_gen_args& a, const uint4* slices, hipStream_t stream) {
  const int64_t n_total = BLOCKS && a.packed2 ? 2 * a.n : a.n, steps = (n_total + DM_ROWS - 1) / DM_ROWS;
  const int cus = akv_cached_cu_count() > 0 ? akv_cached_cu_count() : 256;
  AKV_LAUNCH_TIMED((akv_decode_mfma_kernel<D, BITS, ODT, BLOCKS, WIDE>), (int)(steps < cus ? steps : cus), DM_THREADS, DM_LDS_BYTES, stream, a, slices);
  AKV_LAUNCH_CHECK("akv_decode_mfma_kernel");
  return AKV_OK;
}
template <int D, int BITS, bool BLOCKS, bool WIDE>
static int dm_launch_dt(int out_dtype, const akv_gen_args& a, const uint4* slices, hipStream_t stream) {
  if (out_dtype == AKV_F16) return dm_launch<D, BITS, AKV_F16, BLOCKS, WIDE>(a, slices, stream);
  if (out_dtype == AKV_BF16) return dm_launch<D, BITS, AKV_BF16, BLOCKS, WIDE>(a, slices, stream);
  return dm_launch<D, BITS, AKV_F32, BLOCKS, WIDE>(a, slices, stream);
}

// returns AKV_ERR_UNSUPPORTED when the fast path does not apply (the caller then uses the general kernel)
int akv_decode_mfma_try(const akv_gen_args& a, bool blocks, int d, int bits, int out_dtype, const void* rot_prep,
                        hipStream_t stream) {
  if (dm_disabled() || !(d == 64 || d == 128 || d == 256)) return AKV_ERR_UNSUPPORTED;
  const uintptr_t palign = 3;      // multi-dword loads need dword alignment only
  if (((uintptr_t)a.packed | (uintptr_t)a.packed2 | (uintptr_t)a.ps0) & palign) return AKV_ERR_UNSUPPORTED;
  if (((uintptr_t)a.out | (uintptr_t)a.out2) & 15) return AKV_ERR_UNSUPPORTED;
  if (a.os0 & 7) return AKV_ERR_UNSUPPORTED;      // the output is written 16 bytes (8 or 4 elements) per lane
  if (blocks && (((uintptr_t)a.ps1 | (uintptr_t)a.ps2) & palign || ((a.os1 | a.os2) & 7))) return AKV_ERR_UNSUPPORTED;
  // rows are counted in 32 bits, with room for two strides past the end
  if ((a.packed2 ? 2 : 1) * a.n >= ((int64_t)1 << 31) - ((int64_t)1 << 22)) return AKV_ERR_UNSUPPORTED;
  // strides: of a block (or flat row) 32 bits, inside a block 24 bits and the sum of both products in 32; others in 64
  bool wide = false;
  const int64_t outer[3] = {a.ps0, blocks ? a.ns0 : 0, a.os0};
  for (int i = 0; i < 3; ++i) {
    if (outer[i] < 0) return AKV_ERR_UNSUPPORTED;
    wide = wide || outer[i] >= ((int64_t)1 << 32);
  }
  if (blocks) {      // (listed blocks, at most 2^31 of them, are indexed by 32-bit words)
    const int64_t in1[3] = {a.ps1, a.ns1, a.os1}, in2[3] = {a.ps2, a.ns2, a.os2}, most = (int64_t)1 << 24;
    if ((int64_t)a.block_size * a.heads >= ((int64_t)1 << 31) || a.max_blocks >= ((int64_t)1 << 32)) return AKV_ERR_UNSUPPORTED;
    wide = wide || a.block_size >= most || a.heads >= most;
    for (int i = 0; i < 3; ++i) {
      if (in1[i] < 0 || in2[i] < 0) return AKV_ERR_UNSUPPORTED;
      wide = wide || in1[i] >= most || in2[i] >= most || a.block_size * in1[i] + a.heads * in2[i] >= ((int64_t)1 << 32);
    }
  }
  if (wide && !blocks) return AKV_ERR_UNSUPPORTED;
  const uint4* slices = (const uint4*)((const char*)rot_prep + AKV_PREP_SLICES_OFFSET(d));
#define DM_CASE(DD, BB)                                                                        \
  if (d == DD && bits == BB)                                                                   \
    return !blocks ? dm_launch_dt<DD, BB, false, false>(out_dtype, a, slices, stream)          \
           : wide  ? dm_launch_dt<DD, BB, true, true>(out_dtype, a, slices, stream)            \
                   : dm_launch_dt<DD, BB, true, false>(out_dtype, a, slices, stream)
  DM_CASE(64, 2); DM_CASE(64, 3); DM_CASE(64, 4);
  DM_CASE(128, 2); DM_CASE(128, 3); DM_CASE(128, 4);
  DM_CASE(256, 2); DM_CASE(256, 3); DM_CASE(256, 4);
#undef DM_CASE
  return AKV_ERR_UNSUPPORTED;
}
