// MFMA paged decode attention in which every wavefront works on its own: 4-, 3- and 2-bit caches at head_dim 64 and 256,
// and at head_dim 128 with one or two kv heads (akv_attn_wave_applicable), block_size 16 or 32.
//
// A workgroup owns a range of the global block axis (akv_attn_partition).  Its W wavefronts are laid out as
// (kv head slot) x (R shares of the tokens): wavefront (hs, r) takes chunks r, r + R, ... of 32 tokens of a segment for
// kv head hs, scores AND values, with no barrier until the segment ends; then the R partial results of a head are
// merged through LDS.  The slots are a power of two: from W / 2 + 1 kv heads on R is 1 and nothing is merged, and where only one
// share of a segment has tokens neither.  (The kernel in akv_attn_mfma.hip splits scores and values between the wavefronts of
// a fixed set of eight kv heads: one kv head -- a rank of a sharded model -- leaves seven eighths of it idle.)
//
//   scores   S^T[token, col] = sum_d Khat[token, d] Qop[d, col]         v_mfma_f32_16x16x32_f16
//            A: lane (n = l % 16, g = l / 16) owns quarter g of token n's code row; an LDS table turns a byte (two codes)
//            into (hi pair, lo pair), two look-ups side by side are the operand.  B: the rotated query, every pair
//            twice (it faces hi and lo); columns 0..7 the float16 rounding, columns 8..15 the remainder.
//   softmax  on the accumulator as it lies: lane (col, g) holds tokens 4 g .. 4 g + 3 of both tiles.
//   values   O^T[coord, col] += sum_token Vhat[token, coord] W[token, col].  The tokens a lane weighs are the tokens
//            whose look-ups it makes, so the weights are the operand without crossing a lane.  A byte is the same
//            coordinate of two tokens; columns 0..7 carry the float16 rounding of the weights, 8..15 the remainder.
//
// Precision: codebook, queries and weights are split into two float16 terms each (rounded to nearest: 2^-23 of the
// value), products are exact, sums float32; only the product of two remainders (2^-24) is left out.  The codebook and
// every query row are scaled by powers of two, and the weights are kept below 2^15 rather than 1, so that no remainder
// is a float16 subnormal that matters.
//
// One table serves keys and values: 256 entries x 8 bytes x 32 copies (a lane reads copy lane % 32: no bank conflicts).
// 2-bit codes are looked up as nibbles: two masks and a shift spread a byte of four codes, no second table.  3-bit codes are
// looked up in pairs, six bits as they lie: a group of eight codes is 24 bits, big-endian, spread to a byte a field by six
// instructions (one permute among them, which also takes the group out of unaligned bytes); the table then has 64 entries.
// 3 bits, an attention call (no write), this | the vector kernel that served 64 and 256 and the eight-slot kernel at 128: 32 heads on 8 of 64,
// 48 sequences of 512 to 8,192 tokens 56.3 | 113.2 us; 16 on 4 of 256, 24 sequences 66.7 | 141.5; 8 on 1 of 128, 48 of 1,024
// to 16,384 39.3 | 62.2; 8 on 2 of 128 52.6 | 62.3.
//
// What bounds it: the chain of trips to LDS and memory a wavefront walks, at two to four wavefronts a SIMD.  Share of the kernel's
// cycles (profiles/attn_wave_sq_counters.txt), head_dim 64, 128 and 256: address unit 71, 30 and 59 %, vector unit 49, 46 and 36,
// matrix cores 13, 16 and 18, LDS 19, 27 and 24.
#include <type_traits>

#include "akv_attn_rows.h"
#include "akv_device_once.h"

typedef _Float16 aw_half8 __attribute__((ext_vector_type(8)));
typedef _Float16 aw_half2 __attribute__((ext_vector_type(2)));
typedef float aw_float2 __attribute__((ext_vector_type(2)));
typedef float aw_float4 __attribute__((ext_vector_type(4)));
typedef uint32_t aw_u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t aw_u32x3 __attribute__((ext_vector_type(3), aligned(4)));
typedef uint32_t aw_u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) const aw_u32x2 aw_lds_cu64;
typedef __attribute__((address_space(3))) aw_u32x4 aw_lds_u128;
typedef __attribute__((address_space(3))) float aw_lds_f32;
typedef __attribute__((address_space(3))) aw_float2 aw_lds_f64;
typedef __attribute__((address_space(3))) aw_float4 aw_lds_f128;

#define AW_FRAME 15.f          // weights stay below 2^AW_FRAME
// Value norms count as at least 2^-AW_TINY in the running maximum: the plain exponentials, summed for the denominator, then
// stay below 2^(AW_TINY + AW_FRAME), and a million of them in float32.  A vector of that norm still has 2^15 times the
// smallest float16 the weights need, so only norms below some 2^-110 lose digits (a zero vector weighs nothing).  The encoders
// write none: a norm is the root of a float32 sum of squares, 0 or at least 2^-75.
#define AW_TINY 90
#define AW_WIN 32              // chunks of a wavefront served by one window of 64 block ids

template <int D, int BITS> struct aw_cfg {
  static constexpr int W = D == 64 ? 16 : 8;            // wavefronts: what their registers admit on a CU
  static constexpr int CPL = D / 16;                    // coordinates per lane of a value tile = M-tiles
  static constexpr int KS = D / 16;                     // MFMA steps of a score tile (four coordinates a lane each)
  // keys: a lane reads a quarter of a code row from both tiles of a chunk, or half of one from one tile (KHALF) where that is at
  // most sixteen bytes, and half of it is handed on
  static constexpr bool KHALF = D * BITS / 128 <= 2;
  static constexpr int KDW = KHALF ? D * BITS / 64 : D * BITS / 128;      // dwords of a request
  // values: VB bytes of codes of one token a lane (3 bits: spread to nibbles' room); a request takes twice that of one token, for
  // the lane and the one eight lanes away
  static constexpr int VB = CPL * (BITS == 3 ? 4 : BITS) / 8;
  static constexpr int VRD = BITS == 3 ? (D == 256 ? 3 : 2) : VB >= 2 ? VB / 2 : 1;      // dwords of a request
};
// LDS: table | per wavefront: 32 key norms, 32 value norms, 32 exponents of those | per wavefront: (max, sum) of eight
// heads | per wavefront: accumulators of its heads (merging only)
#define AW_NORM 65536u
#define AW_NORM_WAVE 384u
template <int W> constexpr uint32_t aw_ml_off() { return AW_NORM + W * AW_NORM_WAVE; }
template <int W> constexpr uint32_t aw_acc_off() { return aw_ml_off<W>() + W * 64u; }

struct aw_extra {
  const uint2* qop;        // [S][KVH][D / 16][64 lanes] four float16 (workspace)
  const float* fac;        // [S][QH] power of two taken out of a query row, times scale * log2 e
  const int32_t* wgdesc;   // [G][AKV_WGREC]
  int hp;                  // kv head slots of a workgroup (a power of two)
};

// ----------------------------------------------------------------------------------
// prologue: block 0 cuts the block axis, the others rotate query heads and write them in operand order (akv_attn_rows.h).
// On the vector unit (a matrix column in registers, one row a workgroup at a time) it took 9.1 us for 384 rows of 256, 7.0 now;
// 1,536 rows of 64 6.4, now 4.7.
// ----------------------------------------------------------------------------------
template <int D, int QDT>
__global__ __launch_bounds__(256) void akv_attn_wave_prologue_kernel(
    const void* __restrict__ query, int64_t qs_seq, int64_t qs_head, const float* __restrict__ Pi, const akv_prep_scale* __restrict__ scale,
    int S, int QH, int KVH, int slots, const void* context_lens, int cl_itype, int block_size, int64_t max_blocks_per_seq, int32_t* prefix,
    uint2* __restrict__ qop, float* __restrict__ fac, uint32_t* __restrict__ status, float qscale, int bits, int32_t* __restrict__ wgdesc,
    int32_t* __restrict__ seqw, int G, int shares) {
  __shared__ __align__(16) ar_rows<D, ar_terms<QDT>()> rows;
  __shared__ int32_t scratch[AKV_PART_WORDS];
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) status[0] = 0u;
    akv_attn_partition(prefix, S, G, block_size == 32 ? 1 : 2, wgdesc, seqw, scratch, context_lens, cl_itype, block_size, max_blocks_per_seq, shares, D == 64 ? 2 : 3);
    return;
  }
  ar_rotate_queries<D, QDT, false>(rows, (int)blockIdx.x - 1, (int)gridDim.x - 1, query, qs_seq, qs_head, Pi, scale, S, QH, KVH, slots, qop, fac, qscale, bits);
}

// ----------------------------------------------------------------------------------
// main kernel
// ----------------------------------------------------------------------------------
// address of a table entry: byte k of `word` * 256 + the lane's copy, one byte permute
template <int K> __device__ __forceinline__ aw_u32x2 aw_look(uint32_t lanebits, uint32_t word) {
  return *(aw_lds_cu64*)(uintptr_t)__builtin_amdgcn_perm(word, lanebits, 0x0c020400u + (K << 8));
}
__device__ __forceinline__ aw_half8 aw_operand(aw_u32x2 a, aw_u32x2 b) {
  union { uint32_t u[4]; aw_half8 h; } x;
  x.u[0] = a.x; x.u[1] = a.y; x.u[2] = b.x; x.u[3] = b.y;
  return x.h;
}
// value of the lane eight columns away in the row of sixteen, added
__device__ __forceinline__ float aw_add_cols(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128 /*row_ror:8*/, 0xf, 0xf, false));
}
// (keeps the widening of a 32-bit lane offset next to its load: scalar base + 32-bit lane offset)
__device__ __forceinline__ uint32_t aw_here(uint32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}
// N dwords that are aligned to four bytes
template <int N, int M> __device__ __forceinline__ void aw_request(uint32_t (&r)[M], const unsigned char* p) {
  static_assert(N <= M, "registers");
  if constexpr (N >= 4) {
    const uint4 t = *(const uint4*)p;
    r[0] = t.x; r[1] = t.y; r[2] = t.z; r[3] = t.w;
    if constexpr (N == 6) {
      const uint2 u = *(const uint2*)(p + 16);
      r[4] = u.x; r[5] = u.y;
    }
    if constexpr (N == 8) {
      const uint4 u = *(const uint4*)(p + 16);
      r[4] = u.x; r[5] = u.y; r[6] = u.z; r[7] = u.w;
    }
  } else if constexpr (N == 3) {
    const aw_u32x3 t = *(const aw_u32x3*)p;
    r[0] = t.x; r[1] = t.y; r[2] = t.z;
  } else if constexpr (N == 2) {
    const uint2 t = *(const uint2*)p;
    r[0] = t.x; r[1] = t.y;
  } else {
    r[0] = *(const uint32_t*)p;
  }
}
template <int I, int N, class F> __device__ __forceinline__ void aw_each_from(F& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    aw_each_from<I + 1, N>(f);
  }
}
template <int N, class F> __device__ __forceinline__ void aw_each(F f) { aw_each_from<0, N>(f); }
// N products of two look-ups each, the look-ups A products ahead.  Left to itself the compiler makes every product wait for
// look-ups requested right before it, a trip to LDS each time (decode steps: 100 contexts of 200 to 1,000 with heads of 256 59.1 -> 55.5 us;
// 2 bits 40.2 -> 38.5; one kv head of 128 33.8 -> 33.3; heads of 64 65.2 -> 64.6).
template <int A, int N, class L, class M> __device__ __forceinline__ void aw_products(L look, M product) {
  static_assert(A <= N, "look-ups ahead");
  aw_u32x2 w[A][2];
  auto first = [&](auto i) __attribute__((always_inline)) { look(i, w[i][0], w[i][1]); };
  aw_each<A>(first);
  __builtin_amdgcn_sched_barrier(0x6 /*vector and scalar arithmetic may pass*/);
  auto one = [&](auto i) __attribute__((always_inline)) {
    constexpr int I = decltype(i)::value;
    product(i, aw_operand(w[I % A][0], w[I % A][1]));
    if constexpr (I + A < N) look(std::integral_constant<int, I + A>{}, w[I % A][0], w[I % A][1]);
    __builtin_amdgcn_sched_barrier(0x6);
  };
  aw_each<N>(one);
}
// What lanes 8 p + c of a row hold of one piece each, first and second half x and y of it, the piece of token p: the half p of both
// tokens
__device__ __forceinline__ void aw_trade(uint32_t x, uint32_t y, uint32_t& first, uint32_t& second) {
  first = akv_dpp_banks_u<0x128 /*row_ror:8*/, 0xc>(x, y);
  second = akv_dpp_banks_u<0x128 /*row_ror:8*/, 0x3>(y, x);
}
// 3-bit codes: a group of eight is a big-endian word of 24 bits.  Its four fields of two codes each, one per byte (the first
// field in byte 3); and the same for two half groups of twelve bits in the halves of a word (first field in byte 1 and 3).
__device__ __forceinline__ uint32_t aw_spread12(uint32_t x) { return ((x << 2) & 0x3F003F00u) | (x & 0x003F003Fu); }
__device__ __forceinline__ uint32_t aw_spread24(uint32_t x) { return aw_spread12((x & 0xFFFu) | ((x << 4) & ~0xFFFu)); }

// the words whose bytes are table indices of lane coordinates: pairs (ta, tb) of tokens, words `wa`, `wb` of codes (3 bits: of
// fields)
template <int BITS, int N> struct aw_pairs { uint32_t w[BITS == 2 ? 4 : 2]; };
template <int BITS, int N>
__device__ __forceinline__ void aw_pair(aw_pairs<BITS, N>& p, uint32_t wa, uint32_t wb) {
  if constexpr (BITS == 3) {
    p.w[0] = (wa & 0x38383838u) | ((wb >> 3) & 0x07070707u);
    p.w[1] = ((wa << 3) & 0x38383838u) | (wb & 0x07070707u);
  } else if constexpr (BITS == 4) {
    p.w[0] = (wa & 0xF0F0F0F0u) | ((wb >> 4) & 0x0F0F0F0Fu);      // the even one of a byte's two codes
    p.w[1] = ((wa << 4) & 0xF0F0F0F0u) | (wb & 0x0F0F0F0Fu);
  } else {
    p.w[0] = ((wa >> 2) & 0x30303030u) | ((wb >> 6) & 0x03030303u);   // code 0 of a byte's four, ...
    p.w[1] = (wa & 0x30303030u) | ((wb >> 4) & 0x03030303u);
    p.w[2] = ((wa << 2) & 0x30303030u) | ((wb >> 2) & 0x03030303u);
    p.w[3] = ((wa << 4) & 0x30303030u) | (wb & 0x03030303u);
  }
}

// PACK: lanes of a row that share the eight tokens of a query head from the scores to the weights (below)
template <int D, int BITS, int PACK>
__global__ __launch_bounds__((D == 64 ? 16 : 8) * 64) void akv_attn_wave_kernel(akv_attn_args a, aw_extra x) {
  typedef aw_cfg<D, BITS> cfg;
  constexpr int W = cfg::W, CPL = cfg::CPL, KS = cfg::KS, KDW = cfg::KDW, VB = cfg::VB, VRD = cfg::VRD;
  constexpr bool KHALF = cfg::KHALF;
  constexpr int AHEAD = D == 64 ? 3 : 4;                   // products whose look-ups are under way (at head_dim 64 there are no registers for four)
  constexpr int CPB = BITS == 2 ? 4 : 2;                   // codes of a byte
  constexpr int NV = 8 / PACK;                             // tokens of a lane in the softmax
  // The dynamic LDS block is the kernel's only LDS object: its offsets are LDS addresses.
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  const uint32_t copy = (uint32_t)(lane & 31) * 8u;

  // (one argument of every cache line, requested together: left to the compiler the lines are fetched one after another, each
  // where the first of its arguments is needed)
  asm volatile("" ::"s"(a.kp), "s"(a.vp), "s"(a.block_tables), "s"(a.num_blocks), "s"(x.wgdesc));
  const int32_t* rec = x.wgdesc + (size_t)blockIdx.x * AKV_WGREC;
  const int g0 = rec[AKV_WGREC_G0], g1 = rec[AKV_WGREC_G1], s_first = rec[AKV_WGREC_SEQ];
  const int sb0_first = rec[AKV_WGREC_SB0], sb1_first = rec[AKV_WGREC_SB1], ctx_first = rec[AKV_WGREC_CTX];

  // ---- table; the scale brings the largest level to [2^9, 2^10).  At head_dim 128 it is written once every wavefront has
  // requested its first block ids, rows and queries, so that the fill and the barrier behind it run beside those trips to
  // memory; at 64 and 256 there are no registers left to hold its words until then (they would be spilled).
  constexpr int TPE = W * 64 / 256;                        // threads of an entry
  const float r0 = a.centroids[(threadIdx.x / TPE >> (BITS == 3 ? 3 : 4)) & ((1 << BITS) - 1)], r1 = a.centroids[threadIdx.x / TPE & ((1 << BITS) - 1)];
  float mx_c = 0.f;
  for (int v = 0; v < (1 << BITS); ++v) mx_c = fmaxf(mx_c, fabsf(a.centroids[v]));
  asm volatile("" : "+v"(mx_c) : "s"(g0), "s"(sb0_first));      // (the record and the codebook in one wait)
  if (g0 >= g1) return;
  const uint32_t ex_c = min(max((__float_as_uint(mx_c) >> 23) & 0xffu, 12u), 250u);
  const float inv_cs = __uint_as_float(ex_c << 23) * (1.f / 512.f);
  bool filled = false;
  auto fill_once = [&]() {
    if (filled) return;
    filled = true;
    const float cs = __uint_as_float((254u - ex_c) << 23) * 512.f;
    const float c0 = r0 * cs, c1 = r1 * cs;
    const __half h0 = __float2half_rn(c0), h1 = __float2half_rn(c1);
    const __half l0 = __float2half_rn(c0 - __half2float(h0)), l1 = __float2half_rn(c1 - __half2float(h1));
    const uint32_t hi = (uint32_t)__half_as_ushort(h0) | ((uint32_t)__half_as_ushort(h1) << 16);
    const uint32_t lo = (uint32_t)__half_as_ushort(l0) | ((uint32_t)__half_as_ushort(l1) << 16);
    // (each thread starts a piece further than its neighbour: all in step they would write to the same banks, 2,500 cycles)
    const uint32_t e = threadIdx.x / TPE, at = e * 256u + threadIdx.x % TPE * (256u / TPE);
#pragma unroll
    for (uint32_t i = 0; i < 16 / TPE; ++i) *(aw_lds_u128*)(uintptr_t)(at + (i + e) % (16u / TPE) * 16u) = (aw_u32x4){hi, lo, hi, lo};
    akv_lds_barrier();
  };
  if constexpr (D != 128) fill_once();

  const bool bs32 = a.block_size == 32;
  const int bs = bs32 ? 32 : 16;
  const int gqa = a.QH / a.KVH;
  const int hp = x.hp, R = W / hp;
  const int hs = wave % hp, r = wave / hp;
  const uint32_t nbase = AW_NORM + (uint32_t)wave * AW_NORM_WAVE;
  const int kb = PACK == 4 ? (lane >> 2) & 3 : (lane >> 3) & 1;     // which NV of a head's eight tokens
  const uint32_t nread = nbase + (uint32_t)g * 16u + (PACK == 4 ? 64u * (uint32_t)(kb >> 1) + 8u * (uint32_t)(kb & 1) : 64u * (uint32_t)kb);

  int gcur = g0, s = s_first, sb0 = sb0_first, sb1 = sb1_first, ctx = ctx_first;
  while (gcur < g1) {
    if (gcur != g0) {
      s = akv_next_seq(a.prefix, a.S, s, gcur, sb0, sb1);
      ctx = __builtin_amdgcn_readfirstlane((int)akv_seq_tokens(a.context_lens, a.cl_itype, s, bs, a.max_blocks_per_seq));
    }
    const int blk_lo = gcur - sb0;
    const int blk_hi = min(g1, sb1) - sb0;
    const int t_end = (int)min((int64_t)blk_hi * bs, (int64_t)ctx);
    gcur = sb0 + blk_hi;
    const int nblk = blk_hi - blk_lo;
    const int nchunks = bs32 ? nblk : (nblk + 1) >> 1;
    const int mine = r < nchunks ? (nchunks - r + R - 1) / R : 0;     // chunks r, r + R, ...

    for (int hbase = 0; hbase < a.KVH; hbase += hp) {
      const int h = hbase + hs;
      const bool active = h < a.KVH;
      const int hd = a.hgroup > 1 ? h / a.hgroup : h;                 // the head whose rows are read
      float m_run = -INFINITY, l_run = 0.f;
      aw_float4 o[CPL];
#pragma unroll
      for (int n = 0; n < CPL; ++n) o[n] = (aw_float4){0.f, 0.f, 0.f, 0.f};

      if (active && mine > 0) {
        // ---- block ids of the wavefront's chunks from win_k on: lane 2 i + j block j of chunk win_k + i (blocks of 32: lane i)
        int pbwin = 0, win_k = 0;
        auto load_window = [&](int k0) {
          const int k = k0 + (bs32 ? lane : lane >> 1);
          const int c = r + k * R;
          const int bi = blk_lo + (int)min((int64_t)(nblk - 1), bs32 ? (int64_t)c : 2 * (int64_t)c + (lane & 1));
          pbwin = (int)akv_clamp_block(akv_load_index(a.block_tables, a.bt_itype, s * a.bt_stride + bi), a.num_blocks);
          win_k = k0;
        };
        // Few requests: with two of a quarter row a lane for keys and eight of the lane's own codes for values there were 704,000 a launch
        // at head_dim 64 (48 sequences of 512 to 8,192, 8 kv heads), now 407,000; 234,000 and 176,000 at 256.  (The address unit is busy
        // about as long as before.)  Decode steps: 48 sequences, one kv head of 128
        // 35.1 -> 33.8 us, heads of 64 66.4 -> 65.2, of 256 in 2 bits 42.0 -> 40.2.
        // Lane (8 p + c, g) reads piece c, of 2 VB bytes, of the first (p = 0) or second token of a pair and hands half of it on.
        // 3 bits: whole dwords around the piece; the selectors gather a group's three bytes, first byte on top.
        const int vp = col >> 3, vc = col & 7;
        constexpr int GB = 3 * D / 64;                                  // bytes from one piece to the next (3 bits)
        const int vdw = BITS != 3 ? 0 : min(GB * vc >> 2, 3 * D / 32 - VRD);
        const uint32_t vsel3 = 0x0c000102u + 0x010101u * (uint32_t)(GB * vc - 4 * vdw);
        const uint32_t koff = KHALF ? (uint32_t)(hd * a.kps_head + col * a.kps_pos + KDW * 4 * (g & 1))
                                    : (uint32_t)(hd * a.kps_head + col * a.kps_pos + KDW * 4 * g);
        const uint32_t voff = (uint32_t)(hd * a.vps_head + (4 * g + (VB >= 4 ? vp : 2 * vp)) * a.vps_pos + (BITS == 3 ? 4 * vdw : 2 * VB * vc));
        const uint32_t ktile1 = bs32 ? 16u * (uint32_t)a.kps_pos : 0u, vtile1 = bs32 ? 16u * (uint32_t)a.vps_pos : 0u;
        const int ntok = lane & 31, npos = bs32 ? ntok : ntok & 15;
        const float* nptr = lane >= 32 ? a.vn : a.kn;
        const uint32_t nblk_stride = (uint32_t)(lane >= 32 ? a.vns_blk : a.kns_blk);
        const uint32_t noff = (uint32_t)(lane >= 32 ? hd * a.vns_head + npos * a.vns_pos : hd * a.kns_head + npos * a.kns_pos);

        // Codes and norms sit in one set of registers: the next chunk's keys are requested when this one's are scored, its
        // values when these are weighed (a second set made the compiler spill in the loop at head_dim 256 and move registers
        // elsewhere).
        uint32_t kr[KHALF ? 1 : 2][KDW], vr[2][2][VRD];
        float nrm;
        auto blocks = [&](int k, uint32_t& pb0, uint32_t& pb1) {
          const int w = bs32 ? k - win_k : 2 * (k - win_k);
          pb0 = (uint32_t)__builtin_amdgcn_readlane(pbwin, w);
          pb1 = bs32 ? pb0 : (uint32_t)__builtin_amdgcn_readlane(pbwin, w + 1);
        };
        auto load_keys = [&](int k) {
          uint32_t pb[2];
          blocks(k, pb[0], pb[1]);
          nrm = nptr[(uint64_t)(ntok >= 16 ? pb[1] : pb[0]) * nblk_stride + noff];
#pragma unroll
          for (int j = 0; j < (KHALF ? 1 : 2); ++j) {
            const unsigned char* p = a.kp + (uint64_t)pb[j] * (uint32_t)a.kps_blk + (j ? ktile1 : 0u);
            if constexpr (KHALF) {
              const unsigned char* p1 = a.kp + (uint64_t)pb[1] * (uint32_t)a.kps_blk + ktile1;
              p = g >= 2 ? p1 : p;
            }
            p += aw_here(koff);
            aw_request<KDW>(kr[j], p);
          }
        };
        auto load_values = [&](int k) {
          uint32_t pb[2];
          blocks(k, pb[0], pb[1]);
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const unsigned char* vb = a.vp + (uint64_t)pb[j] * (uint32_t)a.vps_blk + (j ? vtile1 : 0u);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              const unsigned char* p = vb + (uint32_t)((VB >= 4 ? 2 * q : q) * (int)a.vps_pos) + aw_here(voff);
              if constexpr (VB == 1 && BITS != 3) vr[j][q][0] = *(const uint16_t*)p;
              else aw_request<VRD>(vr[j][q], p);
            }
          }
        };

        load_window(0);
        load_keys(0);
        load_values(0);
        uint2 qd[KS];
        {
          const uint2* qp = x.qop + (size_t)(s * a.KVH + h) * (KS * 64) + (KHALF ? 16 * (g < 2 ? 2 * g : 2 * g - 3) + col : lane);      // the quarter the lane ends up with
#pragma unroll
          for (int st = 0; st < KS; ++st) qd[st] = qp[st * 64];
        }
        const float fac = x.fac[(size_t)s * a.QH + h * gqa + min(col & (PACK == 4 ? 3 : 7), gqa - 1)] * inv_cs;
        fill_once();

        for (int k = 0; k < mine; ++k) {
          const int c = r + k * R;
          // ---- norms: lanes 0..31 hold the key norms, 32..63 the value norms; the exponent of a value norm bounds it
          // from above by a power of two
          *(aw_lds_f32*)(uintptr_t)(nbase + (uint32_t)lane * 4u) = nrm;
          if (lane >= 32) {
            const int e = (int)((__float_as_uint(nrm) >> 23) & 0xffu) - 126;
            *(aw_lds_f32*)(uintptr_t)(nbase + 256u + (uint32_t)ntok * 4u) = (float)max(e, -AW_TINY);
          }
          akv_wave_sync();

          // ---- scores
          // the words of both tiles: bytes (3 bits: groups of eight codes) of the lane's quarter of a row.  KHALF: lanes g < 2 hold half g of
          // a row of tile 0, the others half g - 2 of one of tile 1; two pairs of rows of lanes trade a quarter.
          constexpr int KW = BITS == 3 ? D / 32 : D * BITS / 128;
          uint32_t kw[2][KW];
#pragma unroll
          for (int j = 0; j < (KHALF ? 1 : 2); ++j) {
            constexpr int N = KHALF ? 2 * KW : KW;
            uint32_t w[N];
#pragma unroll
            for (int i = 0; i < N; ++i) {
              // (3 bits: four groups in three dwords)
              if constexpr (BITS == 3) {
                const int b = 3 * (i & 3), at = 3 * (i >> 2) + b / 4;
                w[i] = __builtin_amdgcn_perm(kr[j][min(at + 1, KDW - 1)], kr[j][at], 0x0c000102u + 0x010101u * (b % 4));
              } else {
                w[i] = kr[j][i];
              }
            }
#pragma unroll
            for (int i = 0; i < KW; ++i) {
              if constexpr (KHALF) {
                auto t = __builtin_amdgcn_permlane32_swap(w[i], w[KW + i], false, false);
                kw[0][i] = t[0];
                kw[1][i] = t[1];
              } else {
                kw[j][i] = w[i];
              }
            }
          }
          if constexpr (BITS == 3) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
              for (int i = 0; i < KW; ++i) kw[j][i] = aw_spread24(kw[j][i]);
          }
          aw_float4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
          // (the tiles take turns: two chains of sums)
          aw_products<AHEAD, 2 * KS>(
              [&](auto i, aw_u32x2& x, aw_u32x2& y) __attribute__((always_inline)) {
                constexpr int I = decltype(i)::value, st = I / 2;
                const uint32_t w = kw[I % 2][st / (KS / KW)];
                if constexpr (BITS == 4) {
                  x = aw_look<2 * (st & 1)>(copy, w);
                  y = aw_look<2 * (st & 1) + 1>(copy, w);
                } else if constexpr (BITS == 3) {
                  x = aw_look<3 - 2 * (st & 1)>(copy, w);
                  y = aw_look<2 - 2 * (st & 1)>(copy, w);
                } else {
                  x = aw_look<(st & 3)>(copy, (w >> 2) & 0x33333333u);
                  y = aw_look<(st & 3)>(copy, w & 0x33333333u);
                }
              },
              [&](auto i, aw_half8 op) __attribute__((always_inline)) {
                constexpr int I = decltype(i)::value, st = I / 2;
                const aw_u32x2 q0 = {qd[st].x, qd[st].x}, q1 = {qd[st].y, qd[st].y};
                acc[I % 2] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op, aw_operand(q0, q1), acc[I % 2], 0, 0, 0);
              });

          __builtin_amdgcn_sched_barrier(0);
          // (past the end: the last chunk once more, out of the window it is in)
          if (k + 1 < mine && k + 1 - win_k >= AW_WIN) load_window(k + 1);
          load_keys(min(k + 1, mine - 1));
          __builtin_amdgcn_sched_barrier(0);

          // ---- running softmax in the log2 domain over t = score + exponent of the value norm, on a PACKED copy of the scores:
          // the accumulator holds eight tokens per lane, sums of the queries' roundings in columns 0..7 and of their remainders
          // in 8..15.  PACK = 4 (at most four query heads): lane 4 k + c of a row takes the token pair k of head c, the first
          // term from lane c, the second from lane 8 + c; PACK = 2: lane c takes tile 0, lane 8 + c tile 1 of head c.  Every lane
          // on all eight tokens of its column, as the accumulator lies, were 16 exponentials a lane (a quarter of the rate of
          // other vector instructions) in place of 4 or 8.  An attention call, 32 query heads on 8 of 64, 48 sequences of 512 to 8,192
          // tokens: 64.9 -> 60.1 us; 16 on 4 of 256, 24 sequences: 64.4 -> 63.0; 8 on 1 of 128, 48 of 1,024 to 16,384: 36.9 -> 35.9.
          float sv[NV], vn[NV], tv[NV];
          if constexpr (PACK == 4) {
#pragma unroll
            for (int jj = 0; jj < 2; ++jj) {
              float hi = acc[0][jj];
              hi = akv_dpp_bank<0x114 /*row_shr:4*/, 1>(hi, acc[0][2 + jj]);
              hi = akv_dpp_bank<0x118 /*row_shr:8*/, 2>(hi, acc[1][jj]);
              hi = akv_dpp_bank<0x11c /*row_shr:12*/, 3>(hi, acc[1][2 + jj]);
              float lo = acc[1][jj];
              lo = akv_dpp_bank<0x108 /*row_shl:8*/, 0>(lo, acc[0][jj]);
              lo = akv_dpp_bank<0x104 /*row_shl:4*/, 1>(lo, acc[0][2 + jj]);
              lo = akv_dpp_bank<0x114 /*row_shr:4*/, 3>(lo, acc[1][2 + jj]);
              sv[jj] = hi + lo;
            }
            const aw_float2 kn2 = *(aw_lds_f64*)(uintptr_t)nread, vn2 = *(aw_lds_f64*)(uintptr_t)(nread + 128u);
            const aw_float2 ve2 = *(aw_lds_f64*)(uintptr_t)(nread + 256u);
#pragma unroll
            for (int jj = 0; jj < 2; ++jj) {
              sv[jj] *= kn2[jj] * fac;
              vn[jj] = vn2[jj];
              tv[jj] = sv[jj] + ve2[jj];
            }
          } else {
#pragma unroll
            for (int jj = 0; jj < 4; ++jj)
              sv[jj] = akv_dpp_banks<0x118 /*row_shr:8*/, 0xc>(acc[0][jj], acc[1][jj]) + akv_dpp_banks<0x108 /*row_shl:8*/, 0x3>(acc[1][jj], acc[0][jj]);
            const aw_float4 kn4 = *(aw_lds_f128*)(uintptr_t)nread, vn4 = *(aw_lds_f128*)(uintptr_t)(nread + 128u);
            const aw_float4 ve4 = *(aw_lds_f128*)(uintptr_t)(nread + 256u);
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
              sv[jj] *= kn4[jj] * fac;
              vn[jj] = vn4[jj];
              tv[jj] = sv[jj] + ve4[jj];
            }
          }
          if (c == nchunks - 1) {        // only the last chunk of a segment holds tokens past its end
            // (such a row may hold anything, NaN norms included.  The empty statement keeps this a branch: as selects the
            // comparisons cost every chunk instructions.)
            asm volatile("");
            const int tok0 = blk_lo * bs + 32 * c + 4 * g + (PACK == 4 ? 16 * (kb >> 1) + 2 * (kb & 1) : 16 * kb);
#pragma unroll
            for (int jj = 0; jj < NV; ++jj)
              if (tok0 + jj >= t_end) { sv[jj] = -INFINITY; vn[jj] = 0.f; tv[jj] = -INFINITY; }
          }
          float mx = fmaxf(tv[0], tv[1]);
          if constexpr (PACK == 2) {
            mx = fmaxf(mx, fmaxf(tv[2], tv[3]));
            mx = fmaxf(mx, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(mx), 0x128 /*row_ror:8*/, 0xf, 0xf, false)));
          } else {
            mx = akv_banks_max(mx);
          }
          akv_wave_sync();      // the norms have been read: the next chunk overwrites them
          mx = akv_rows_max(mx);
          const float m_new = fmaxf(m_run, mx - AW_FRAME);
          const float resc = __builtin_amdgcn_exp2f(m_run - m_new);      // 0 on the first chunk
          m_run = m_new;
          float psum = 0.f;
          uint32_t wh[NV / 2], wl[NV / 2];       // the lane's token pairs as float16 rounding and remainder
#pragma unroll
          for (int p = 0; p < NV / 2; ++p) {
            const float p0 = __builtin_amdgcn_exp2f(sv[2 * p] - m_new), p1 = __builtin_amdgcn_exp2f(sv[2 * p + 1] - m_new);
            psum += p0 + p1;
            const aw_float2 w2 = {p0 * vn[2 * p], p1 * vn[2 * p + 1]};
            const aw_half2 h2 = __builtin_convertvector(w2, aw_half2);
            const aw_half2 l2 = __builtin_convertvector(w2 - __builtin_convertvector(h2, aw_float2), aw_half2);
            union { aw_half2 h; uint32_t u; } hu, lu;
            hu.h = h2;
            lu.h = l2;
            wh[p] = hu.u;
            wl[p] = lu.u;
          }
          l_run = l_run * resc + psum;
          // back to the operand's columns: roundings in 0..7, remainders in 8..15, zeros where there is no query head
          aw_half8 wop[2];
          if constexpr (PACK == 4) {
            const uint32_t w0 = akv_pair_from_bank<0>(wh[0], wl[0]), w1 = akv_pair_from_bank<1>(wh[0], wl[0]);
            const uint32_t w2 = akv_pair_from_bank<2>(wh[0], wl[0]), w3 = akv_pair_from_bank<3>(wh[0], wl[0]);
            wop[0] = aw_operand((aw_u32x2){w0, w0}, (aw_u32x2){w1, w1});
            wop[1] = aw_operand((aw_u32x2){w2, w2}, (aw_u32x2){w3, w3});
          } else {
            uint32_t w0[2], w1[2];
#pragma unroll
            for (int p = 0; p < 2; ++p) {
              w0[p] = akv_dpp_banks_u<0x118 /*row_shr:8*/, 0xc>(wh[p], wl[p]);
              w1[p] = akv_dpp_banks_u<0x108 /*row_shl:8*/, 0x3>(wl[p], wh[p]);
            }
            wop[0] = aw_operand((aw_u32x2){w0[0], w0[0]}, (aw_u32x2){w0[1], w0[1]});
            wop[1] = aw_operand((aw_u32x2){w1[0], w1[0]}, (aw_u32x2){w1[1], w1[1]});
          }
          if (__builtin_amdgcn_ballot_w64(resc != 1.f) != 0) {
#pragma unroll
            for (int n = 0; n < CPL; ++n)
#pragma unroll
              for (int i = 0; i < 4; ++i) o[n][i] *= resc;
          }

          // ---- values
          if constexpr (VB >= 4) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              constexpr int VW = VB / 4;
              uint32_t word[4][VW];                  // of a tile's four tokens: words of codes (3 bits: of fields)
#pragma unroll
              for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int d = 0; d < VW; ++d) {
                  const uint32_t(&r)[VRD] = vr[j][q];
                  if constexpr (BITS != 3) {
                    aw_trade(r[d], r[VW + d], word[2 * q][d], word[2 * q + 1][d]);
                  } else {
                    uint32_t x, y;
                    if constexpr (D == 256) {        // four groups in three dwords
                      auto group = [&](int i) { return __builtin_amdgcn_perm(r[min(3 * i / 4 + 1, 2)], r[3 * i / 4], 0x0c000102u + 0x010101u * (3 * i % 4)); };
                      x = group(d);
                      y = group(2 + d);
                    } else {
                      x = __builtin_amdgcn_perm(r[1], r[0], vsel3);
                      y = __builtin_amdgcn_perm(r[1], r[0], vsel3 + 0x030303u);
                    }
                    aw_trade(x, y, word[2 * q][d], word[2 * q + 1][d]);
                    word[2 * q][d] = aw_spread24(word[2 * q][d]);
                    word[2 * q + 1][d] = aw_spread24(word[2 * q + 1][d]);
                  }
                }
              aw_pairs<BITS, 0> p01[VW], p23[VW];
#pragma unroll
              for (int d = 0; d < VW; ++d) {
                aw_pair(p01[d], word[0][d], word[1][d]);
                aw_pair(p23[d], word[2][d], word[3][d]);
              }
              aw_products<AHEAD, CPL>(
                  [&](auto i, aw_u32x2& x, aw_u32x2& y) __attribute__((always_inline)) {
                    constexpr int I = decltype(i)::value, q = I % CPB, K = I / CPB % 4, d = I / CPB / 4;
                    x = aw_look<K>(copy, p01[d].w[q]);
                    y = aw_look<K>(copy, p23[d].w[q]);
                  },
                  [&](auto i, aw_half8 op) __attribute__((always_inline)) {
                    constexpr int I = decltype(i)::value, q = I % CPB, K = I / CPB % 4, d = I / CPB / 4, n = (4 * d + (BITS == 3 ? 3 - K : K)) * CPB + q;
                    o[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op, wop[j], o[n], 0, 0, 0);
                  });
            }
          } else if constexpr (VB == 2) {
            // two bytes per token: both token pairs of a tile side by side in one word (a request's pair: tokens two apart)
            aw_pairs<BITS, 0> p[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              auto word = [&](int q) __attribute__((always_inline)) {
                if constexpr (BITS != 3) {
                  const uint32_t x = vr[j][q][0];
                  const uint32_t y = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x128 /*row_ror:8*/, 0xf, 0xf, false);
                  return __builtin_amdgcn_perm(y, x, vp ? 0x03020706u : 0x05040100u);
                }
                // the group of eight codes of both tokens, then twelve bits of each
                const uint32_t x = __builtin_amdgcn_perm(vr[j][q][VRD - 1], vr[j][q][0], vsel3);
                uint32_t t0, t1;
                aw_trade(x, x, t0, t1);
                return aw_spread12((t0 >> (vp ? 0 : 12) & 0xFFFu) | (t1 << (vp ? 16 : 4) & 0x0FFF0000u));
              };
              aw_pair(p[j], word(0), word(1));
            }
            // (3 bits: the first field is the upper byte of a half)
            aw_products<AHEAD, 2 * CPL>(
                [&](auto i, aw_u32x2& x, aw_u32x2& y) __attribute__((always_inline)) {
                  constexpr int I = decltype(i)::value, j = I / CPL, half = I / CPB % 2, K = BITS == 3 ? 1 - half : half;
                  x = aw_look<K>(copy, p[j].w[I % CPB]);
                  y = aw_look<K + 2>(copy, p[j].w[I % CPB]);
                },
                [&](auto i, aw_half8 op) __attribute__((always_inline)) {
                  constexpr int I = decltype(i)::value;
                  o[I % CPL] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op, wop[I / CPL], o[I % CPL], 0, 0, 0);
                });
          } else {
            // one byte per token: the pairs of both tiles side by side
            aw_pairs<BITS, 0> p;
            auto join = [&](int q) {
              const uint32_t x = vr[0][q][0] | (vr[1][q][0] << 16);
              const uint32_t y = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x128 /*row_ror:8*/, 0xf, 0xf, false);
              return __builtin_amdgcn_perm(y, x, vp ? 0x03070105u : 0x06020400u);
            };
            aw_pair(p, join(0), join(1));
            aw_products<AHEAD, 2 * CPL>(
                [&](auto i, aw_u32x2& x, aw_u32x2& y) __attribute__((always_inline)) {
                  constexpr int I = decltype(i)::value, j = I / CPL;
                  x = aw_look<2 * j>(copy, p.w[I % CPL]);
                  y = aw_look<2 * j + 1>(copy, p.w[I % CPL]);
                },
                [&](auto i, aw_half8 op) __attribute__((always_inline)) {
                  constexpr int I = decltype(i)::value;
                  o[I % CPL] = __builtin_amdgcn_mfma_f32_16x16x32_f16(op, wop[I / CPL], o[I % CPL], 0, 0, 0);
                });
          }
          __builtin_amdgcn_sched_barrier(0);
          load_values(min(k + 1, mine - 1));
          __builtin_amdgcn_sched_barrier(0);
        }
        l_run = akv_rows_sum(l_run);      // (every lane of a row had its own tokens)
        if constexpr (PACK == 4) l_run = akv_banks_sum(l_run);
        else l_run = aw_add_cols(l_run);
      } else {
        fill_once();
      }

      // ---- partial result: lane (col < gqa, g) holds rows 4 g + i of value tile n for query head col: coordinates o_at + 2 CPL i + n
      // (row 8 p + c is half p of piece c)
      const int o_at = CPL * (8 * (g & 1) + (g >> 1));
      const size_t slot = (size_t)(blockIdx.x + s) * a.QH + h * gqa;
      float M = m_run, wgt = inv_cs, L = l_run;
      const int shares = min(R, nchunks);      // wavefronts of the head that hold a result
      if (shares > 1) {
        if (lane < 8) *(aw_lds_f64*)(uintptr_t)(aw_ml_off<W>() + (uint32_t)wave * 64u + (uint32_t)lane * 8u) = (aw_float2){m_run, l_run};
        akv_lds_barrier();
        // (AT requested at a time, at 128 and 256 all there can be; past the last share that one again, for nothing)
        constexpr int AT = D == 64 ? 4 : W;
        const int rounds = D == 64 ? shares : 1;
        auto of_share = [&](int rr) { return *(aw_lds_f64*)(uintptr_t)(aw_ml_off<W>() + (uint32_t)(min(rr, shares - 1) * hp + hs) * 64u + (uint32_t)(col & 7) * 8u); };
        L = 0.f;
        for (int r0 = 0; r0 < rounds; r0 += AT) {
          aw_float2 ml[AT];
#pragma unroll
          for (int i = 0; i < AT; ++i) ml[i] = of_share(r0 + i);
#pragma unroll
          for (int i = 0; i < AT; ++i) M = fmaxf(M, ml[i].x);
        }
        for (int r0 = 0; r0 < rounds; r0 += AT) {
          aw_float2 ml[AT];
#pragma unroll
          for (int i = 0; i < AT; ++i) ml[i] = of_share(r0 + i);
#pragma unroll
          for (int i = 0; i < AT; ++i) {
            const float part = ml[i].x > -INFINITY ? __builtin_amdgcn_exp2f(ml[i].x - M) * ml[i].y : ml[i].y;      // (-inf: no token, or sums that are NaN)
            L += r0 + i < shares ? part : 0.f;
          }
        }
        wgt = m_run > -INFINITY ? __builtin_amdgcn_exp2f(m_run - M) * inv_cs : inv_cs;
      }
#pragma unroll
      for (int n = 0; n < CPL; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[n][i] = aw_add_cols(o[n][i]) * wgt;
      if (shares <= 1) {
        if (active && r == 0 && col < gqa) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int n = 0; n < CPL; n += 4)
              *(float4*)(a.part_acc + (slot + col) * D + o_at + 2 * CPL * i + n) = make_float4(o[n][i], o[n + 1][i], o[n + 2][i], o[n + 3][i]);
        }
      } else {
        const uint32_t wave_bytes = (uint32_t)gqa * D * 4u;
        if (active && r < shares && col < gqa) {
          const uint32_t at = aw_acc_off<W>() + (uint32_t)wave * wave_bytes + (uint32_t)(col * D + o_at) * 4u;
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int n = 0; n < CPL; n += 4)
              *(aw_lds_f128*)(uintptr_t)(at + (uint32_t)(2 * CPL * i + n) * 4u) = (aw_float4){o[n][i], o[n + 1][i], o[n + 2][i], o[n + 3][i]};
        }
        akv_lds_barrier();
        if (active) {
          // (no barrier after these reads: the next segment's accumulators are written behind its first barrier)
          for (int idx = r * 64 + lane; idx < gqa * D / 4; idx += R * 64) {
            aw_float4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
            for (int rr = 0; rr < shares; ++rr) sum += *(aw_lds_f128*)(uintptr_t)(aw_acc_off<W>() + (uint32_t)(rr * hp + hs) * wave_bytes + (uint32_t)idx * 16u);
            *(float4*)(a.part_acc + slot * D + 4 * (size_t)idx) = make_float4(sum.x, sum.y, sum.z, sum.w);
          }
        }
      }
      if (active && r == 0 && lane < gqa) {
        a.part_ml[(slot + lane) * 2] = M * 0.6931471805599453f;     // back to the natural-log domain
        a.part_ml[(slot + lane) * 2 + 1] = L;
      }
    }
  }
}

// ----------------------------------------------------------------------------------
// host side
// ----------------------------------------------------------------------------------
bool akv_attn_mfma_takes(const akv_attn_args& a, int bits);       // the conditions both matrix-core kernels share
int akv_attn_mfma_head_groups(int gqa);

// At head_dim 128 the kernel of akv_attn_mfma.hip has eight head slots, most of them idle where a rank keeps one or two (groups
// of) kv heads.  The rule takes nothing that the width of the tables changes: a serving engine's are as wide as its longest
// context may become, whatever the contexts are.  Measured, prologue, main kernel and reduce in a graph (us, this | that), eight
// query heads a group, 4 bits:
//   one group     32 of 700 15.3 | 14.9; 64 of 100 14.2 | 13.8, of 700 16.5 | 17.0, of 3,000 21.3 | 29.2; 128 of 100 15.9 | 15.0, of
//                 1,000 20.8 | 25.0, of 1,000 to 4,000 32.4 | 44.4; 200 of 300 21.5 | 21.4, of 1,000 27.8 | 33.6; 256 of 1,000 24.5 | 35.7
//   two groups    32 of 700 17.1 | 16.1; 64 of 100 15.1 | 15.0, of 700 18.6 | 18.3, of 3,000 27.0 | 30.7;
//                 100 of 100 17.0 | 16.3, of 300 19.7 | 18.2, of 1,000 24.6 | 26.2, of 1,000 to 8,000 50.7 | 58.3; 128 of 300
//                 19.9 | 18.9, of 1,000 25.6 | 27.3; 200 of 300 28.0 | 26.3, of 1,000 35.8 | 37.5
// Short contexts are up to 1.5 us faster there (it starts sooner), long ones faster here.  One group loses at most 6 % and gains up to
// 46.  Two lose up to 8 % below 1,000 tokens and gain up to 16 above, with few sequences as with many; the host cannot see the contexts,
// and batches of more than 64 sequences, where neither choice is the better one throughout, are left to that kernel.
bool akv_attn_wave_applicable(const akv_attn_args& a, int d, int bits) {
  if (!(d == 64 || d == 128 || d == 256) || bits < 2 || bits > 4 || !akv_attn_mfma_takes(a, bits)) return false;
  if (d != 128) return true;
  const int heads = a.KVH * akv_attn_mfma_head_groups(a.QH / a.KVH);
  return heads == 1 || (heads == 2 && a.S <= 64);
}

// kv head slots of a workgroup of w wavefronts
static int aw_slots(int kv_heads, int w) {
  int hp = 1;
  while (hp < kv_heads && hp < w) hp *= 2;
  return hp;
}

template <int D, int BITS, int PACK>
static int aw_launch_as(const akv_attn_args& a, const aw_extra& x_in, int grid, hipStream_t stream) {
  constexpr int W = aw_cfg<D, BITS>::W;
  aw_extra x = x_in;
  x.hp = aw_slots(a.KVH, W);
  const int gqa = a.QH / a.KVH;
  constexpr int most = (int)aw_acc_off<W>() + W * 8 * D * 4;
  static_assert(most <= 160 * 1024, "LDS of a CU");
  const int lds = (int)aw_acc_off<W>() + (x.hp < W ? W * gqa * D * 4 : 0);
  static akv_device_once allowed;
  int dev = -1;
  AKV_HIP(hipGetDevice(&dev));
  const int rc = allowed(dev, []() -> int {
    AKV_HIP(hipFuncSetAttribute((const void*)akv_attn_wave_kernel<D, BITS, PACK>, hipFuncAttributeMaxDynamicSharedMemorySize, most));
    return AKV_OK;
  });
  if (rc) return rc;
  AKV_LAUNCH_TIMED((akv_attn_wave_kernel<D, BITS, PACK>), grid, W * 64, lds, stream, a, x);
  AKV_LAUNCH_CHECK("akv_attn_wave_kernel");
  return AKV_OK;
}

template <int D>
static int aw_launch(const akv_attn_args& a, const aw_extra& x, int bits, int grid, hipStream_t stream) {
  const bool four = a.QH / a.KVH <= 4;
  if (bits == 4) return four ? aw_launch_as<D, 4, 4>(a, x, grid, stream) : aw_launch_as<D, 4, 2>(a, x, grid, stream);
  if (bits == 3) return four ? aw_launch_as<D, 3, 4>(a, x, grid, stream) : aw_launch_as<D, 3, 2>(a, x, grid, stream);
  return four ? aw_launch_as<D, 2, 4>(a, x, grid, stream) : aw_launch_as<D, 2, 2>(a, x, grid, stream);
}

int akv_attn_wave_run(const void* query, int q_dtype, int64_t qs_seq, int64_t qs_head, const float* PiT, const akv_attn_args& a_in,
                      int d, int bits, const akv_attn_ws& ws, void* extra_ws, int grid, hipStream_t stream) {
  akv_attn_args a = a_in;
  a.hgroup = akv_attn_mfma_head_groups(a.QH / a.KVH);
  a.KVH *= a.hgroup;                        // from here on: groups of at most eight query heads
  aw_extra x;
  x.qop = (const uint2*)extra_ws;           // 32 d bytes per group: at most what the other kernel's operand takes (d <= 256)
  x.fac = ws.qrot;
  x.wgdesc = ws.wgdesc;
  x.hp = 0;
  const float qscale = a.scale * 1.4426950408889634f;   // scores come out in the log2 domain
  const int slots = aw_slots(a.KVH, d == 64 ? 16 : 8), shares = (d == 64 ? 16 : 8) / slots;
  const int cus = akv_cached_cu_count(), qslots = a.QH / a.KVH <= 4 ? 4 : 8;
  // rotation blocks, up to three on a CU (then they loop: a slice of the matrix is read once per block)
  const int pgrid = ar_query_blocks(d, a.S, a.KVH, qslots, 3 * (cus > 0 ? cus : 256)) + 1;
  const float* Pi = PiT - (size_t)d * d;
  const akv_prep_scale* scale = (const akv_prep_scale*)((const char*)Pi + AKV_PREP_SCALE_OFFSET(d));
#define AW_PRO(DD, DT) akv_attn_wave_prologue_kernel<DD, DT><<<pgrid, 256, 0, stream>>>(query, qs_seq, qs_head, Pi, scale, a.S, a.QH, a.KVH, qslots, a.context_lens, a.cl_itype, a.block_size, a.max_blocks_per_seq, ws.prefix, (uint2*)extra_ws, ws.qrot, ws.status, qscale, bits, ws.wgdesc, ws.seqw, grid, shares)
#define AW_PRO_D(DD) do { if (q_dtype == AKV_F16) AW_PRO(DD, AKV_F16); else if (q_dtype == AKV_BF16) AW_PRO(DD, AKV_BF16); else AW_PRO(DD, AKV_F32); } while (0)
  if (d == 64) AW_PRO_D(64);
  else if (d == 128) AW_PRO_D(128);
  else AW_PRO_D(256);
#undef AW_PRO_D
#undef AW_PRO
  AKV_LAUNCH_CHECK("akv_attn_wave_prologue_kernel");
  if (d == 64) return aw_launch<64>(a, x, bits, grid, stream);
  if (d == 128) return aw_launch<128>(a, x, bits, grid, stream);
  return aw_launch<256>(a, x, bits, grid, stream);
}
