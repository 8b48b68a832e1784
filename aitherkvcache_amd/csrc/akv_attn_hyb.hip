// Paged decode attention on hybrid rows (tq35 and tq25), on the matrix cores, every wavefront on its own.
//
// A row holds four parts: A0 and A1, codes of the two coordinate groups, and B0 and B1, the signs of their residuals; a decoded
// group is n (Inv_had(c[code]) + r kappa Inv_qjl(sign)) with two float16 factors n, r per group (akv_hybrid_layout.h).  With
// the query transformed once, the score of a token is n0 (A0.qa0 + r0 kappa B0.qb0) + n1 (A1.qa1 + r1 kappa B1.qb1), and the
// value sums are kept per part, with weights p n0, p n0 r0, p n1, p n1 r1, and transformed back at the end.
//
// A workgroup is four wavefronts, (head slot) x (share of the tokens); the groups of four query heads beyond the slots are
// other workgroups on the same range of blocks.  A wavefront takes chunks of 32 tokens:
//
//   rows     requested a chunk ahead straight into LDS (16 rows an instruction); nothing passes through registers, and an
//            instruction touches every row once.  The 16-byte pieces of rows are permuted so that the sixteen lanes that read
//            the same place of sixteen rows meet different banks.
//   scores   v_mfma_i32_16x16x64_i8, 16 tokens a tile.  A level is an integer of three signed bytes, looked up four codes at
//            a time by byte permutes from registers; signs are +-64, their bits as they lie (no look-up).  The query is three
//            signed bytes too (23 bits and a sign, one scale a head), in the columns 4 d + head of digit d.  Sums are exact.
//   softmax  on packed scores: the lanes of a row add the digits up so that lane 4 k + c ends up with two of the eight
//            tokens of head c, as in akv_attn_wave_kernel.
//   values   v_mfma_f32_16x16x32_f16, all 32 tokens of a chunk in one product.  The transposing LDS read hands a lane one byte
//            position of eight tokens; codes are looked up four tokens at a time (two byte permutes, two to interleave), signs
//            are the sign bit of 1.0.  A weight is two float16 terms, columns 0..3 and 4..7.
//
// What bounds it: the issue of vector instructions, 660 a chunk and kv head (64 sequences of 8,192 tokens: vector unit 73 % of the
// cycles, matrix cores 15 %, LDS 36 %).  The kernel before this one (four score and four value wavefronts that handed chunks over
// through polled counters, codes spread to nibbles and looked up in LDS) issued some 1,300 at two wavefronts a SIMD.  A decode
// step, its write included, this | that, bfloat16:
// 64 sequences of 4,000 to 8,192 tokens, 32 heads on 8: 166 | 211 us; 256 of 64 to 512: 84 | 111; 64 of 300: 45 | 54; 4 of 300:
// 24 | 38; 32 of 1,000 to 9,000 with 64 heads on 8: 134 | 188, 8 on 1: 42 | 61.  (With levels of keys in two bytes the first was 159
// and the last but one 127, but they are off by 1e-6 of the largest: float32 outputs whose scores reach some hundreds had
// twice the error.)  Head counts that are no multiple of four a kv head (values of float32's accuracy, see hw35) | the vector
// kernel: 28 on 4: 106 | 570; 16 on 16: 165 | 238.
// tq25 rows | the vector kernel (tables of partial products in LDS): 64 of 4,000 to 8,192, 32 heads on 8: 156 | 335; 256 of 64 to
// 512: 88 | 114; 32 of 1,000 to 9,000 with 8 heads on 1: 43 | 246, 28 on 4: 78 | 278, 16 on 16: 126 | 144; 4 of 300: the same.
#include <type_traits>

#include "akv_attn_common.h"
#include "akv_hybrid_layout.h"

typedef _Float16 hw_half8 __attribute__((ext_vector_type(8)));
typedef _Float16 hw_half2 __attribute__((ext_vector_type(2)));
typedef float hw_float2 __attribute__((ext_vector_type(2)));
typedef float hw_float4 __attribute__((ext_vector_type(4)));
typedef unsigned short hw_ushort2 __attribute__((ext_vector_type(2)));
typedef int hw_int2 __attribute__((ext_vector_type(2)));
typedef int hw_int4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) const uint32_t hw_lds_cu32;
typedef __attribute__((address_space(3))) const uint16_t hw_lds_cu16;
typedef __attribute__((address_space(3))) const uint8_t hw_lds_cu8;
typedef __attribute__((address_space(3))) const long hw_lds_l64;
typedef __attribute__((address_space(3))) uint32_t hw_lds_u32;
typedef __attribute__((address_space(3))) hw_int2 hw_lds_i64;
typedef __attribute__((address_space(3))) float hw_lds_f32;
typedef __attribute__((address_space(3))) hw_float2 hw_lds_f64;
typedef __attribute__((address_space(3))) hw_float4 hw_lds_f128;
typedef __attribute__((address_space(3))) hw_int4 hw_lds_i128;

#define HW_W 4                 // wavefronts of a workgroup
#define HW_FRAME 8.f           // a new maximum weighs at most 2^HW_FRAME, and
#define HW_SLACK 7.f           // weights stay below 2^(HW_FRAME + HW_SLACK)
#define HW_TINY 90             // value factors count as at least 2^-HW_TINY in the running maximum
#define HW_WIN 32              // chunks served by one window of 64 block ids
#define HW_QMAX 8290000.f      // largest query integer: 126.5 * 2^16, its top byte stays in range
#define HW_SEARCH 65536        // candidates for the factor of the value levels
// LDS: per wavefront two chunk buffers | per wavefront factors of 32 keys (16 bytes each), of 32 values and their exponents (32) |
// per wavefront (max, sum) of four heads | per wavefront its query operand (in registers it would make the loop spill)
#define HW_BUF 8192u
#define HW_FAC (HW_W * HW_BUF)
#define HW_FAC_WAVE 1536u
#define HW_ML (HW_FAC + HW_W * HW_FAC_WAVE)
#define HW_Q (HW_ML + HW_W * 32u)
#define HW_Q_PART 768u         // of a part: the twelve columns of digits
#define HW_LDS (HW_Q + HW_W * 4u * HW_Q_PART)
static_assert(HW_LDS <= 52 * 1024, "three workgroups a CU, whatever the granularity");
// words of the table block kept in the workspace.  Tag and mark lie where the other kernels' table blocks have them, so that
// whichever kernel used the workspace last is known.
#define HW_W_KA0 0             // bytes of the 3-bit levels, three digits, top first: levels 0..3, 4..7 of each
#define HW_W_KA1 6             // of the 2-bit levels
#define HW_W_VA0 9             // bytes of float16(alpha c): low 0..3, 4..7, high 0..3, 4..7
#define HW_W_VA1 13            // low, high
#define HW_W_VP0 15            // their remainders, likewise
#define HW_W_VP1 19
#define HW_W_UNIT 21           // units of the two level sets
#define HW_W_ALPHA 23          // alpha of the two value sets
#define HW_W_DELTA 25          // tq25: half the distance of the two levels of a 1-bit code, and their middle
#define HW_W_MIDDLE 26
#define HW_W_TAG 768
#define HW_W_MARK 784
#define HW_MARK 0x48570000u    // plus the format
#define HW_VALUES 2048u        // of a chunk buffer: the value rows

struct hw_args {
  const uint8_t* kc; int64_t kps_blk, kps_pos, kps_head;
  const uint8_t* vc; int64_t vps_blk, vps_pos, vps_head;
  const void* block_tables; int bt_itype; int64_t bt_stride;
  const void* context_lens; int cl_itype;
  int S, QH, KVH, hgroup, gqa, block_size; // KVH counts groups of up to four query heads, hgroup of them a kv head
  int64_t max_blocks_per_seq, num_blocks;
  const int32_t* prefix;
  const int32_t* wgdesc;                   // [ranges][AKV_WGREC]
  const uint32_t* lut;
  const uint4* qop;                        // [S][KVH][4 parts][64 lanes] sixteen int8
  const float* fac;                        // [S][QH] scale of a head's query integers, times scale * log2 e
  float* part_acc;                         // [ranges + S][QH][256]: A0 | B0 | A1 | B1, natural coordinate order
  float* part_ml;
  int hp, hgroups;                         // head slots of a workgroup (a power of two), workgroups of a range
};

__device__ __forceinline__ hw_half8 hw_operand(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  union { uint32_t u[4]; hw_half8 h; } x;
  x.u[0] = a; x.u[1] = b; x.u[2] = c; x.u[3] = d;
  return x.h;
}
__device__ __forceinline__ hw_int4 hw_as_int4(uint4 u) {
  union { uint4 u; hw_int4 v; } x;
  x.u = u;
  return x.v;
}
// (x & mask) | rest in one instruction
__device__ __forceinline__ uint32_t hw_and_or(uint32_t x, uint32_t mask, uint32_t rest) { return __builtin_amdgcn_bitop3_b32(x, mask, rest, 0xEA); }
// N bytes per lane from base + voff into LDS at lds + N lane.  (The compiler does not see the request: whoever reads waits by
// hw_landed(); a wavefront's buffers are its own.  No earlier LDS read of the wavefront is in flight any more.  Five wait states
// before the request: its base may come from a lane read, a restored register for one, and the compiler counts none of them here;
// nor the one behind m0.)
template <int N> __device__ __forceinline__ void hw_request(const uint8_t* base, uint32_t voff, uint32_t lds) {
  if constexpr (N == 16)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "{m0}"(lds) : "memory");
  else
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_nop 3\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(base), "{m0}"(lds) : "memory");
}
__device__ __forceinline__ void hw_landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// float16 levels of the codes of four tokens, low and high bytes: tokens 0 and 2, tokens 1 and 3
__device__ __forceinline__ void hw_expand(uint32_t low, uint32_t high, uint32_t& e, uint32_t& o) {
  e = __builtin_amdgcn_perm(high, low, 0x06020400u);
  o = __builtin_amdgcn_perm(high, low, 0x07030501u);
}
// signs of four tokens, bit 7 - t of their bytes: 1.0 where it is clear, -1.0 where it is set
__device__ __forceinline__ void hw_signs(uint32_t w, int t, uint32_t& e, uint32_t& o) {
  e = hw_and_or(w << (8 + t), 0x80008000u, 0x3C003C00u);
  o = hw_and_or(w << t, 0x80008000u, 0x3C003C00u);
}
// value of the lane four columns up in the row of sixteen, added (columns 0..3)
__device__ __forceinline__ float hw_add_four(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x104 /*row_shl:4*/, 0xf, 0xf, false));
}
__device__ __forceinline__ long hw_as_long(uint32_t a, uint32_t b) { return (long)((uint64_t)a | ((uint64_t)b << 32)); }

// ----------------------------------------------------------------------------------
// tq35 rows
// ----------------------------------------------------------------------------------
// coordinate (inside its part) of byte b of dword r of the score operand, lane group g
__device__ __forceinline__ int hw35_kcoord(int part, int g, int r, int b) {
  if (part == 0) return 8 * (2 * g + (b & 1)) + 2 * r + (b >> 1);
  if (part == 2) return 16 * g + 4 * b + r;
  return 8 * (2 * g + (b & 1)) + r + 4 * (b >> 1);
}

// P: for float32's accuracy -- levels of values in two float16 terms, not one
template <bool P> struct hw35 {
  static constexpr uint32_t MARK = HW_MARK + (P ? 36 : 35);      // (the value levels of the two have factors of their own)
  static constexpr int PER_SIMD = P ? 2 : 3; // wavefronts that the registers admit
  static constexpr float KAPPA = (float)(1.2533141373155001 / 64.0);         // sqrt(pi/2) / 64
  static constexpr int KD = 3;               // digits of a level of keys
  static constexpr int TILE = 1024;          // bytes of sixteen rows in LDS
  static constexpr int NT = 18;              // value tiles: A0 of bytes 0..15 (3), of 16..23 (3), A1 (4), B0 (4), B1 (4)
  // lane (n, g) of a score tile, row n: addresses of its pieces
  uint32_t a0a, a0b, a1, b0, b1;
  uint32_t tr;                               // value tiles: address of the lane's eight bytes of window 0 (of window p: ^ 16 p)
  uint32_t ka0[2 * KD], ka1[KD], va0[P ? 8 : 4], va1[P ? 4 : 2];
  // value side: shifts and masks of the lane's byte of A0 (a third of a group of eight codes)
  uint32_t s0, s1, sown, snb, mown, mnb;
  bool right;
  uint32_t bsh0, bsh1;                       // lanes that take the lower four sign bits

  static __device__ __forceinline__ uint32_t at(uint32_t row, uint32_t o) { return row * 64u + ((((o >> 4) ^ (row >> 2)) & 3u) << 4) + (o & 15u); }

  // buf: the wavefront's chunk buffers; the addresses are those of the first one
  __device__ __forceinline__ hw35(const uint32_t* lut, int lane, uint32_t buf) {
    const uint32_t col = lane & 15, g = lane >> 4;
    a0a = buf + at(col, 6u * g);                             // (bytes 0..3 of six; a piece may end behind them)
    a0b = buf + at(col, 6u * g + 4u);
    a1 = buf + at(col, 36u + 4u * g);
    b0 = buf + at(col, 24u + 2u * g);
    b1 = buf + at(col, 52u + 2u * g);
    // lane 2 r + h of a row of sixteen supplies half h of a window of token r: tokens 4 g .. 4 g + 3 of tile 0, then of tile 1
    const uint32_t r = col >> 1, row = 4u * g + (r & 3u);
    tr = buf + HW_VALUES + (r >> 2) * TILE + row * 64u + (col & 1u) * 8u + (g << 4);
#pragma unroll
    for (int i = 0; i < 2 * KD; ++i) ka0[i] = lut[HW_W_KA0 + i];
#pragma unroll
    for (int i = 0; i < KD; ++i) ka1[i] = lut[HW_W_KA1 + i];
#pragma unroll
    for (int i = 0; i < (P ? 8 : 4); ++i) va0[i] = lut[i < 4 ? HW_W_VA0 + i : HW_W_VP0 + i - 4];
#pragma unroll
    for (int i = 0; i < (P ? 4 : 2); ++i) va1[i] = lut[i < 2 ? HW_W_VA1 + i : HW_W_VP1 + i - 2];
    set_a0(col);
    bsh0 = col >= 8 ? 4u : 0u;
    bsh1 = col >= 4 && col < 12 ? 0u : 4u;
  }
  // byte c of A0: c % 3 = 0 holds codes 0, 1 and the upper two bits of code 2 of its group, 1 the last bit of code 2, codes 3, 4
  // and the first bit of code 5, 2 the rest of code 5 and codes 6, 7
  __device__ __forceinline__ void set_a0(uint32_t c) {
    const uint32_t k = c % 3u;
    s0 = 5u - k;
    s1 = 2u - k;
    right = k == 0;
    sown = k == 0 ? 31u : 6u;
    snb = k == 0 ? 7u : 30u;
    mown = k == 0 ? 0x06060606u : 0x03030303u;
    mnb = k == 0 ? 0x01010101u : 0x04040404u;
  }

  template <int N> static __device__ __forceinline__ void request_tile(const uint8_t* base, int64_t pos, int lane, uint32_t lds) {
    if constexpr (N == 16) {
      const uint32_t row = (uint32_t)lane >> 2, piece = ((uint32_t)lane ^ ((uint32_t)lane >> 4)) & 3u;
      hw_request<16>(base, row * (uint32_t)pos + piece * 16u, lds);
    } else {
#pragma unroll
      for (uint32_t q = 0; q < 4; ++q) {
        const uint32_t row = 4u * q + ((uint32_t)lane >> 4), piece = (((uint32_t)lane >> 2) & 3u) ^ q;
        hw_request<4>(base, row * (uint32_t)pos + piece * 16u + ((uint32_t)lane & 3u) * 4u, lds + 256u * q);
      }
    }
  }
  __device__ __forceinline__ void start(uint32_t) {}
  // the dword of factors of group `group` of row `row`
  static __device__ __forceinline__ uint32_t factors(uint32_t row, int group) { return at(row, group ? 60u : 32u); }
  static __device__ __forceinline__ uint32_t look8(uint32_t t0, uint32_t t1, uint32_t sel) { return __builtin_amdgcn_perm(t1, t0, sel); }

  // sums of the four parts for the tokens of both tiles of the buffer `keys` bytes on: t[8] = f . (A0, B0, A1, B1), f from `fac`
  __device__ __forceinline__ void scores(uint32_t keys, uint32_t fac, uint32_t query, float (&t)[8]) const {
    auto q = [&](int part) __attribute__((always_inline)) { return *(hw_lds_i128*)(uintptr_t)(query + HW_Q_PART * part); };
    // two bytes of the lane's six of A0 a word, tile 0 below tile 1
    auto two = [&](uint32_t o) __attribute__((always_inline)) {
      const hw_ushort2 v = {*(hw_lds_cu16*)(uintptr_t)(o + keys), *(hw_lds_cu16*)(uintptr_t)(o + keys + TILE)};
      union { hw_ushort2 v; uint32_t u; } x;
      x.v = v;
      return x.u;
    };
    const uint32_t w0 = two(a0a), w1 = two(a0a + 2u), w2 = two(a0b);
    uint32_t a1w[2], s[2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      a1w[j] = *(hw_lds_cu32*)(uintptr_t)(a1 + keys + TILE * j);
      s[j][0] = *(hw_lds_cu16*)(uintptr_t)(b0 + keys + TILE * j);
      s[j][1] = *(hw_lds_cu16*)(uintptr_t)(b1 + keys + TILE * j);
    }
    // bytes 0, 1, 2 of the lane's two groups of A0, of both tiles side by side; then its eight codes, a word each
    uint32_t b[3], c[8];
    b[0] = __builtin_amdgcn_perm(w1, w0, 0x07020500u);
    b[1] = __builtin_amdgcn_perm(w2, w0, 0x06030401u);
    b[2] = __builtin_amdgcn_perm(w2, w1, 0x07020500u);
    c[0] = (b[0] >> 5) & 0x07070707u;
    c[1] = (b[0] >> 2) & 0x07070707u;
    c[2] = ((b[0] << 1) & 0x06060606u) | ((b[1] >> 7) & 0x01010101u);
    c[3] = (b[1] >> 4) & 0x07070707u;
    c[4] = (b[1] >> 1) & 0x07070707u;
    c[5] = ((b[1] << 2) & 0x04040404u) | ((b[2] >> 6) & 0x03030303u);
    c[6] = (b[2] >> 3) & 0x07070707u;
    c[7] = b[2] & 0x07070707u;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const hw_int4 zero = {0, 0, 0, 0};
      hw_int4 a0[KD], a1s[KD], sg[2];       // sums: digits of the levels, top first; signs
      {
        uint32_t sel[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) sel[r] = __builtin_amdgcn_perm(c[2 * r + 1], c[2 * r], j ? 0x07060302u : 0x05040100u);
#pragma unroll
        for (int d = 0; d < KD; ++d) {
          hw_int4 v;
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = (int)look8(ka0[2 * d], ka0[2 * d + 1], sel[r]);
          a0[d] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v, q(0), zero, 0, 0, 0);
        }
      }
      {
        uint32_t sel[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) sel[r] = (a1w[j] >> (6 - 2 * r)) & 0x03030303u;
#pragma unroll
        for (int d = 0; d < KD; ++d) {
          hw_int4 v;
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = (int)__builtin_amdgcn_perm(ka1[d], ka1[d], sel[r]);
          a1s[d] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v, q(2), zero, 0, 0, 0);
        }
      }
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const uint32_t both = s[j][x] | (s[j][x] << 20);      // two bytes, and the two moved up by four bits
        hw_int4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = (int)hw_and_or(both << r, 0x80808080u, 0x40404040u);
        sg[x] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v, q(1 + 2 * x), zero, 0, 0, 0);
      }
      auto whole = [&](const hw_int4 (&d)[KD], int i) __attribute__((always_inline)) {
        return fmaf((float)d[0][i], 65536.f, (float)((d[1][i] << 8) + d[2][i]));
      };
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const hw_float4 f = *(hw_lds_f128*)(uintptr_t)(fac + 256u * j + 16u * i);
        float x = whole(a0, i) * f[0];
        x = fmaf((float)sg[0][i], f[1], x);
        x = fmaf(whole(a1s, i), f[2], x);
        t[4 * j + i] = fmaf((float)sg[1][i], f[3], x);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  template <class W> __device__ __forceinline__ void values(uint32_t keys, W weights, hw_float4 (&o)[NT]) const {
    hw_int2 win[4];
#pragma unroll
    for (uint32_t p = 0; p < 4; ++p) win[p] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((hw_lds_i64*)(uintptr_t)((tr ^ (p << 4)) + keys));
    auto product = [&](int tile, const hw_half8& w, uint32_t (&a)[4]) __attribute__((always_inline)) {
      o[tile] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hw_operand(a[0], a[1], a[2], a[3]), w, o[tile], 0, 0, 0);
    };
    // ---- A0: bytes 0..15 a lane each, then bytes 16..23 in lanes 1..8 (so that a lane's byte is of the same class in both)
    {
      const hw_half8 w = weights(0);
#pragma unroll
      for (int part = 0; part < 2; ++part) {
        uint32_t sel[3][2];
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const int x = win[0][d], y = win[1][d];
          uint32_t own, nb;
          if (part == 0) {
            const int wrap = __builtin_amdgcn_update_dpp(0, y, 0x12f /*row_ror:15*/, 0xf, 0xf, false);      // byte 16 beside byte 15
            const int xr = __builtin_amdgcn_update_dpp(wrap, x, 0x101 /*row_shl:1*/, 0xf, 0xf, false);
            const int xl = __builtin_amdgcn_update_dpp(0, x, 0x111 /*row_shr:1*/, 0xf, 0xf, false);
            own = (uint32_t)x;
            nb = (uint32_t)(right ? xr : xl);
          } else {
            const int yl = __builtin_amdgcn_update_dpp(0, y, 0x112 /*row_shr:2*/, 0xf, 0xf, false);
            own = (uint32_t)__builtin_amdgcn_update_dpp(0, y, 0x111 /*row_shr:1*/, 0xf, 0xf, false);
            nb = (uint32_t)(right ? y : yl);
          }
          sel[0][d] = (own >> s0) & 0x07070707u;
          sel[1][d] = (own >> s1) & 0x07070707u;
          sel[2][d] = (__builtin_amdgcn_alignbit(own, own, sown) & mown) | (__builtin_amdgcn_alignbit(nb, nb, snb) & mnb);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int term = 0; term < (P ? 2 : 1); ++term) {
            uint32_t a[4];
            const uint32_t* lv = va0 + 4 * term;
#pragma unroll
            for (int d = 0; d < 2; ++d) hw_expand(look8(lv[0], lv[1], sel[i][d]), look8(lv[2], lv[3], sel[i][d]), a[2 * d], a[2 * d + 1]);
            product(3 * part + i, w, a);
          }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- A1: window 2 from lane 4 on, window 3 in lanes 0..3
    const hw_half8 wa1 = weights(2);
    uint32_t b1w[2];
#pragma unroll
    for (int d = 0; d < 2; ++d) b1w[d] = (uint32_t)__builtin_amdgcn_update_dpp(win[2][d], win[3][d], 0xE4 /*the lane's own*/, 0xf, 0x1, false);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int term = 0; term < (P ? 2 : 1); ++term) {
        uint32_t a[4];
        const uint32_t* lv = va1 + 2 * term;
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const uint32_t c = (b1w[d] >> (6 - 2 * i)) & 0x03030303u;
          hw_expand(__builtin_amdgcn_perm(lv[0], lv[0], c), __builtin_amdgcn_perm(lv[1], lv[1], c), a[2 * d], a[2 * d + 1]);
        }
        product(6 + i, wa1, a);
      }
    __builtin_amdgcn_sched_barrier(0);
    // ---- B0: window 1, bytes in lanes 8..15, which take the lower four bits; lanes 0..7 have them again and take the upper four.
    // B1: window 3, lanes 4..11 (upper four), lanes 12..15 and 0..3 have them again
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const hw_half8 wb = weights(1 + 2 * x);
      uint32_t w[2];
#pragma unroll
      for (int d = 0; d < 2; ++d)
        w[d] = x == 0 ? (uint32_t)__builtin_amdgcn_update_dpp(win[1][d], win[1][d], 0x128 /*row_ror:8*/, 0xf, 0x3, false) << bsh0
                      : (uint32_t)__builtin_amdgcn_update_dpp(win[3][d], win[3][d], 0x128 /*row_ror:8*/, 0xf, 0x9, false) << bsh1;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        uint32_t a[4];
#pragma unroll
        for (int d = 0; d < 2; ++d) hw_signs(w[d], i, a[2 * d], a[2 * d + 1]);
        product(10 + 4 * x + i, wb, a);
      }
    }
  }
  // row m of all value tiles: store(place among the 256 sums of a head, tile).  Tiles come in an order in which a row that holds
  // nothing is stored where a later one of the same lane belongs.
  template <class S> static __device__ __forceinline__ void places(int m, S store) {
    const int k = m % 3;
    const int x = m / 3 * 8 + (k == 0 ? 0 : k == 1 ? 3 : 6), y = (m + 15) / 3 * 8 + (k == 0 ? 0 : k == 1 ? 3 : 6);
    const bool held = m >= 1 && m <= 8;                   // bytes 16..23
    const int back = k == 0 ? 2 : k == 1 ? 0 : -1;        // code 2 of the class: places beyond code 0 (class 1 has two)
    store(held ? y + back : x, 5);
    store(held ? y : x, 3);
    store(held ? y + 1 : x, 4);
    store(x + back, 2);
    store(x, 0);
    store(x + 1, 1);
    const int a1 = 128 + 4 * (m >= 4 ? m - 4 : 12 + m), b0 = 64 + (m < 8 ? 8 * m : 8 * (m - 8) + 4);
    const int b1 = 192 + (m < 4 ? 8 * (m + 4) + 4 : m < 12 ? 8 * (m - 4) : 8 * (m - 12) + 4);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      store(a1 + t, 6 + t);
      store(b0 + t, 10 + t);
      store(b1 + t, 14 + t);
    }
  }
  // constants of the factors: (n0, n0 r0, n1, n1 r1) times these on the score side
  static __device__ __forceinline__ hw_float4 kscale(const uint32_t* lut) {
    const float sign = -KAPPA / 64.f;
    return (hw_float4){__uint_as_float(lut[HW_W_UNIT]), sign, __uint_as_float(lut[HW_W_UNIT + 1]), sign};
  }
  // row i of the lane's rows of the finished tiles
  static __device__ __forceinline__ void finish(const uint32_t* lut, hw_float4 (&o)[NT], int i, float (&v)[NT]) {
    const float ia0 = 1.f / __uint_as_float(lut[HW_W_ALPHA]), ia1 = 1.f / __uint_as_float(lut[HW_W_ALPHA + 1]);
#pragma unroll
    for (int n = 0; n < NT; ++n) v[n] = hw_add_four(o[n][i]) * (n < 6 ? ia0 : n < 10 ? ia1 : -KAPPA);
  }
  // ---- transforms of queries and outputs: lane l holds four of the 256 sums' coordinates
  static __device__ __forceinline__ int sum_of(int lane, int p) { return 64 * p + lane; }
  // the sum faced by byte b of dword r of slot x of the query operand, lane group g
  static __device__ __forceinline__ int faced(int x, int g, int r, int b) { return 64 * x + hw35_kcoord(x, g, r, b); }
  static __device__ __forceinline__ int coord(int lane, int i) { return 64 * i + lane; }
  static __device__ __forceinline__ void forward(float q0, float q1, int lane, const float* table, float (&y)[4]) {
    y[0] = hyb_fwht64(q0 * table[HYB_HAD0 + lane], lane) * 0.125f;
    y[1] = hyb_fwht64(q0 * table[HYB_QJL0 + lane], lane) * 0.125f;
    y[2] = hyb_fwht64(q1 * table[HYB_HAD1 + lane], lane) * 0.125f;
    y[3] = hyb_fwht64(q1 * table[HYB_QJL1 + lane], lane) * 0.125f;
  }
  static __device__ __forceinline__ void back(const float (&acc)[4], int lane, const float* table, float& o0, float& o1) {
    o0 = (hyb_fwht64(acc[0], lane) * table[HYB_HAD0 + lane] + hyb_fwht64(acc[1], lane) * table[HYB_QJL0 + lane]) * 0.125f;
    o1 = (hyb_fwht64(acc[2], lane) * table[HYB_HAD1 + lane] + hyb_fwht64(acc[3], lane) * table[HYB_QJL1 + lane]) * 0.125f;
  }
  static constexpr int TAGS = 12, TAG_AT = HYB_CEN0;        // the codebooks, which the tables are built from
  static __device__ void tables(const float* table, uint32_t* lut);
};

// ----------------------------------------------------------------------------------
// tq25 rows (44 bytes): A0 32 codes of 2 bits, B0 32 signs, two factors, A1 96 codes of 1 bit, B1 96 signs, two factors
// ----------------------------------------------------------------------------------
// In LDS a row is twelve dwords: A0 A0 B0 f0 | A1 A1 A1 f1 | B1 B1 B1 f1 (16 rows of 48 bytes meet sixteen different sets of banks).
// A code of one bit is a sign around the middle of its two levels: c = middle - delta (+-1).  The sum of the query against the
// middle is a constant of the head, and the sum of the weights comes out of the value product in a row nobody else has.
struct hw25 {
  static constexpr uint32_t MARK = HW_MARK + 25;
  static constexpr int PER_SIMD = 3;
  static constexpr int TILE = 768;
  static constexpr int NT = 20;              // value tiles: A0 (2), B0 (2), A1 (8), B1 (8)
  static constexpr int SUM_B = 128;          // sums: A0 0..31, A1 32..127, B0 and B1 from 128 on in the same order
  uint32_t half, byte;                       // lane (n, g) of a score tile: address of row n, plus 2 g, plus g
  uint32_t tr;
  uint32_t ka[3], va[4];
  float delta;
  uint32_t sh4, sh2, not15;
  float middle;                              // what the middle of the 1-bit levels adds, for the lane's column

  __device__ __forceinline__ hw25(const uint32_t* lut, int lane, uint32_t buf) {
    const uint32_t col = lane & 15, g = lane >> 4;
    half = buf + col * 48u + 2u * g;
    byte = buf + col * 48u + g;
    const uint32_t r = col >> 1, row = 4u * g + (r & 3u);
    tr = buf + HW_VALUES + (r >> 2) * TILE + row * 48u + (col & 1u) * 8u;
#pragma unroll
    for (int i = 0; i < 3; ++i) ka[i] = lut[HW_W_KA1 + i];
#pragma unroll
    for (int i = 0; i < 4; ++i) va[i] = lut[i < 2 ? HW_W_VA1 + i : HW_W_VP1 + i - 2];
    delta = __uint_as_float(lut[HW_W_DELTA]);
    middle = __uint_as_float(lut[HW_W_MIDDLE]) * -64.f;
    sh4 = col >= 8 ? 4u : 0u;
    sh2 = 2u * (col >> 2);
    not15 = col == 15 ? 0u : ~0u;
  }
  template <int N> static __device__ __forceinline__ void request_tile(const uint8_t* base, int64_t pos, int lane, uint32_t lds) {
    static_assert(N == 4, "rows of eleven dwords");
#pragma unroll
    for (uint32_t q = 0; q < 3; ++q) {
      const uint32_t i = 64u * q + (uint32_t)lane, row = i / 12u, at = i % 12u, from = at < 7u ? at : at == 7u || at == 11u ? 10u : at - 1u;
      hw_request<4>(base, row * (uint32_t)pos + from * 4u, lds + 256u * q);
    }
  }
  // (the sum of the query integers over the 96 coordinates, column by column, against ones)
  __device__ __forceinline__ void start(uint32_t query) {
    const hw_int4 ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
    const hw_int4 zero = {0, 0, 0, 0};
    const hw_int4 a = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, *(hw_lds_i128*)(uintptr_t)(query + HW_Q_PART), zero, 0, 0, 0);
    const hw_int4 b = __builtin_amdgcn_mfma_i32_16x16x32_i8(hw_as_long(0x01010101u, 0x01010101u), *(hw_lds_l64*)(uintptr_t)(query + 2 * HW_Q_PART), zero, 0, 0, 0);
    middle_now = middle * (float)(a[0] + b[0]);
  }
  float middle_now;
  static __device__ __forceinline__ uint32_t factors(uint32_t row, int group) { return row * 48u + (group ? 28u : 12u); }

  __device__ __forceinline__ void scores(uint32_t keys, uint32_t fac, uint32_t query, float (&t)[8]) const {
    auto q16 = [&](int slot) __attribute__((always_inline)) { return *(hw_lds_i128*)(uintptr_t)(query + HW_Q_PART * slot); };
    auto q8 = [&](int slot, int up) __attribute__((always_inline)) { return *(hw_lds_l64*)(uintptr_t)(query + HW_Q_PART * slot + 8u * up); };
    uint32_t a0[2], b0[2], h[2][2], e[2][2];      // two bytes of A0, one of B0; two and one of A1, B1
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      a0[j] = *(hw_lds_cu16*)(uintptr_t)(half + keys + TILE * j);
      b0[j] = *(hw_lds_cu8*)(uintptr_t)(byte + keys + TILE * j + 8u);
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        h[j][x] = *(hw_lds_cu16*)(uintptr_t)(half + keys + TILE * j + 16u + 16u * x);
        e[j][x] = *(hw_lds_cu8*)(uintptr_t)(byte + keys + TILE * j + 24u + 16u * x);
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const hw_int4 zero = {0, 0, 0, 0};
      auto eight = [&](uint32_t v) __attribute__((always_inline)) {      // a byte's signs: bits 7 - b in byte b, then 3 - b
        uint32_t x = v | (v << 9);
        x = x | (x << 18);
        return hw_as_long(hw_and_or(x, 0x80808080u, 0x40404040u), hw_and_or(x << 4, 0x80808080u, 0x40404040u));
      };
      // (the two products of a part are added up here: wrong sums came out when the second one, of another shape, started from the
      // first one's.  Why was not found.)
      hw_int4 c[3], sg[3], sh[2];
      {
        const uint32_t x = a0[j] | (a0[j] << 18), s0 = (x >> 6) & 0x03030303u, s1 = (x >> 2) & 0x03030303u;
#pragma unroll
        for (int d = 0; d < 3; ++d)
          c[d] = __builtin_amdgcn_mfma_i32_16x16x32_i8(hw_as_long(__builtin_amdgcn_perm(ka[d], ka[d], s0), __builtin_amdgcn_perm(ka[d], ka[d], s1)), q8(0, 0), zero, 0, 0, 0);
      }
      sg[2] = __builtin_amdgcn_mfma_i32_16x16x32_i8(eight(b0[j]), q8(0, 1), zero, 0, 0, 0);
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const uint32_t both = h[j][x] | (h[j][x] << 20);
        hw_int4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = (int)hw_and_or(both << r, 0x80808080u, 0x40404040u);
        sg[x] = __builtin_amdgcn_mfma_i32_16x16x64_i8(v, q16(1 + 2 * x), zero, 0, 0, 0);
        sh[x] = __builtin_amdgcn_mfma_i32_16x16x32_i8(eight(e[j][x]), q8(2, x), zero, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const hw_float4 f = *(hw_lds_f128*)(uintptr_t)(fac + 256u * j + 16u * i);
        float x = fmaf((float)c[0][i], 65536.f, (float)((c[1][i] << 8) + c[2][i])) * f[0];
        x = fmaf((float)sg[2][i], f[1], x);
        x = fmaf(fmaf((float)(sg[0][i] + sh[0][i]), delta, middle_now), f[2], x);
        t[4 * j + i] = fmaf((float)(sg[1][i] + sh[1][i]), f[3], x);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  template <class W> __device__ __forceinline__ void values(uint32_t keys, W weights, hw_float4 (&o)[NT]) const {
    hw_int2 win[3];
#pragma unroll
    for (uint32_t p = 0; p < 3; ++p) win[p] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((hw_lds_i64*)(uintptr_t)(tr + keys + 16u * p));
    auto product = [&](int tile, const hw_half8& w, uint32_t (&a)[4]) __attribute__((always_inline)) {
      o[tile] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hw_operand(a[0], a[1], a[2], a[3]), w, o[tile], 0, 0, 0);
    };
    // ---- A0: bytes in lanes 0..7 (upper two codes), again in 8..15 (lower two)
    {
      const hw_half8 w = weights(0);
      uint32_t c[2];
#pragma unroll
      for (int d = 0; d < 2; ++d) c[d] = (uint32_t)__builtin_amdgcn_update_dpp(win[0][d], win[0][d], 0x128 /*row_ror:8*/, 0xf, 0xc, false) << sh4;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int term = 0; term < 2; ++term) {
          uint32_t a[4];
#pragma unroll
          for (int d = 0; d < 2; ++d) {
            const uint32_t sel = (c[d] >> (6 - 2 * i)) & 0x03030303u;
            hw_expand(__builtin_amdgcn_perm(va[2 * term], va[2 * term], sel), __builtin_amdgcn_perm(va[2 * term + 1], va[2 * term + 1], sel), a[2 * d], a[2 * d + 1]);
          }
          product(i, w, a);
        }
    }
    // ---- B0: four bytes in lanes 8..11, again in every four lanes; bank k takes bits 7 - 2 k and 6 - 2 k
    {
      const hw_half8 w = weights(1);
      uint32_t b[2];
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        int x = __builtin_amdgcn_update_dpp(win[0][d], win[0][d], 0x108 /*row_shl:8*/, 0xf, 0x1, false);
        x = __builtin_amdgcn_update_dpp(x, win[0][d], 0x104 /*row_shl:4*/, 0xf, 0x2, false);
        x = __builtin_amdgcn_update_dpp(x, win[0][d], 0x114 /*row_shr:4*/, 0xf, 0x8, false);
        b[d] = (uint32_t)x << sh2;
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        uint32_t a[4];
#pragma unroll
        for (int d = 0; d < 2; ++d) hw_signs(b[d], i, a[2 * d], a[2 * d + 1]);
        product(2 + i, w, a);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- A1 and B1: twelve bytes in lanes 0..11, a bit a tile.  (Lane 15 of A1's: +1 for every token, the sum of the weights.)
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const hw_half8 w = weights(2 + x);
      uint32_t b[2];
#pragma unroll
      for (int d = 0; d < 2; ++d) b[d] = x == 0 ? (uint32_t)win[1][d] & not15 : (uint32_t)win[2][d];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        uint32_t a[4];
#pragma unroll
        for (int d = 0; d < 2; ++d) hw_signs(b[d], i, a[2 * d], a[2 * d + 1]);
        product(4 + 8 * x + i, w, a);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  template <class S> static __device__ __forceinline__ void places(int m, S store) {
    // (rows 12..15 of A1 and B1 hold nothing: stored where A0 and B0 of the same lane belong, which come later)
    const int a0 = m < 8 ? 4 * m : 4 * (m - 8) + 2, b0 = SUM_B + 8 * (m & 3) + 2 * (m >> 2);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      store(m < 12 ? 32 + 8 * m + t : a0, 4 + t);
      store(m < 12 ? SUM_B + 32 + 8 * m + t : b0, 12 + t);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      store(a0 + t, t);
      store(b0 + t, 2 + t);
    }
  }
  static __device__ __forceinline__ hw_float4 kscale(const uint32_t* lut) {
    return (hw_float4){__uint_as_float(lut[HW_W_UNIT + 1]), -kH25Kappa0 / 64.f, -1.f / 64.f, -kH25Kappa1 / 64.f};
  }
  static __device__ __forceinline__ void finish(const uint32_t* lut, hw_float4 (&o)[NT], int i, float (&v)[NT]) {
    const float ia = 1.f / __uint_as_float(lut[HW_W_ALPHA + 1]), dl = __uint_as_float(lut[HW_W_DELTA]), md = __uint_as_float(lut[HW_W_MIDDLE]);
    const float all = __shfl(hw_add_four(o[4][3]), 48 + (int)(threadIdx.x & 15)) * md;      // (row 15 of A1's tiles)
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const float x = hw_add_four(o[n][i]);
      v[n] = n < 2 ? x * ia : n < 4 ? x * -kH25Kappa0 : n < 12 ? fmaf(x, -dl, all) : x * -kH25Kappa1;
    }
  }
  static __device__ __forceinline__ int sum_of(int lane, int p) { return (p & 1 ? SUM_B : 0) + coord(lane, p >> 1); }
  static __device__ __forceinline__ int faced(int x, int g, int r, int b) {
    const int eight = 8 * g + 4 * (r & 1) + b;       // of a byte a lane group
    if (x == 0) return r < 2 ? 4 * (2 * g + (b & 1)) + 2 * r + (b >> 1) : SUM_B + eight;
    if (x == 2) return (r < 2 ? 32 : SUM_B + 32) + 64 + eight;
    return (x == 1 ? 32 : SUM_B + 32) + 8 * (2 * g + (b & 1)) + r + 4 * (b >> 1);
  }
  static __device__ __forceinline__ int coord(int lane, int i) {
    const h25_roles r(lane);
    return i == 0 ? r.ca : r.cb;
  }
  static __device__ __forceinline__ void forward(float qa, float qb, int lane, const float* table, float (&y)[4]) {
    const h25_roles r(lane);
    const float root_b = r.b0 ? kH25Root0 : kH25Root1;
    y[0] = hyb_fwht64(qa * table[H25_HAD + r.ca], lane) / kH25Root1;
    y[1] = hyb_fwht64(qa * table[H25_QJL + r.ca], lane) / kH25Root1;
    y[2] = h25_fwht32(qb * table[H25_HAD + r.cb], lane) / root_b;
    y[3] = h25_fwht32(qb * table[H25_QJL + r.cb], lane) / root_b;
  }
  static __device__ __forceinline__ void back(const float (&acc)[4], int lane, const float* table, float& o0, float& o1) {
    const h25_roles r(lane);
    const float inv_b = r.b0 ? 1.f / kH25Root0 : 1.f / kH25Root1;
    o0 = (hyb_fwht64(acc[0], lane) * table[H25_HAD + r.ca] + hyb_fwht64(acc[1], lane) * table[H25_QJL + r.ca]) * (1.f / kH25Root1);
    o1 = (h25_fwht32(acc[2], lane) * table[H25_HAD + r.cb] + h25_fwht32(acc[3], lane) * table[H25_QJL + r.cb]) * inv_b;
  }
  static constexpr int TAGS = 6, TAG_AT = H25_CEN0;
  static __device__ void tables(const float* table, uint32_t* lut);
};

// ----------------------------------------------------------------------------------
// main kernel
// ----------------------------------------------------------------------------------
// N: bytes of a request, 16 where rows allow it, else 4
template <class F, int N>
__global__ __launch_bounds__(HW_W * 64, F::PER_SIMD) void akv_attn_hyb_kernel(hw_args a) {
  // The dynamic LDS block is the kernel's only LDS object: its offsets are LDS addresses.
  constexpr int NT = F::NT;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, g = lane >> 4;
  const int range = blockIdx.x / a.hgroups, hset = blockIdx.x % a.hgroups;
  const int32_t* rec = a.wgdesc + (size_t)range * AKV_WGREC;
  const int g0 = rec[AKV_WGREC_G0], g1 = rec[AKV_WGREC_G1], s_first = rec[AKV_WGREC_SEQ];
  const int sb0_first = rec[AKV_WGREC_SB0], sb1_first = rec[AKV_WGREC_SB1], ctx_first = rec[AKV_WGREC_CTX];
  if (g0 >= g1) return;

  const bool bs32 = a.block_size == 32;
  const int bs = bs32 ? 32 : 16;
  const int hp = a.hp, R = HW_W / hp;
  const int hs = wave % hp, r = wave / hp;
  const int h = hset * hp + hs;
  const bool active = h < a.KVH;
  const int hd = h / a.hgroup, sub = h % a.hgroup;         // the head whose rows are read, which of its groups of query heads
  const int q0 = hd * a.gqa + 4 * sub, nq = min(4, a.gqa - 4 * sub);
  const uint32_t buf = (uint32_t)wave * HW_BUF;
  F f(a.lut, lane, buf);
  const uint32_t fac_at = HW_FAC + (uint32_t)wave * HW_FAC_WAVE;
  const uint32_t fread = fac_at + (uint32_t)g * 64u;       // key factors of tokens 4 g of tile 0
  const int kb = (lane >> 2) & 3;                          // softmax: the lane has tokens kb % 2 and 2 + kb % 2 of tile kb / 2
  const int tok = 16 * (kb >> 1) + 4 * g + (kb & 1);
  // (place of value token t: t % 4 first, so that the sixteen tokens read together lie side by side)
  auto vplace = [](int t) { return (uint32_t)((t & 3) * 8 + (t >> 2)) * 32u; };
  const uint32_t vread = fac_at + 512u + vplace(tok);
  // factors: lanes 0..31 a key each, 32..63 a value each
  const hw_float4 ks = F::kscale(a.lut);
  const uint32_t fsrc = buf + (uint32_t)(lane >> 5) * HW_VALUES + (uint32_t)((lane >> 4) & 1) * F::TILE;
  const uint32_t fsrc0 = fsrc + F::factors(col, 0), fsrc1 = fsrc + F::factors(col, 1);
  const uint32_t fwrite = fac_at + (lane < 32 ? (uint32_t)lane * 16u : 512u + vplace(lane & 31));
  // digits of a head's scores, columns 4 d + c: place 4 (d ^ g) + c of the lane group, so that groups meet different banks
  const uint32_t twrite = buf + (uint32_t)(g * 256 + (col ^ (4 * g)) * 16);
  const uint32_t tread = buf + (uint32_t)((kb >> 1) * 1024 + g * 256 + (4 * g + (col & 3)) * 16 + (kb & 1) * 8);      // digit d: ^ 64 d
  const uint32_t wwrite = buf + (uint32_t)(g * 64 + (col & 3) * 16 + kb * 4);
  const uint32_t wread = buf + (uint32_t)(g * 64 + (col & 3) * 16 + ((col >> 2) & 1) * 256);
  const uint32_t qat = HW_Q + (uint32_t)wave * 4u * HW_Q_PART + (uint32_t)(12 * g + min(col, 11)) * 16u;     // (columns 12..15: scaled by zero)
  const uint8_t* kbase = a.kc + (int64_t)hd * a.kps_head;
  const uint8_t* vbase = a.vc + (int64_t)hd * a.vps_head;

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

    float m_run = -INFINITY, l_run = 0.f;
    hw_float4 o[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) o[n] = (hw_float4){0.f, 0.f, 0.f, 0.f};

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
      auto request = [&](int k) {
        if (k - win_k >= HW_WIN) load_window(k);
        const int w = bs32 ? k - win_k : 2 * (k - win_k);
        const uint32_t pb0 = (uint32_t)__builtin_amdgcn_readlane(pbwin, w), pb1 = bs32 ? pb0 : (uint32_t)__builtin_amdgcn_readlane(pbwin, w + 1);
        const uint32_t to = buf + (k & 1 ? HW_BUF / 2 : 0u);
        F::template request_tile<N>(kbase + (uint64_t)pb0 * (uint32_t)a.kps_blk, a.kps_pos, lane, to);
        F::template request_tile<N>(kbase + (uint64_t)pb1 * (uint32_t)a.kps_blk + (bs32 ? 16 * a.kps_pos : 0), a.kps_pos, lane, to + F::TILE);
        F::template request_tile<N>(vbase + (uint64_t)pb0 * (uint32_t)a.vps_blk, a.vps_pos, lane, to + HW_VALUES);
        F::template request_tile<N>(vbase + (uint64_t)pb1 * (uint32_t)a.vps_blk + (bs32 ? 16 * a.vps_pos : 0), a.vps_pos, lane, to + HW_VALUES + F::TILE);
      };
      load_window(0);
      request(0);
      {
        const uint4* qp = a.qop + (size_t)(s * a.KVH + h) * 256 + lane;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const uint4 u = qp[p * 64];
          if (col < 12) *(hw_lds_i128*)(uintptr_t)(qat + HW_Q_PART * p) = hw_as_int4(u);
        }
      }
      akv_wave_sync();
      f.start(qat);
      const float qfac = a.fac[(size_t)s * a.QH + q0 + min(col & 3, nq - 1)];

      for (int k = 0; k < mine; ++k) {
        const uint32_t keys = k & 1 ? HW_BUF / 2 : 0u;      // (two copies of the body, the buffer in their instructions, spill)
        const int c = r + k * R;
        hw_landed();
        if (k + 1 < mine) request(k + 1);

        // ---- factors of the chunk's rows: n0, n0 r0, n1, n1 r1; of values their largest exponent too
        {
          union { uint32_t u; hw_half2 h; } u0, u1;
          u0.u = *(hw_lds_cu32*)(uintptr_t)(fsrc0 + keys);
          u1.u = *(hw_lds_cu32*)(uintptr_t)(fsrc1 + keys);
          const float n0 = (float)u0.h[0], n1 = (float)u1.h[0], x0 = n0 * (float)u0.h[1], x1 = n1 * (float)u1.h[1];
          int half = lane;
          asm volatile("" : "+v"(half));        // (the four choices would be kept in registers)
          const bool key = half < 32;
          *(hw_lds_f128*)(uintptr_t)fwrite = (hw_float4){key ? n0 * ks[0] : n0, key ? x0 * ks[1] : x0, key ? n1 * ks[2] : n1, key ? x1 * ks[3] : x1};
          if (!key) {
            const float top = fmaxf(fmaxf(fabsf(n0), fabsf(x0)), fmaxf(fabsf(n1), fabsf(x1)));
            const int e = (int)((__float_as_uint(top) >> 23) & 0xffu) - 126;
            *(hw_lds_f32*)(uintptr_t)(fwrite + 16u) = (float)max(e, -HW_TINY);
          }
        }
        akv_wave_sync();

        float t[8];
        f.scores(keys, fread, qat, t);
        __builtin_amdgcn_sched_barrier(0);      // (stages kept apart: interleaved they need more registers than three wavefronts have)
        // ---- a lane's tokens come from the columns of its head's three digits, through the place of the keys (done with): plane
        // of a tile, lane, tokens 0 2 1 3.  (Adding up over the lanes of a row by row shifts is 28 vector instructions more.)
        *(hw_lds_f128*)(uintptr_t)(twrite + keys) = (hw_float4){t[0], t[2], t[1], t[3]};
        *(hw_lds_f128*)(uintptr_t)(twrite + keys + 1024u) = (hw_float4){t[4], t[6], t[5], t[7]};
        akv_wave_sync();
        float sv[2], tv[2];
        {
          hw_float2 dg[3];
#pragma unroll
          for (int d = 0; d < 3; ++d) dg[d] = *(hw_lds_f64*)(uintptr_t)((tread ^ (64u * d)) + keys);
#pragma unroll
          for (int jj = 0; jj < 2; ++jj) sv[jj] = fmaf(fmaf(dg[0][jj], 256.f, dg[1][jj]), 256.f, dg[2][jj]) * qfac;
        }
        hw_float4 vf[2];
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
          vf[jj] = *(hw_lds_f128*)(uintptr_t)(vread + 512u * jj);
          tv[jj] = sv[jj] + *(hw_lds_f32*)(uintptr_t)(vread + 512u * jj + 16u);
        }
        if (c == nchunks - 1) {        // only the last chunk of a segment holds tokens past its end, whose rows may hold anything
          asm volatile("");            // (keeps this a branch)
#pragma unroll
          for (int jj = 0; jj < 2; ++jj)
            if (blk_lo * bs + 32 * c + tok + 2 * jj >= t_end) {
              sv[jj] = -INFINITY;
              tv[jj] = -INFINITY;
              vf[jj] = (hw_float4){0.f, 0.f, 0.f, 0.f};
            }
        }
        // ---- running softmax in the log2 domain over t = score + exponent of the value factors
        // (the frame moves only when the maximum has outgrown it: moving the sums costs more than all of the softmax, and looking
        // for the maximum over the lanes some 25 instructions: a step of 64 contexts of 4,000 to 8,192 168.1 -> 165.7 us)
        if (__builtin_amdgcn_ballot_w64(tv[0] > m_run + (HW_FRAME + HW_SLACK) || tv[1] > m_run + (HW_FRAME + HW_SLACK)) != 0) {
          const float mx = akv_rows_max(akv_banks_max(fmaxf(tv[0], tv[1])));
          const float m_new = mx - HW_FRAME > m_run + HW_SLACK ? mx - HW_FRAME : m_run;
          const float resc = __builtin_amdgcn_exp2f(m_run - m_new);      // 0 on the first chunk
          m_run = m_new;
          l_run *= resc;
#pragma unroll
          for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[n][i] *= resc;
        }
        const float p0 = __builtin_amdgcn_exp2f(sv[0] - m_run), p1 = __builtin_amdgcn_exp2f(sv[1] - m_run);
        l_run += p0 + p1;
        // ---- weights of the four parts, two float16 terms each, in the same place: part, term, lane group, head, token pair.
        // Columns 0..3 read term 0, 4..7 term 1 (8..15 the same again, for nobody).
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const hw_float2 w2 = {p0 * vf[0][x], p1 * vf[1][x]};
          const hw_half2 h2 = __builtin_convertvector(w2, hw_half2);
          const hw_half2 l2 = __builtin_convertvector(w2 - __builtin_convertvector(h2, hw_float2), hw_half2);
          union { hw_half2 h; uint32_t u; } hu, lu;
          hu.h = h2;
          lu.h = l2;
          *(hw_lds_u32*)(uintptr_t)(wwrite + keys + 512u * x) = hu.u;
          *(hw_lds_u32*)(uintptr_t)(wwrite + keys + 512u * x + 256u) = lu.u;
        }
        akv_wave_sync();
        auto weights = [&](int x) __attribute__((always_inline)) {
          const hw_int4 w = *(hw_lds_i128*)(uintptr_t)(wread + keys + 512u * x);
          return hw_operand((uint32_t)w[0], (uint32_t)w[1], (uint32_t)w[2], (uint32_t)w[3]);
        };
        __builtin_amdgcn_sched_barrier(0);
        f.values(keys, weights, o);
      }
      l_run = akv_banks_sum(akv_rows_sum(l_run));
    }

    // ---- partial result: sums in natural order through the wavefront's buffer, shares of a head merged
    const size_t slot = (size_t)(range + s) * a.QH + q0;
    const int shares = min(R, nchunks);      // wavefronts of the head that hold a result
    float M = m_run, wgt = 1.f, L = l_run;
    if (shares > 1) {
      if (lane < 4) *(hw_lds_f64*)(uintptr_t)(HW_ML + (uint32_t)wave * 32u + (uint32_t)lane * 8u) = (hw_float2){m_run, l_run};
      akv_lds_barrier();
      hw_float2 ml[HW_W];
#pragma unroll
      for (int i = 0; i < HW_W; ++i) ml[i] = *(hw_lds_f64*)(uintptr_t)(HW_ML + (uint32_t)(min(i, shares - 1) * hp + hs) * 32u + (uint32_t)(col & 3) * 8u);
#pragma unroll
      for (int i = 0; i < HW_W; ++i) M = fmaxf(M, ml[i].x);
      L = 0.f;
#pragma unroll
      for (int i = 0; i < HW_W; ++i) {
        const float part = ml[i].x > -INFINITY ? __builtin_amdgcn_exp2f(ml[i].x - M) * ml[i].y : ml[i].y;   // (-inf: no token, or sums that are NaN)
        L += i < shares ? part : 0.f;
      }
      wgt = m_run > -INFINITY ? __builtin_amdgcn_exp2f(m_run - M) : 1.f;
    }
    if (active && r < shares) {
      int row = 4 * g;
      asm volatile("" : "+v"(row));      // (the places would be computed ahead of all segments, a register each)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v[NT];
        F::finish(a.lut, o, i, v);
#pragma unroll
        for (int n = 0; n < NT; ++n) v[n] *= wgt;
        if (col < nq) F::places(row + i, [&](int at, int n) __attribute__((always_inline)) { *(hw_lds_f32*)(uintptr_t)(buf + (uint32_t)(col * 256 + at) * 4u) = v[n]; });
      }
    }
    if (shares > 1) akv_lds_barrier();
    else akv_wave_sync();
    if (active) {
      const int step = shares > 1 ? R * 64 : 64;
      for (int idx = (shares > 1 || r == 0) ? r * 64 + lane : 256; idx < 64 * nq; idx += step) {
        hw_float4 sum = {0.f, 0.f, 0.f, 0.f};
        for (int rr = 0; rr < shares; ++rr) sum += *(hw_lds_f128*)(uintptr_t)((uint32_t)(rr * hp + hs) * HW_BUF + (uint32_t)idx * 16u);
        *(float4*)(a.part_acc + slot * 256 + 4 * (size_t)idx) = make_float4(sum[0], sum[1], sum[2], sum[3]);
      }
      if (r == 0 && lane < nq) {
        a.part_ml[(slot + lane) * 2] = M * 0.6931471805599453f;     // back to the natural-log domain
        a.part_ml[(slot + lane) * 2 + 1] = L;
      }
    }
    // (the next segment's rows land in these buffers)
    if (shares > 1) akv_lds_barrier();
    else akv_wave_sync();
  }
}

// ----------------------------------------------------------------------------------
// tables, built by a workgroup of 256 threads
// ----------------------------------------------------------------------------------
// byte `byte_of` of four levels, table[0..3], a word: of their integers in units of `unit` (three digits, top first), or of the
// float16 form of alpha times a level (low byte first), rounding or remainder
__device__ __forceinline__ uint32_t hw_key_bytes(const float* table, float unit, int byte_of) {
  uint32_t word = 0;
  for (int v = 0; v < 4; ++v) {
    const int n = (int)rintf(table[v] / unit), d0 = ((n + 128) & 255) - 128, n1 = (n - d0) >> 8, d1 = ((n1 + 128) & 255) - 128;
    word |= ((uint32_t)(byte_of == 2 ? d0 : byte_of == 1 ? d1 : (n1 - d1) >> 8) & 255u) << (8 * v);
  }
  return word;
}
__device__ __forceinline__ uint32_t hw_value_bytes(const float* table, float alpha, bool remainder, int byte_of) {
  uint32_t word = 0;
  for (int v = 0; v < 4; ++v) {
    const float x = alpha * table[v];
    const __half hi = __float2half_rn(x);
    const uint32_t bits = __half_as_ushort(remainder ? __float2half_rn(x - __half2float(hi)) : hi);
    word |= (byte_of == 0 ? bits & 255u : bits >> 8) << (8 * v);
  }
  return word;
}
// largest magnitude of n levels, and the power of two that brings it to [2^9, 2^10)
__device__ __forceinline__ float hw_top(const float* table, int n) {
  float top = 0.f;
  for (int v = 0; v < n; ++v) top = fmaxf(top, fabsf(table[v]));
  return top;
}
__device__ __forceinline__ float hw_base(float top) {
  return top > 0.f ? __uint_as_float((min(max(254u + 9u - ((__float_as_uint(top) >> 23) & 0xffu), 1u), 253u)) << 23) : 1.f;
}

// Factor of N value levels whose float16 forms are used without remainders: a free factor makes them nearly exact.  Of HW_SEARCH
// candidates within a factor of two, a quarter here for each wavefront of the workgroup, the one with the smallest largest error
// relative to each level, and that error.  Four candidates a lane side by side; levels beyond the fourth only where one of the
// wavefront's 256 still is better than its best so far.  (The first call with a new workspace waits for this: 34 us more
// than a later one.  658 with a division a level, one candidate at a time, and units of two sets of key levels searched for
// too; 187 on the kernel before this one.)
template <int N> __device__ __forceinline__ float hw_search(const float* table, float base, float& factor) {
  float c[N], rel[N];
#pragma unroll
  for (int v = 0; v < N; ++v) {
    c[v] = table[v] * base;
    rel[v] = c[v] != 0.f ? 1.f / fabsf(c[v]) : 0.f;
  }
  float least = INFINITY, mine = INFINITY, at = 1.f;      // of the wavefront, of the lane and where
#pragma unroll 1
  for (int k = 0; k < HW_SEARCH / 256; k += 4) {
    float al[4], worst[4] = {0.f, 0.f, 0.f, 0.f};         // (errors times al)
#pragma unroll
    for (int i = 0; i < 4; ++i) al[i] = 1.f + (float)((int)threadIdx.x * (HW_SEARCH / 256) + k + i) * (1.f / HW_SEARCH);
    auto levels = [&](int v0, int v1) __attribute__((always_inline)) {
#pragma unroll
      for (int v = v0; v < v1; ++v)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float x = c[v] * al[i];
          worst[i] = fmaxf(worst[i], fabsf(__half2float(__float2half_rn(x)) - x) * rel[v]);
        }
    };
    auto better = [&]() __attribute__((always_inline)) {
      bool any = false;
#pragma unroll
      for (int i = 0; i < 4; ++i) any = any || worst[i] < least * al[i];
      return __builtin_amdgcn_ballot_w64(any) != 0;
    };
    levels(0, 4);
    if (!better()) continue;
    if constexpr (N > 4) {
      levels(4, N);
      if (!better()) continue;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (worst[i] < mine * al[i]) { mine = worst[i] / al[i]; at = al[i]; }
    least = -akv_wave_max(-mine);
  }
  const uint64_t who = __builtin_amdgcn_ballot_w64(mine == least);
  factor = who ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(at), __builtin_ctzll(who))) : 1.f;
  return least;
}

template <bool P> __device__ void hw35<P>::tables(const float* table, uint32_t* lut) {
  __shared__ float err[2][4], at[2][4];
  __shared__ float unit[2], alpha[2];
  const int tid = threadIdx.x;
  const float *c0 = table + HYB_CEN0, *c1 = c0 + 8;
  const float top[2] = {hw_top(c0, 8), hw_top(c1, 4)};
  // alpha of float16(alpha c): the largest alpha c lies in [2^9, 2^11), so that no remainder is a subnormal
  if constexpr (!P) {
    float a0, a1;
    const float e0 = hw_search<8>(c0, hw_base(top[0]), a0), e1 = hw_search<4>(c1, hw_base(top[1]), a1);
    if ((tid & 63) == 0) {
      err[0][tid >> 6] = e0;
      at[0][tid >> 6] = a0;
      err[1][tid >> 6] = e1;
      at[1][tid >> 6] = a1;
    }
    __syncthreads();
  }
  if (tid < 2) {
    float al = 1.f, least = INFINITY;
    if constexpr (!P)
      for (int w = 0; w < 4; ++w)
        if (err[tid][w] < least) { least = err[tid][w]; al = at[tid][w]; }
    alpha[tid] = al * hw_base(top[tid]);
    unit[tid] = top[tid] > 0.f ? top[tid] * (1.f / HW_QMAX) : 1.f;
  }
  __syncthreads();
  if (tid < 2) {
    lut[HW_W_UNIT + tid] = __float_as_uint(unit[tid]);
    lut[HW_W_ALPHA + tid] = __float_as_uint(alpha[tid]);
  }
  // thread = a word of the bytes of four levels
  if (tid < HW_W_KA1) lut[tid] = hw_key_bytes(c0 + 4 * (tid & 1), unit[0], tid >> 1);
  else if (tid < HW_W_VA0) lut[tid] = hw_key_bytes(c1, unit[1], tid - HW_W_KA1);
  else if (tid < HW_W_UNIT) {
    const bool remainder = tid >= HW_W_VP0;
    const int i = tid - (remainder ? HW_W_VP0 : HW_W_VA0);
    lut[tid] = i < 4 ? hw_value_bytes(c0 + 4 * (i & 1), alpha[0], remainder, i >> 1) : hw_value_bytes(c1, alpha[1], remainder, i - 4);
  }
}

__device__ void hw25::tables(const float* table, uint32_t* lut) {
  const int tid = threadIdx.x;
  const float* lv = table + H25_CEN0;
  const float top = hw_top(lv, 4), alpha = hw_base(top), unit = top > 0.f ? top * (1.f / HW_QMAX) : 1.f;
  const float c0 = table[H25_CEN1], c1 = table[H25_CEN1 + 1];
  if (tid < 3) lut[HW_W_KA1 + tid] = hw_key_bytes(lv, unit, tid);
  if (tid < 2) lut[HW_W_VA1 + tid] = hw_value_bytes(lv, alpha, false, tid);
  if (tid < 2) lut[HW_W_VP1 + tid] = hw_value_bytes(lv, alpha, true, tid);
  if (tid == 0) {
    lut[HW_W_UNIT + 1] = __float_as_uint(unit);
    lut[HW_W_ALPHA + 1] = __float_as_uint(alpha);
    lut[HW_W_DELTA] = __float_as_uint(0.5f * (c1 - c0));
    lut[HW_W_MIDDLE] = __float_as_uint(0.5f * (c1 + c0));
  }
}

// ----------------------------------------------------------------------------------
// prologue: block 0 cuts the block axis, block 1 builds the tables (only when the codebooks are not the ones they were built
// from), the others take a group of four query heads of a sequence: transform, scale, three signed bytes, operand order
// ----------------------------------------------------------------------------------
template <class F, int QDT>
__global__ __launch_bounds__(256) void akv_attn_hyb_prologue_kernel(
    const void* __restrict__ query, int64_t qs_seq, int64_t qs_head, const float* __restrict__ table, float qscale, int S, int QH,
    int KVH, int hgroup, int gqa, const void* context_lens, int cl_itype, int block_size, int64_t max_blocks_per_seq, int32_t* prefix,
    uint4* __restrict__ qop, float* __restrict__ fac, uint32_t* __restrict__ lut, uint32_t* __restrict__ status, uint32_t start_status,
    int32_t* __restrict__ wgdesc, int32_t* __restrict__ seqw, int G, int shares, int longer) {
  __shared__ int8_t dig[3][4][256];       // [digit][query head][sum]
  __shared__ int32_t scratch[AKV_PART_WORDS];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  if (blockIdx.x == 0) {
    if (tid == 0) status[0] = start_status;
    akv_attn_partition(prefix, S, G, block_size == 32 ? 1 : 2, wgdesc, seqw, scratch, context_lens, cl_itype, block_size, max_blocks_per_seq, shares, longer);
    return;
  }
  if (blockIdx.x == 1) {
    __shared__ int stale;
    if (tid == 0) stale = lut[HW_W_MARK] != F::MARK ? 1 : 0;
    __syncthreads();
    if (tid < F::TAGS && __float_as_uint(table[F::TAG_AT + tid]) != lut[HW_W_TAG + tid]) stale = 1;
    __syncthreads();
    if (!stale) return;
    F::tables(table, lut);
    if (tid < F::TAGS) lut[HW_W_TAG + tid] = __float_as_uint(table[F::TAG_AT + tid]);
    __threadfence();
    __syncthreads();
    if (tid == 0) lut[HW_W_MARK] = F::MARK;
    return;
  }
  const int item = (int)blockIdx.x - 2, s = item / KVH, hv = item % KVH;
  const int q_first = hv / hgroup * gqa + hv % hgroup * 4, nq = min(4, gqa - hv % hgroup * 4);
  if (w < nq) {
    const int64_t off = s * qs_seq + (int64_t)(q_first + w) * qs_head;
    const float q0 = akv_elem<QDT>::load(query, off + F::coord(lane, 0)), q1 = akv_elem<QDT>::load(query, off + F::coord(lane, 1));
    float y[4];
    F::forward(q0, q1, lane, table, y);
    const float top = akv_wave_max(fmaxf(fmaxf(fabsf(y[0]), fabsf(y[1])), fmaxf(fabsf(y[2]), fabsf(y[3]))));
    const float nan = akv_wave_sum((q0 + q1) * 0.f);       // NaN when the query holds one, or an infinity
    // (a head of zeros, or one so small that the scale would overflow: integers of zero)
    const float sc = top > 1e-30f ? HW_QMAX / top : 0.f;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int n = (int)rintf(fminf(fmaxf(y[p] * sc, -HW_QMAX), HW_QMAX));
      const int d0 = ((n + 128) & 255) - 128, n1 = (n - d0) >> 8, d1 = ((n1 + 128) & 255) - 128;
      const int at = F::sum_of(lane, p);
      dig[0][w][at] = (int8_t)((n1 - d1) >> 8);
      dig[1][w][at] = (int8_t)d1;
      dig[2][w][at] = (int8_t)d0;
    }
    if (lane == 0) fac[(size_t)s * QH + q_first + w] = top * (1.f / HW_QMAX) * qscale + nan;
  }
  __syncthreads();
  // thread = (slot w, lane (column 4 d + head, lane group g)): sixteen coordinates of its head's digit d; columns of no digit or
  // head zero
  const int col = lane & 15, g = lane >> 4, d = col >> 2;
  uint32_t v[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    v[r] = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) v[r] |= d < 3 && (col & 3) < nq ? (uint32_t)(uint8_t)dig[d][col & 3][F::faced(w, g, r, b)] << (8 * b) : 0u;
  }
  qop[((size_t)item * 4 + w) * 64 + lane] = make_uint4(v[0], v[1], v[2], v[3]);
}

// ----------------------------------------------------------------------------------
// reduce: a wavefront per query head of a sequence merges the partial results and transforms them back
// ----------------------------------------------------------------------------------
template <class F, int ODT>
__global__ __launch_bounds__(256) void akv_attn_hyb_reduce_kernel(const float* __restrict__ part_acc, const float* __restrict__ part_ml,
                                                                  const float* __restrict__ table, int S, int QH, void* __restrict__ out,
                                                                  int64_t os_seq, int64_t os_head, const uint32_t* __restrict__ status,
                                                                  const int32_t* __restrict__ seqw) {
  const int lane = threadIdx.x & 63;
  const int item = __builtin_amdgcn_readfirstlane((int)blockIdx.x * 4 + (int)(threadIdx.x >> 6));
  if (item >= S * QH) return;
  const int s = item / QH, h = item % QH;
  const int w_lo = seqw[2 * s], w_hi = seqw[2 * s + 1];
  const int64_t obase = s * os_seq + h * os_head;
  // (a call marked as failed says so in every output)
  const float poison = status[0] != 0u ? __uint_as_float(0x7fc00000u) : 0.f;
  int at[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) at[i] = F::sum_of(lane, i);
  // the first PF partial sums are requested before their weights are known
  constexpr int PF = 8;
  float pre[PF][4];
#pragma unroll
  for (int u = 0; u < PF; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i) pre[u][i] = w_lo + u <= w_hi ? part_acc[((size_t)(w_lo + u + s) * QH + h) * 256 + at[i]] : 0.f;
  float M = -INFINITY;
  for (int w = w_lo + lane; w <= w_hi; w += 64) M = fmaxf(M, part_ml[((size_t)(w + s) * QH + h) * 2]);
  M = akv_wave_max(M);
  float l = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int w0 = w_lo; w0 <= w_hi; w0 += 64) {
    float wgt = 0.f;
    if (w0 + lane <= w_hi) {
      const float2 ml = *(const float2*)(part_ml + ((size_t)(w0 + lane + s) * QH + h) * 2);
      // (-inf: no token, or sums that are NaN)
      wgt = ml.x > -INFINITY ? __expf(ml.x - M) : 0.f;
      l += ml.x > -INFINITY ? wgt * ml.y : ml.y;
    }
    const int n = min(64, w_hi - w0 + 1);
    for (int u0 = 0; u0 < n; u0 += PF) {
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        const float wu = u0 + u < n ? __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(wgt), u0 + u)) : 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = fmaf(wu, pre[u][i], acc[i]);
      }
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        const int w = w0 + u0 + PF + u;
#pragma unroll
        for (int i = 0; i < 4; ++i) pre[u][i] = w <= w_hi ? part_acc[((size_t)(w + s) * QH + h) * 256 + at[i]] : 0.f;
      }
    }
  }
  l = akv_wave_sum(l);
  const float inv = l > 0.f ? 1.f / l : l == 0.f ? 1.f : l;       // (NaN stays)
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] *= inv;
  float o0, o1;
  F::back(acc, lane, table, o0, o1);
  akv_elem<ODT>::store(out, obase + F::coord(lane, 0), o0 + poison);
  akv_elem<ODT>::store(out, obase + F::coord(lane, 1), o1 + poison);
}

// ----------------------------------------------------------------------------------
// host side
// ----------------------------------------------------------------------------------
bool akv_attn_mfma_disabled();

// akv_debug_set_handoff_spin_limit: 0 marks calls as failed, so that callers can see what a failed call looks like.  (No kernel has
// a wait that could give up.)
static int g_spin_limit = -1;
extern "C" int akv_debug_set_handoff_spin_limit(int polls) {
  g_spin_limit = polls;
  return AKV_OK;
}

// (a group may hold a single query head)
size_t akv_attn_hyb_extra_bytes(int S, int QH) { return akv_align256((size_t)S * QH * 4 * 64 * 16); }

// rows are dword-aligned (the caller checks); blocks of 16 or 32 tokens
bool akv_attn_hyb_applicable(int block_size, const int64_t* strides6) {
  if (akv_attn_mfma_disabled()) return false;
  if (block_size != 16 && block_size != 32) return false;
  for (int i = 0; i < 6; ++i)
    if (strides6[i] < 0 || strides6[i] >= ((int64_t)1 << 27)) return false;
  return true;
}

// ranges the block axis is cut into: three workgroups a CU over all head slots, what the registers of hw35<false> and hw25 admit
// (hw35<true> runs two of them at a time), but no more than akv_attn_grid(), two a CU: the workspace holds records and partial
// results for so many, and calls of up to four groups of query heads get no more.  (The other choices have not been measured.)
static int hw_ranges(int kv_groups, int hp) {
  const int cus = akv_cached_cu_count(), most = akv_attn_grid();
  const int per = (kv_groups + hp - 1) / hp, want = (cus > 0 ? cus : 256) * 3 / per;
  return want < 1 ? 1 : want > most ? most : want;
}

template <class F, int N>
static int hw_launch(const hw_args& a, int grid, hipStream_t stream) {
  AKV_LAUNCH_TIMED((akv_attn_hyb_kernel<F, N>), grid, HW_W * 64, HW_LDS, stream, a);
  AKV_LAUNCH_CHECK("akv_attn_hyb_kernel");
  return AKV_OK;
}

template <class F> struct hw_type { typedef F type; };
// the three kernels of a call; `main` launches the middle one
template <class F, class M>
static int hw_run(const void* query, int q_dtype, int64_t qs_seq, int64_t qs_head, const float* table, float scale, const hw_args& a,
                  const akv_attn_ws& ws, void* out, int out_dtype, int64_t os_seq, int64_t os_head, hipStream_t stream, M main) {
  const int G = hw_ranges(a.KVH, a.hp), shares = HW_W / a.hp, cus = akv_cached_cu_count();
  // (akv_attn_partition: a second segment in chunks; nothing where more workgroups take turns than the chip holds)
  const int longer = G * a.hgroups > F::PER_SIMD * (cus > 0 ? cus : 256) ? 0 : F::PER_SIMD == 3 ? 3 : 2;
  const float qscale = scale * 1.4426950408889634f;      // scores come out in the log2 domain
  const uint32_t start_status = g_spin_limit == 0 ? AKV_STATUS_HANDOFF_TIMEOUT : 0u;
#define HW_PRO(DT) akv_attn_hyb_prologue_kernel<F, DT><<<a.S * a.KVH + 2, 256, 0, stream>>>(query, qs_seq, qs_head, table, qscale, a.S, a.QH, a.KVH, a.hgroup, a.gqa, a.context_lens, a.cl_itype, a.block_size, a.max_blocks_per_seq, ws.prefix, (uint4*)a.qop, ws.qrot, ws.lut, ws.status, start_status, ws.wgdesc, ws.seqw, G, shares, longer)
  if (q_dtype == AKV_F16) HW_PRO(AKV_F16); else if (q_dtype == AKV_BF16) HW_PRO(AKV_BF16); else HW_PRO(AKV_F32);
#undef HW_PRO
  AKV_LAUNCH_CHECK("akv_attn_hyb_prologue_kernel");
  const int rc = main(G * a.hgroups);
  if (rc) return rc;
  const int rgrid = (a.S * a.QH + 3) / 4;
#define HW_RED(DT) akv_attn_hyb_reduce_kernel<F, DT><<<rgrid, 256, 0, stream>>>(a.part_acc, a.part_ml, table, a.S, a.QH, out, os_seq, os_head, ws.status, ws.seqw)
  if (out_dtype == AKV_F16) HW_RED(AKV_F16); else if (out_dtype == AKV_BF16) HW_RED(AKV_BF16); else HW_RED(AKV_F32);
#undef HW_RED
  AKV_LAUNCH_CHECK("akv_attn_hyb_reduce_kernel");
  return AKV_OK;
}

int akv_attn_hyb_run(int format, const void* query, int q_dtype, int64_t qs_seq, int64_t qs_head, const float* table, float scale,
                     const akv_hyb_attn_args& in, const akv_attn_ws& ws, void* extra_ws, void* out, int out_dtype, int64_t os_seq,
                     int64_t os_head, hipStream_t stream) {
  hw_args a;
  a.kc = in.kc; a.kps_blk = in.kps_blk; a.kps_pos = in.kps_pos; a.kps_head = in.kps_head;
  a.vc = in.vc; a.vps_blk = in.vps_blk; a.vps_pos = in.vps_pos; a.vps_head = in.vps_head;
  a.block_tables = in.block_tables; a.bt_itype = in.bt_itype; a.bt_stride = in.bt_stride;
  a.context_lens = in.context_lens; a.cl_itype = in.cl_itype;
  a.S = in.S; a.QH = in.QH; a.gqa = in.QH / in.KVH; a.hgroup = (a.gqa + 3) / 4; a.KVH = in.KVH * a.hgroup; a.block_size = in.block_size;
  a.max_blocks_per_seq = in.max_blocks_per_seq; a.num_blocks = in.num_blocks;
  a.prefix = ws.prefix; a.wgdesc = ws.wgdesc; a.lut = ws.lut; a.qop = (const uint4*)extra_ws; a.fac = ws.qrot;
  a.part_acc = ws.part_acc; a.part_ml = ws.part_ml;
  a.hp = a.KVH >= 3 ? 4 : a.KVH;
  a.hgroups = (a.KVH + a.hp - 1) / a.hp;
  if (format == 25)
    return hw_run<hw25>(query, q_dtype, qs_seq, qs_head, table, scale, a, ws, out, out_dtype, os_seq, os_head, stream,
                        [&](int grid) { return hw_launch<hw25, 4>(a, grid, stream); });
  const uint64_t all = (uint64_t)(uintptr_t)a.kc | (uint64_t)(uintptr_t)a.vc | a.kps_blk | a.kps_pos | a.kps_head | a.vps_blk | a.vps_pos | a.vps_head;
  // groups of four query heads: the accuracy that one float16 a level of values leaves; other counts: float32's, which they always had
  const bool wide = (all & 15) == 0, exact = a.gqa % 4 != 0;
  auto run = [&](auto f) {
    typedef typename decltype(f)::type F;
    return hw_run<F>(query, q_dtype, qs_seq, qs_head, table, scale, a, ws, out, out_dtype, os_seq, os_head, stream,
                     [&](int grid) { return wide ? hw_launch<F, 16>(a, grid, stream) : hw_launch<F, 4>(a, grid, stream); });
  };
  return exact ? run(hw_type<hw35<true>>()) : run(hw_type<hw35<false>>());
}
