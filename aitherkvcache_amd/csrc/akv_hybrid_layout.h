// tq35 rows and tables: what the codec, the vector attention kernel and the matrix-core attention
// kernel share.
//
// Row of one (token, kv head), 64 bytes (aither_kvcache/hybrid_quantizer.py:92-123,771-779):
//   [0,24)  group-0 codes, 3 bits each, MSB-first stream        [24,32) group-0 QJL sign bits (bit 7 first)
//   [32,34) group-0 norm fp16 LE    [34,36) group-0 residual norm fp16 LE
//   [36,52) group-1 codes, 2 bits each                           [52,60) group-1 QJL sign bits
//   [60,62) group-1 norm            [62,64) group-1 residual norm
// Table of floats handed to every entry point: sign vectors of the two structured transforms per
// group, the two codebooks, their decision boundaries.
#pragma once
#include "akv_common.h"

#define HYB_HAD0 0
#define HYB_HAD1 64
#define HYB_QJL0 128
#define HYB_QJL1 192
#define HYB_CEN0 256
#define HYB_CEN1 264
#define HYB_BND0 268
#define HYB_BND1 275

// 64-point Walsh-Hadamard transform across the lanes of a wavefront
template <int H>
__device__ __forceinline__ float hyb_fwht_step(float v, int lane) {
  const float o = akv_lane_xor<H>(v);
  return (lane & H) ? akv_sub_rn(o, v) : akv_add_rn(v, o);
}
__device__ __forceinline__ float hyb_fwht64(float v, int lane) {
  v = hyb_fwht_step<1>(v, lane);
  v = hyb_fwht_step<2>(v, lane);
  v = hyb_fwht_step<4>(v, lane);
  v = hyb_fwht_step<8>(v, lane);
  v = hyb_fwht_step<16>(v, lane);
  v = hyb_fwht_step<32>(v, lane);
  return v;
}

// ---- a lane per vector or group: transforms, sums and bit streams in the lane's registers.
// (The reference rounds every operation: the products come from akv_mul_rn, which the compiler may not fuse into a
// multiply-add.  Where a product that is not exact feeds a tree of sums it also passes through hyb_rounded(), an empty asm
// statement the optimiser cannot see through, so the tree is not reassociated around it either.)
typedef const __attribute__((address_space(4))) float* hyb_uniform;       // a table read at the same place by all lanes: scalar loads
__device__ __forceinline__ float hyb_rounded(float x) {
  asm volatile("" : "+v"(x));
  return x;
}
// N-point Walsh-Hadamard transform of v[0 .. N)
template <int N>
__device__ __forceinline__ void hyb_fwht_regs(float* v) {
#pragma unroll
  for (int h = 1; h < N; h <<= 1)
#pragma unroll
    for (int i = 0; i < N; ++i)
      if ((i & h) == 0) {
        const float lo = v[i], hi = v[i + h];
        v[i] = akv_add_rn(lo, hi);
        v[i + h] = akv_sub_rn(lo, hi);
      }
}
// sum in the order of the reduction over lanes (partners N/2, ..., 1 apart); t is used up
template <int N>
__device__ __forceinline__ float hyb_tree_sum(float* t) {
#pragma unroll
  for (int m = N / 2; m >= 1; m >>= 1)
#pragma unroll
    for (int i = 0; i < m; ++i) t[i] = akv_add_rn(t[i], t[i + m]);
  return t[0];
}
// N coordinates of a row (16-byte aligned) as floats
template <int XDT, int N>
__device__ __forceinline__ void hyb_load_row(const void* x, int64_t off, float* u) {
  if constexpr (XDT == AKV_F32) {
    const float4* p = (const float4*)((const float*)x + off);
#pragma unroll
    for (int i = 0; i < N / 4; ++i) { const float4 q = p[i]; u[4 * i] = q.x; u[4 * i + 1] = q.y; u[4 * i + 2] = q.z; u[4 * i + 3] = q.w; }
  } else {
    const uint4* p = (const uint4*)((const unsigned short*)x + off);
#pragma unroll
    for (int i = 0; i < N / 8; ++i) {
      const uint4 q = p[i];
      const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (XDT == AKV_F16) {
          u[8 * i + 2 * j] = __half2float(__ushort_as_half((unsigned short)(w[j] & 0xffffu)));
          u[8 * i + 2 * j + 1] = __half2float(__ushort_as_half((unsigned short)(w[j] >> 16)));
        } else {
          u[8 * i + 2 * j] = __uint_as_float(w[j] << 16);
          u[8 * i + 2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
        }
      }
    }
  }
}
// the signs of v[0 .. 32) (a bit set where v scale >= 0), first value in the top bit: both halves of the word side by side, so that
// two wait states lie between a compare and its use (akv_append_codes)
__device__ __forceinline__ uint32_t hyb_sign_word(const float* v, float scale) {
  uint32_t a = 0u, b = 0u;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    uint64_t m;
    asm("v_cmp_le_f32 vcc, 0, %[ya]\n\t"
        "v_cmp_le_f32 %[m], 0, %[yb]\n\t"
        "s_nop 0\n\t"
        "v_addc_co_u32 %[wa], vcc, %[wa], %[wa], vcc\n\t"
        "v_addc_co_u32 %[wb], %[m], %[wb], %[wb], %[m]"
        : [wa] "+v"(a), [wb] "+v"(b), [m] "=&s"(m)
        : [ya] "v"(akv_mul_rn(v[i], scale)), [yb] "v"(akv_mul_rn(v[16 + i], scale))
        : "vcc");
  }
  return (a << 16) | b;
}

// 32 values of every lane's row to memory: through LDS (64 rows of 36 floats, a wavefront's own), so that eight lanes write 128
// bytes of a row at a time.  out: the first row's 32 values, 16-byte aligned; rows from `rows` on are not stored.
#define HYB_TURN_FLOATS (64 * 36)
__device__ __forceinline__ void hyb_store_turned(const float* v, float* turn, float* out, int64_t os, int rows, int lane) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int i = 0; i < 8; ++i) *(float4*)&turn[36 * lane + 4 * i] = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int r = 8 * i + (lane >> 3), c = 4 * (lane & 7);
    const float4 q = *(const float4*)&turn[36 * r + c];
    if (r < rows) *(float4*)(out + (int64_t)r * os + c) = q;
  }
}

// ---- tq25 (the row: akv_hybrid25.hip): tables, transforms
#define H25_HAD 0          // [128] Hadamard signs in coordinate order (group 0's 32, then group 1's 96)
#define H25_QJL 128        // [128] QJL signs likewise
#define H25_CEN0 256       // 4 centroids
#define H25_CEN1 260       // 2 centroids
#define H25_BND0 262       // 3 boundaries
#define H25_BND1 265       // 1 boundary
#define H25_ROW 44

// float32 values of sqrt(32), sqrt(96) and of sqrt(pi/2) / dim (hybrid_quantizer.py:232,540-541)
constexpr float kH25Root0 = 5.656854249492381f;
constexpr float kH25Root1 = 9.797958971132712f;
constexpr float kH25Kappa0 = (float)(1.2533141373155001 / 32.0);
constexpr float kH25Kappa1 = (float)(1.2533141373155001 / 96.0);
// 32-point Walsh-Hadamard transform inside each half of the wavefront
__device__ __forceinline__ float h25_fwht32(float v, int lane) {
  v = hyb_fwht_step<1>(v, lane);
  v = hyb_fwht_step<2>(v, lane);
  v = hyb_fwht_step<4>(v, lane);
  v = hyb_fwht_step<8>(v, lane);
  v = hyb_fwht_step<16>(v, lane);
  return v;
}
// the lane's two coordinates
struct h25_roles {
  int ca, cb;       // coordinate of the first value (group 1, 64-point block) and of the second
  bool b0;          // the second value belongs to group 0
  int ja, jb;       // position inside the group's code / sign streams
  __device__ __forceinline__ explicit h25_roles(int lane)
      : ca(32 + lane), cb(lane < 32 ? lane : 64 + lane), b0(lane < 32), ja(lane), jb(lane < 32 ? lane : 32 + lane) {}
};

// the lane forms of the codecs: rows they can read and write wide, and calls that are large enough (`large`) unless an
// environment variable asks for one of the forms
static inline bool hyb_lane_aligned(const void* x, const void* x2, int64_t xs0, int64_t xs1, int dt, const void* out, const void* out2,
                                    int64_t out_strides, int out_align) {
  const int64_t xal = dt == AKV_F32 ? 3 : 7;      // elements per 16 bytes, minus one
  return (((uintptr_t)x | (uintptr_t)x2) & 15) == 0 && ((xs0 | xs1) & xal) == 0 &&
         (((uintptr_t)out | (uintptr_t)out2 | (uintptr_t)out_strides) & (uintptr_t)(out_align - 1)) == 0;
}
static inline bool hyb_lane_form(bool large) {
  static const bool never = [] { const char* e = getenv("AKV_HYBRID_WAVE_ENCODE"); return e && e[0] == '1'; }();
  const char* e = getenv("AKV_HYBRID_LANE_ENCODE");        // (read per call: tests switch it)
  return !never && (large || (e && e[0] == '1'));
}

// matrix-core attention on hybrid rows (akv_attn_hyb.hip)
struct akv_attn_ws;
struct akv_hyb_attn_args {
  const uint8_t* kc; int64_t kps_blk, kps_pos, kps_head;
  const uint8_t* vc; int64_t vps_blk, vps_pos, vps_head;
  const void* block_tables; int bt_itype; int64_t bt_stride;
  const void* context_lens; int cl_itype;
  int S, QH, KVH, block_size;
  int64_t max_blocks_per_seq;
  int64_t num_blocks;          // physical blocks in the cache; table entries are clamped into [0, num_blocks)
};
size_t akv_attn_hyb_extra_bytes(int S, int QH);
bool akv_attn_hyb_applicable(int block_size, const int64_t* strides6);
// format: 35 or 25
int akv_attn_hyb_run(int format, const void* query, int q_dtype, int64_t qs_seq, int64_t qs_head, const float* table, float scale,
                     const akv_hyb_attn_args& in, const akv_attn_ws& ws, void* extra_ws, void* out, int out_dtype, int64_t os_seq,
                     int64_t os_head, hipStream_t stream);
