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
