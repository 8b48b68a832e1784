// Rotation matrices as register-resident operands of v_mfma_f32_32x32x16_f16.
//
// The codec and the attention kernels multiply a few rows by Pi or Pi^T.  They do it transposed,
//
//   Y^T[coordinate, row] = sum_k M[coordinate, k] * X^T[k, row],
//
// with the MATRIX as the A operand and the rows as the columns of B: a wavefront keeps one or more tiles of 32 output
// coordinates of M in registers for its whole life (stationary: nothing of the matrix passes through LDS), and lane l
// ends up with SIXTEEN NEIGHBOURING coordinates of ONE row (row l % 32, coordinates 16 (l / 32) + 0..15 of the tile) --
// so a row's codes are packed, or its outputs converted and stored, inside a lane.
//
// The matrix is split into two float16 terms (hi + lo, scaled by 64 to stay clear of float16 subnormals: ~22 bits).
// A table holds the fragments in the order in which the lanes load them: [hi | lo][tile][k-step][lane] x 16 bytes,
// lane l of a fragment = elements 16 ks + 8 (l / 32) + 0..7 of matrix row akv_frag_coord(l % 32) of the tile.
#pragma once
#include "akv_common.h"

typedef _Float16 akv_h8 __attribute__((ext_vector_type(8)));
typedef float akv_f16v __attribute__((ext_vector_type(16)));
#define AKV_FRAG_SCALE 64.f

// head sizes the fragment tables exist for (512 would need 256 registers a tile)
static inline bool akv_frag_dim(int d) { return d == 64 || d == 128 || d == 256; }
static inline size_t akv_frag_table_bytes(int d) { return (size_t)d * d * 4; }
// bytes of the prepared-rotation buffer: float matrices and the 16x16 operand tables, then a flag word (1: a row of the
// matrix is so long that a rotated unit vector may leave the range of the cell table), then the fragments of Pi
// and of Pi^T
static inline size_t akv_frag_flag_offset(int d) { return akv_prep_floats(d) * sizeof(float); }
static inline size_t akv_frag_fwd_offset(int d) { return akv_frag_flag_offset(d) + 256; }
static inline size_t akv_frag_inv_offset(int d) { return akv_frag_fwd_offset(d) + akv_frag_table_bytes(d); }
static inline size_t akv_prep_bytes(int d) {
  return akv_frag_dim(d) ? akv_frag_inv_offset(d) + akv_frag_table_bytes(d) : akv_prep_floats(d) * sizeof(float);
}

// coordinate (0..31 inside the tile) that matrix-operand row r stands for: accumulator register v of a lane in half h
// is row 8 (v / 4) + 4 h + v % 4, and is to be coordinate 16 h + v
__host__ __device__ constexpr int akv_frag_coord(int r) { return 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3); }

__device__ __forceinline__ akv_h8 akv_as_h8(uint4 u) {
  union { uint4 u; akv_h8 h; } cv;
  cv.u = u;
  return cv.h;
}
__device__ __forceinline__ akv_f16v akv_zero16() {
  return (akv_f16v){0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
}

// Cell table of the codebook search: code = #{b < y}.  AKV_CELLS uniform cells over y in (-1.004, 1.004) map cell ->
// (number of boundaries in lower cells, the one boundary inside the cell or +inf); the cell index is a monotone function
// of y evaluated by the same instructions for y and, when the table is built, for the boundaries, so
// base + (boundary < y) is exact for every float in range.
#define AKV_CELLS 512
#define AKV_CELL_S 2040.f                       // 8 x cells per unit of y: the table is addressed in bytes
#define AKV_CELL_C (8388608.f + 2048.f)         // 2^23 + centre: the sum's mantissa is 8 x the cell coordinate
#define AKV_CELL_MASK 0xff8u
#define AKV_MAX_ROW_NORM 1.0015f                // |y| <= |row of Pi| <= this keeps y inside the table
__device__ __forceinline__ uint32_t akv_cell(float y) {
  return __float_as_uint(fmaf(y, AKV_CELL_S, AKV_CELL_C)) & AKV_CELL_MASK;
}
