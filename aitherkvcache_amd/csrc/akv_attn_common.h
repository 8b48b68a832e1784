// Work partition shared by the paged decode-attention kernels.
//
// The (sequence, KV block) pairs of a batch are laid end to end into one global block axis
// of length total = sum_i ceil(ctx_i / block_size).  The main kernel runs a fixed grid of G
// workgroups; workgroup w owns global blocks [w*per, (w+1)*per) with per = ceil(total / G),
// for ALL kv heads, and walks the sequences that range intersects.  Every (workgroup,
// sequence) intersection produces one partial (running max, running sum, unnormalised
// accumulator) per query head, stored in slot w + seq -- unique because both w and seq are
// non-decreasing along the walk and at least one of them grows at every step.  A reduce
// kernel merges the slots of a sequence with the log-sum-exp rule
// (aither_kvcache/fused_attention.py:513-522) and applies the inverse rotation.
// Everything is derived on the device from context_lens, so the launch needs no host
// synchronisation and the sequence can be recorded into a HIP graph.
#pragma once
#include "akv_common.h"

#define AKV_ATTN_WG_PER_CU 2

struct akv_attn_args {
  const uint8_t* kp; int64_t kps_blk, kps_pos, kps_head;
  const float* kn;   int64_t kns_blk, kns_pos, kns_head;
  const uint8_t* vp; int64_t vps_blk, vps_pos, vps_head;
  const float* vn;   int64_t vns_blk, vns_pos, vns_head;
  const void* block_tables; int bt_itype; int64_t bt_stride;
  const void* context_lens; int cl_itype;
  const float* centroids;
  int S, QH, KVH, block_size;
  int64_t max_blocks_per_seq;
  int64_t num_blocks;      // physical blocks in the cache; table entries are clamped into [0, num_blocks)
  float scale;
  const int32_t* prefix;
  const float* qrot;
  float* part_acc;
  float* part_ml;
  // matrix-core kernel only: a kv head with more than eight query heads is presented as `hgroup`
  // heads of QH / (KVH * hgroup) query heads each that read the same rows (KVH then counts those)
  int hgroup;
};

static inline int akv_attn_grid() {
  int cus = akv_cached_cu_count();
  return (cus > 0 ? cus : 256) * AKV_ATTN_WG_PER_CU;
}

static inline size_t akv_align256(size_t v) { return (v + 255) & ~(size_t)255; }

// Workspace carve-up.  acc_floats = floats of accumulator per query head
// (head_dim for the uniform codec, 256 for tq35).  The workspace starts with a header whose place
// does not depend on the batch: the cached lookup tables of the matrix-core kernels (their
// validity tag would otherwise outlive a call at another batch size that overwrote the words it
// vouches for) and the status words of the most recent call.
#define AKV_WS_LUT_BYTES 4096
#define AKV_WS_STATUS_BYTES 256
#define AKV_WS_HEADER_BYTES (AKV_WS_LUT_BYTES + AKV_WS_STATUS_BYTES)
// status word 0: nonzero when the most recent call failed (cleared by the prologue, turned into NaN outputs by the reduce).  No
// kernel has a wait that could give up; the prologue of hybrid calls sets it when akv_debug_set_handoff_spin_limit(0) says so.
#define AKV_STATUS_HANDOFF_TIMEOUT 1u
// record of a workgroup (int32 words): its range [g0, g1) of the global block axis; then its first segment: the
// sequence (-1: the range is empty), the sequence's first and one-past-last global block, its context length in
// tokens (clamped to the table width)
#define AKV_WGREC 8
#define AKV_WGREC_G0 0
#define AKV_WGREC_G1 1
#define AKV_WGREC_SEQ 2
#define AKV_WGREC_SB0 3
#define AKV_WGREC_SB1 4
#define AKV_WGREC_CTX 5
struct akv_attn_ws {
  uint32_t* lut;     // AKV_WS_LUT_BYTES of cached tables (matrix-core kernels)
  uint32_t* status;  // AKV_WS_STATUS_BYTES
  int32_t* wgdesc;   // [G][AKV_WGREC] record of every workgroup of the matrix-core kernel: its range of the global
                     // block axis and what its first segment starts from (written by that kernel's prologue; see
                     // akv_attn_partition)
  int32_t* seqw;     // [S][2] first and last workgroup whose range meets the sequence (same prologue)
  int32_t* prefix;   // [S + 1] exclusive prefix of blocks per sequence; prefix[S] = total
  float* qrot;       // [S][QH][acc_floats] transformed queries
  float* part_acc;   // [G + S][QH][acc_floats]
  float* part_ml;    // [G + S][QH][2]  (max, sum)
  size_t bytes;
};

static inline akv_attn_ws akv_attn_ws_layout(void* base, int S, int QH, int acc_floats, int G) {
  akv_attn_ws w;
  w.lut = (uint32_t*)base;
  w.status = (uint32_t*)((char*)base + AKV_WS_LUT_BYTES);
  size_t off = AKV_WS_HEADER_BYTES;
  w.wgdesc = (int32_t*)((char*)base + off);
  off += akv_align256((size_t)G * AKV_WGREC * 4);
  w.seqw = (int32_t*)((char*)base + off);
  off += akv_align256((size_t)(S > 0 ? S : 1) * 2 * 4);
  w.prefix = (int32_t*)((char*)base + off);
  off += akv_align256((size_t)(S + 1) * 4);
  w.qrot = (float*)((char*)base + off);
  off += akv_align256((size_t)S * QH * acc_floats * 4);
  w.part_acc = (float*)((char*)base + off);
  off += akv_align256((size_t)(G + S) * QH * acc_floats * 4);
  w.part_ml = (float*)((char*)base + off);
  off += akv_align256((size_t)(G + S) * QH * 2 * 4);
  w.bytes = off;
  return w;
}

// blocks a sequence occupies, clamped to the table width
__device__ __forceinline__ int akv_seq_blocks(const void* context_lens, int cl_itype, int s,
                                              int block_size, int64_t max_blocks_per_seq) {
  int64_t ctx = akv_load_index(context_lens, cl_itype, s);
  if (ctx < 0) ctx = 0;
  int64_t nb = (ctx + block_size - 1) / block_size;
  if (nb > max_blocks_per_seq) nb = max_blocks_per_seq;
  return (int)nb;
}

// physical block id of a table entry, clamped into the cache (a corrupt entry then reads a wrong
// block instead of memory outside the cache)
__device__ __forceinline__ int64_t akv_clamp_block(int64_t id, int64_t num_blocks) {
  return id < 0 ? 0 : (id >= num_blocks ? num_blocks - 1 : id);
}

__device__ __forceinline__ int64_t akv_seq_tokens(const void* context_lens, int cl_itype, int s,
                                                  int block_size, int64_t max_blocks_per_seq) {
  int64_t ctx = akv_load_index(context_lens, cl_itype, s);
  if (ctx < 0) ctx = 0;
  const int64_t cap = max_blocks_per_seq * block_size;
  return ctx < cap ? ctx : cap;
}

// One workgroup (256 threads or more: those past 255 hold nothing) writes prefix[0..S].  Returns the entry of the thread's first
// sequence, min(S, tid * ceil(S / 256)), and in `end` that of the next thread's.
__device__ __forceinline__ int akv_block_prefix_scan(const void* context_lens, int cl_itype, int S,
                                                     int block_size, int64_t max_blocks_per_seq,
                                                     int32_t* prefix, int32_t* scratch /*[>= 4] LDS*/, int* end = nullptr) {
  const int tid = threadIdx.x;
  const int chunk = (S + 255) / 256;
  const int lo = min(S, tid * chunk), hi = min(S, lo + chunk);
  int sum = 0;
  for (int s = lo; s < hi; ++s) sum += akv_seq_blocks(context_lens, cl_itype, s, block_size, max_blocks_per_seq);
  // exclusive scan over the 256 threads: inclusive scan inside each wavefront by lane shifts, then
  // the four wavefront totals through LDS
  const int lane = tid & 63, wave = tid >> 6;
  const int inc = akv_wave_inclusive_scan(sum);
  if (lane == 63) scratch[wave] = inc;
  __syncthreads();
  int base = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const int t = scratch[w];
    if (w < wave) base += t;
  }
  int run = base + inc - sum;
  for (int s = lo; s < hi; ++s) {
    prefix[s] = run;
    run += akv_seq_blocks(context_lens, cl_itype, s, block_size, max_blocks_per_seq);
  }
  if (tid == 255) prefix[S] = base + inc;
  if (end) *end = base + inc;
  return base + inc - sum;
}

// longest range of whole workgroups against an equal cut, in chunks (akv_attn_partition)
__device__ __forceinline__ bool akv_attn_aligned_pays(int aligned, int equal, int shares, int longer) {
  return shares > 1 ? (aligned + shares - 1) / shares <= (equal + shares - 1) / shares + 1 : aligned <= equal + max(longer, equal <= 8 ? 1 : 0);
}

// the last i < n (a power of two) with entry[i] <= v, for two v side by side: entries non-decreasing, entry[0] <= v
__device__ __forceinline__ void akv_last_at_most(const int32_t* entry, int n, int v0, int v1, int& i0, int& i1) {
  i0 = i1 = 0;
  for (int step = n >> 1; step > 0; step >>= 1) {
    const int e0 = entry[i0 + step], e1 = entry[i1 + step];
    i0 += e0 <= v0 ? step : 0;
    i1 += e1 <= v1 ? step : 0;
  }
}

// ----------------------------------------------------------------------------------
// Block prefix of the batch and partition of the global block axis among the G workgroups of the matrix-core
// kernel, written by one workgroup of 256 threads or more.
//
// A workgroup whose range crosses a sequence boundary starts twice (query operand, block ids, first rows, a
// partial chunk at both ends): measured, such workgroups finish 5 us after the others and ARE the tail of
// the launch.  So sequences get whole workgroups where that pays: the smallest lambda (chunks per workgroup) with
// sum_s ceil(c_s / lambda) <= G is found by bisection (the sum is non-increasing in lambda), sequence s takes
// k_s = ceil(c_s / lambda) consecutive workgroups and splits its c_s chunks evenly among them; left-over workgroups get an
// empty range.  Otherwise the axis is cut into G equal ranges.  Either way workgroups and sequences both advance
// monotonically along the axis, so slot = workgroup + sequence stays unique, and seqw[s] = (first, last
// workgroup that meets sequence s), which the reduce kernel reads instead of dividing by the range length.
// `cb` = blocks per chunk of the main kernel (2 for blocks of 16 tokens, 1 for blocks of 32).  `shares` > 1: so many wavefronts
// of a workgroup go through its chunks side by side and merge their results at the end of every segment.
//
// Whole workgroups: with at most 64 sequences always where the non-empty ones are at most G / 8.  A second segment costs a
// workgroup as much as some chunks or one more round of chunks of its shares, so also with up to 256 sequences, the non-empty
// ones at most half the workgroups, while the longest range is no more than that longer than an equal one (`longer`, from eight
// chunks down at least one).  One
// kv head, 48 sequences: of 700 tokens 21.3 -> 17.7 us, of 1k to 16k the step 41.2 -> 36.6.  Eight kv heads: the step of 40
// sequences of 300 to 3,000 39.3 -> 35.0 us, of 64 of 100 to 1,500 40.6 -> 33.7, of 100 of 200 to 1,000 42.0 -> 37.6, of 128 of 300 33.1, 41.9 before;
// heads of 256 55.5 -> 49.5, tq35 65.2 -> 56.1.
// Attention of batches of G / 8 to G / 2 sequences of 250 to 6,000 tokens, equal ranges over whole workgroups, by what these are longer:
//   kernel of akv_attn_mfma.hip        none 1.00 to 1.33, 1 chunk 1.04 to 1.33, 2 1.04 to 1.15, 3 1.03 to 1.06, 12 0.95 to 0.99
//   independent wavefronts, one share  none 0.97 to 1.35, 1 1.00 to 1.26, 2 0.99 to 1.15; 3 heads of 256 0.98 to 1.03, hybrid rows 0.98
//     to 1.12 (64 contexts of 4,000 to 8,192 1.01), but heads of 64 0.98 to 1.00, and tq35 with two workgroups a CU 0.96 to 1.01; 4 0.97 to 1.06
//   as many workgroups as half again the chip holds (tq35, groups of other than four heads, from three groups or heads on): the ranges of a CU
//     take turns, a second segment hides behind another's products and a longer range does not: none 0.97 to 1.58, 1 chunk up to
//     ranges of eight 1.00 to 1.17, beyond 0.91 to 1.02, 2 0.90 to 1.03, 3 0.91 to 0.99
//
// At most 64 sequences are held by one wavefront, more by a thread each (or several each); records are written by a thread per
// workgroup, which finds its sequence among the starts in LDS.  (By a thread per sequence, one of 30,000 tokens among 99 of
// 200 had 150 records to write alone: the kernel 10.9 us, now 6.3.)
// ----------------------------------------------------------------------------------
#define AKV_PART_WORDS 784              // LDS of akv_attn_partition (int32 words)
__device__ __forceinline__ void akv_attn_partition(int32_t* prefix, int S, int G, int cb, int32_t* wgdesc, int32_t* seqw,
                                                   int32_t* lds /*[AKV_PART_WORDS]*/, const void* context_lens, int cl_itype,
                                                   int block_size, int64_t max_blocks_per_seq, int shares, int longer) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int n = S > 64 ? 256 : 64;      // starts in LDS: of every sequence, beyond 256 of every `chunk`-th
  const int chunk = (S + 255) / 256;
  int32_t* p_wfirst = lds;              // [n + 1] first workgroup of each sequence; [n] = workgroups in use
  int32_t* p_pref = lds + 257;          // [n + 1] block prefix; [n] = total
  int32_t* p_ctx = lds + 514;           // [256] context length in tokens, clamped to the table width (at most 256 sequences)
  int32_t* p_mode = lds + 770;          // [0] 1 = whole workgroups per sequence (at most 64 sequences)
  int32_t* p_part = lds + 771;          // [2][4] sums of the wavefronts (more)
  int32_t* p_scan = lds + 779;          // [4]
  bool aligned = false;
  if (S > 64) {
    if (S <= 256 && tid < S) p_ctx[tid] = (int)akv_seq_tokens(context_lens, cl_itype, tid, block_size, max_blocks_per_seq);
    int b1;
    const int b0 = akv_block_prefix_scan(context_lens, cl_itype, S, block_size, max_blocks_per_seq, prefix, p_scan, &b1);
    if (tid < 256) p_pref[tid] = b0;
    if (tid == 255) p_pref[256] = b1;
    __threadfence_block();
    __syncthreads();                    // the prefix written by this workgroup is readable by all of it
    if (S <= 256) {
      const int c = (b1 - b0 + cb - 1) / cb;                     // chunks of the thread's sequence (0: none, or an empty one)
      int turn = 0;
      auto sum_all = [&](int v) {
        const int mine = akv_wave_sum(v);
        if (lane == 0 && tid < 256) p_part[4 * turn + (tid >> 6)] = mine;
        __syncthreads();
        const int all = p_part[4 * turn] + p_part[4 * turn + 1] + p_part[4 * turn + 2] + p_part[4 * turn + 3];
        turn ^= 1;                        // (the other half is written next: nobody reads that one any more)
        return all;
      };
      const int sumc = sum_all(c), nz = sum_all(c > 0 ? 1 : 0);
      const int equal = max(1, (sumc + G - 1) / G);
      int lo = equal;
      if (nz >= 1 && 2 * nz <= G) {
        int hi = (sumc + (G - nz) - 1) / (G - nz);      // always feasible
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (sum_all((c + mid - 1) / mid) <= G) hi = mid; else lo = mid + 1;
        }
        aligned = akv_attn_aligned_pays(lo, equal, shares, longer);
      }
      if (aligned) {
        const int k = (c + lo - 1) / lo;
        const int inc = akv_wave_inclusive_scan(k);
        if (lane == 63 && tid < 256) p_part[4 * turn + (tid >> 6)] = inc;
        __syncthreads();
        int first = inc - k;
        for (int w = 0; w < 3; ++w)
          if (w < (tid >> 6)) first += p_part[4 * turn + w];
        if (tid < 256) p_wfirst[tid] = first;
        if (tid == 255) p_wfirst[256] = first + k;
        if (tid < S) {
          seqw[2 * tid] = first;
          seqw[2 * tid + 1] = first + k - 1;
        }
        // a few records a sequence: by its thread (100 contexts of 100 to 1,000, tq35, 16 heads on 4: the step 37.7 us; looked up
        // below, 38.4)
        if (!__syncthreads_or(k > 8)) {
          const int pc = k > 0 ? (c + k - 1) / k * cb : 0;
          for (int j = 0; j < k; ++j) {
            int32_t* rec = wgdesc + (size_t)(first + j) * AKV_WGREC;
            rec[AKV_WGREC_G0] = b0 + j * pc;              // (below b1: k - 1 ranges of at most lo chunks do not hold c)
            rec[AKV_WGREC_G1] = min(b1, b0 + (j + 1) * pc);
            rec[AKV_WGREC_SEQ] = tid;
            rec[AKV_WGREC_SB0] = b0;
            rec[AKV_WGREC_SB1] = b1;
            rec[AKV_WGREC_CTX] = p_ctx[tid];
          }
          for (int w = p_wfirst[256] + tid; w < G; w += blockDim.x) {
            int32_t* rec = wgdesc + (size_t)w * AKV_WGREC;
            rec[AKV_WGREC_G0] = rec[AKV_WGREC_G1] = 0;
            rec[AKV_WGREC_SEQ] = -1;
          }
          return;
        }
      }
    }
    if (!aligned) {
      const int per = (p_pref[256] + G - 1) / G;
      for (int s = tid; s < S; s += blockDim.x) {
        const int first = prefix[s], last = prefix[s + 1];
        const int w_lo = per > 0 ? first / per : 0;
        seqw[2 * s] = w_lo;
        seqw[2 * s + 1] = (per > 0 && last > first) ? (last - 1) / per : w_lo - 1;
      }
    }
  } else if (tid < 64) {
    int blocks = 0, ctx = 0;
    if (lane < S) {
      ctx = (int)akv_seq_tokens(context_lens, cl_itype, lane, block_size, max_blocks_per_seq);
      blocks = (ctx + block_size - 1) / block_size;
    }
    const int inc = akv_wave_inclusive_scan(blocks);
    const int total = __builtin_amdgcn_readlane(inc, 63);
    const int b0 = inc - blocks;
    if (lane < S) prefix[lane] = b0;
    if (lane == 0) prefix[S] = total;
    p_pref[lane] = b0;
    p_ctx[lane] = ctx;
    const int c = (blocks + cb - 1) / cb;                        // chunks of the lane's sequence
    const int sumc = akv_wave_sum(c);
    const int nz = __popcll(__ballot(c > 0));
    aligned = nz >= 1 && nz * 8 <= G;
    int lo = (sumc + G - 1) / G;
    if (lo < 1) lo = 1;
    if (aligned || (nz >= 1 && 2 * nz <= G)) {
      const int equal = lo;
      int hi = (sumc + (G - nz) - 1) / (G - nz);      // always feasible
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        const int tot = akv_wave_sum((c + mid - 1) / mid);
        if (tot <= G) hi = mid; else lo = mid + 1;
      }
      if (akv_attn_aligned_pays(lo, equal, shares, longer)) aligned = true;
    }
    if (aligned) {
      const int k = (c + lo - 1) / lo;
      const int kinc = akv_wave_inclusive_scan(k);
      p_wfirst[lane] = kinc - k;
      if (lane == 63) p_wfirst[64] = kinc;
      if (lane < S) {
        seqw[2 * lane] = kinc - k;
        seqw[2 * lane + 1] = kinc - 1;
      }
    } else if (lane < S) {
      const int per = (total + G - 1) / G;
      const int w_lo = per > 0 ? b0 / per : 0;
      seqw[2 * lane] = w_lo;
      seqw[2 * lane + 1] = (per > 0 && blocks > 0) ? (b0 + blocks - 1) / per : w_lo - 1;
    }
    if (lane == 0) {
      p_pref[64] = total;
      p_mode[0] = aligned ? 1 : 0;
    }
  }
  __syncthreads();
  if (S <= 64) aligned = p_mode[0] != 0;
  const int total = p_pref[n], per = (total + G - 1) / G;
  auto record = [&](int w, int s) {
    int g0 = 0, g1 = 0, b0 = p_pref[s], b1 = p_pref[s + 1];
    if (aligned) {
      if (w < p_wfirst[n]) {
        const int k = p_wfirst[s + 1] - p_wfirst[s];
        const int c = (b1 - b0 + cb - 1) / cb;
        const int pc = (c + k - 1) / k;
        g0 = min(b1, b0 + (w - p_wfirst[s]) * pc * cb);
        g1 = min(b1, g0 + pc * cb);
      }
    } else {
      g0 = min(total, w * per);
      g1 = min(total, g0 + per);
      if (g0 < g1 && chunk > 1) {
        int hi = min(S, (s + 1) * chunk);     // prefix[s] <= g0 < prefix[hi]
        s *= chunk;
        while (hi - s > 1) {
          const int mid = (s + hi) >> 1;
          if (prefix[mid] <= g0) s = mid; else hi = mid;
        }
        b0 = prefix[s];
        b1 = prefix[s + 1];
      }
    }
    int32_t* rec = wgdesc + (size_t)w * AKV_WGREC;
    rec[AKV_WGREC_G0] = g0;
    rec[AKV_WGREC_G1] = g1;
    rec[AKV_WGREC_SEQ] = g0 < g1 ? s : -1;
    if (g0 < g1) {
      rec[AKV_WGREC_SB0] = b0;
      rec[AKV_WGREC_SB1] = b1;
      rec[AKV_WGREC_CTX] = S > 256 ? (int)akv_seq_tokens(context_lens, cl_itype, s, block_size, max_blocks_per_seq) : p_ctx[s];
    }
  };
  for (int w = tid; w < G; w += 2 * blockDim.x) {
    // The sequence of a workgroup: the last whose first workgroup, or whose start, does not lie behind it.  (One without
    // workgroups or blocks shares the next one's entry and is passed over; entries past the batch equal the number of workgroups in use,
    // or of blocks.  Workgroups that get nothing: any.)
    const int w1 = w + (int)blockDim.x;
    int s0, s1;
    if (aligned) akv_last_at_most(p_wfirst, n, min(w, p_wfirst[n] - 1), min(w1, p_wfirst[n] - 1), s0, s1);
    else akv_last_at_most(p_pref, n, min(w * per, total - 1), min(w1 * per, total - 1), s0, s1);
    record(w, s0);
    if (w1 < G) record(w1, s1);
  }
}

// largest s with prefix[s] <= g  (prefix non-decreasing, prefix[0] = 0, g < prefix[S])
__device__ __forceinline__ int akv_find_seq(const int32_t* __restrict__ prefix, int S, int g) {
  int lo = 0, hi = S;  // invariant: prefix[lo] <= g < prefix[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (prefix[mid] <= g) lo = mid; else hi = mid;
  }
  return lo;
}

// The sequence of a workgroup's next segment, for a whole wavefront: `s` held the segment before, the range goes on at global block
// `g` = that sequence's end < prefix[S].  Mostly the next one, its end one load away; empty sequences are passed over 64 at a time.
// (A binary search was a chain of dependent loads, eight for 256 sequences, in every segment, the first
// included: a step of 200 contexts of 300 took 57.2 us, now 54.5; 100 of 600 46.4, now 43.7.)
__device__ __forceinline__ int akv_next_seq(const int32_t* __restrict__ prefix, int S, int s, int g, int& sb0, int& sb1) {
  ++s;
  sb0 = g;
  sb1 = __builtin_amdgcn_readfirstlane(prefix[s + 1]);
  if (sb1 <= g) {
    int below;
    do {
      const int end = prefix[min(s + 1 + (int)(threadIdx.x & 63), S)];
      below = __popcll(__ballot(end <= g));
      if (below < 64) sb1 = __builtin_amdgcn_readlane(end, below);
      s += below;
    } while (below == 64);
  }
  return s;
}

// merge (m, l, acc) <- (m, l, acc) (+) (ms, ls, accs)
__device__ __forceinline__ void akv_lse_merge(float& m, float& l, float ms, float ls,
                                              float& alpha, float& beta) {
  const float mn = fmaxf(m, ms);
  if (mn == -INFINITY) { alpha = 1.f; beta = 0.f; return; }
  alpha = __expf(m - mn);
  beta = __expf(ms - mn);
  l = alpha * l + beta * ls;
  m = mn;
}

// ----------------------------------------------------------------------------------
// 128 x 128 rotations of a few float32 rows on the matrix cores (query rotation of the prologue,
// inverse rotation of the reduce).  The matrix comes as the float16 hi + lo operand tables of the
// prepared-rotation buffer (entries x 64; [hi | lo][8 N-tiles][4 k-steps][64 lanes] x 16 bytes, lane
// (col, g) = output coordinate 8 col + N-tile, contracted coordinates 32 g + 8 k-step + e).  A row is
// scaled by a power of two that brings its largest element to [1, 2) (exact), split into two float16
// terms rounded to nearest, and a tile is three products: hi.hi + hi.lo + lo.hi (~22 bits).
// ----------------------------------------------------------------------------------
typedef _Float16 akv_half8 __attribute__((ext_vector_type(8)));
typedef float akv_float4v __attribute__((ext_vector_type(4)));

// max over the four 16-lane rows of a wavefront, for every column (lane % 16)
__device__ __forceinline__ float akv_rows_max(float v) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
// biased exponent used to scale a row whose largest magnitude is m (clamped so that both factors are normal)
__device__ __forceinline__ uint32_t akv_row_exponent(float m) {
  const uint32_t e = (__float_as_uint(m) >> 23) & 0xffu;
  return e < 1u ? 1u : (e > 253u ? 253u : e);
}
__device__ __forceinline__ float akv_row_scale(uint32_t e) { return __uint_as_float((254u - e) << 23); }     // 2^(127 - e)
__device__ __forceinline__ float akv_row_unscale(uint32_t e) { return __uint_as_float(e << 23); }             // 2^(e - 127)
// eight scaled values as two float16 operands
__device__ __forceinline__ void akv_split8(const float (&v)[8], float sc, akv_half8& hi, akv_half8& lo) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float x = v[e] * sc;
    const _Float16 h = (_Float16)x;
    hi[e] = h;
    lo[e] = (_Float16)(x - (float)h);
  }
}
__device__ __forceinline__ akv_half8 akv_as_half8(uint4 u) {
  union { uint4 u; akv_half8 h; } cv;
  cv.u = u;
  return cv.h;
}
// acc += (hi + lo) . (bh + bl) without the lo.lo term
__device__ __forceinline__ akv_float4v akv_mfma3(akv_half8 hi, akv_half8 lo, akv_half8 bh, akv_half8 bl, akv_float4v acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, bh, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, bl, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, bh, acc, 0, 0, 0);
  return acc;
}

// Row shifts that write ONE bank (four neighbouring lanes) of every row of sixteen; the other lanes keep `old`.
// akv_to_bank<K>: lane 4K + c of a row receives `src` of lane c.
template <int K>
__device__ __forceinline__ float akv_to_bank(float old, float src) {
  static_assert(K >= 1 && K <= 3, "bank 0 holds its own values");
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(src), 0x110 + 4 * K /*row_shr:4K*/, 0xf, 1 << K, false));
}
// akv_dpp_bank<CTRL, K>: lanes of bank K receive `src` through the row operation CTRL, the others keep `old`;
// akv_dpp_banks<CTRL, MASK>: the same for a set of banks
template <int CTRL, int K>
__device__ __forceinline__ float akv_dpp_bank(float old, float src) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(src), CTRL, 0xf, 1 << K, false));
}
template <int CTRL, int MASK>
__device__ __forceinline__ float akv_dpp_banks(float old, float src) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(src), CTRL, 0xf, MASK, false));
}
template <int CTRL, int MASK>
__device__ __forceinline__ uint32_t akv_dpp_banks_u(uint32_t old, uint32_t src) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)src, CTRL, 0xf, MASK, false);
}
// akv_pair_from_bank<Q>: lanes 0..3 of a row receive `hi` of lanes 4Q + c, lanes 8..11 receive `lo` of lanes 4Q + c,
// every other lane zero (quad_perm 0,1,2,3 is the shift by nothing)
template <int Q>
__device__ __forceinline__ uint32_t akv_pair_from_bank(uint32_t hi, uint32_t lo) {
  constexpr int hi_ctrl = Q == 0 ? 0xE4 : 0x100 + 4 * Q;                                            // row_shl:4Q
  constexpr int lo_ctrl = Q == 2 ? 0xE4 : (Q < 2 ? 0x110 + (8 - 4 * Q) : 0x100 + (4 * Q - 8));      // row_shr:8-4Q / row_shl:4Q-8
  int w = __builtin_amdgcn_update_dpp(0, (int)hi, hi_ctrl, 0xf, 0x1, false);
  w = __builtin_amdgcn_update_dpp(w, (int)lo, lo_ctrl, 0xf, 0x4, false);
  return (uint32_t)w;
}
// sum / maximum over the four banks of a row (every lane gets the result of the lanes c, c + 4, c + 8, c + 12)
__device__ __forceinline__ float akv_banks_max(float v) {
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124 /*row_ror:4*/, 0xf, 0xf, false)));
  return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128 /*row_ror:8*/, 0xf, 0xf, false)));
}
__device__ __forceinline__ float akv_banks_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124 /*row_ror:4*/, 0xf, 0xf, false));
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128 /*row_ror:8*/, 0xf, 0xf, false));
}
// sum over the four 16-lane rows of a wavefront, for every column
__device__ __forceinline__ float akv_rows_sum(float v) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
// LDS written by a lane of the wavefront is read by another
__device__ __forceinline__ void akv_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// workgroup barrier that orders LDS traffic only (what has been requested from memory keeps flying)
__device__ __forceinline__ void akv_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
