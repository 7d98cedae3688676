// mac_prefill.hip -- prefill rectification for MI355X (gfx950).
//
// A ring entry at logical position p holds the attention state of the query
// of p over the keys [0, E), E = p + 1 - S (S = semantic_pos_ahead), so that a
// later decode step that matches it only has to add the band [E, now).  The
// prefill attention computes the state over [0, p + 1); the reference removes
// the trailing window [E, p + 1) with a second, windowed FlashInfer pass and a
// log-sum-exp "downdate" (flashinfer_hooks.py:2436-2482,
// mac_merge_downdate_cache.cu:116-288).  This file provides:
//
//  * downdate_kernel: the reference's downdate op on its own (any head_dim,
//    f32/bf16/f16 lse), for callers that keep the reference's three calls.
//  * window_kernel<RT, kPlain, ..>: causal sliding-window attention over a
//    ragged batch with a page-size-1 KV pool (the windowed FlashInfer pass).
//  * window_kernel<RT, kRectify, ..>: the fused form.  Only the rows the ring keeps
//    (the last min(len, M) of each request) are computed; for them the window
//    state never leaves registers: it is downdated from the full state and
//    stored straight into the ring with the pre-RoPE query, followed by the
//    request_length bump (bump_kernel).
//
// Both forms run S^T[key][row] = K Q^T and O^T[d][row] += V^T P^T on
// v_mfma_f32_16x16x32_bf16 as the decode kernel does, with 16 query rows in
// place of the GQA heads: the lane holding row l%16 keeps that row's softmax
// state and 32 O^T accumulators per head.  A workgroup takes rows of one
// request and query heads of one KV head, 128 or 64 (row, head) columns in all;
// its four waves share double-buffered LDS K/V tiles.  The layouts are described
// above window_kernel.

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <climits>
#include <cmath>

#include "mac_attention_amd.h"
#include "mac_common.h"

namespace mac {
int fail(int code, const char* fmt, ...);
}  // namespace mac

namespace {

typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

using namespace mac;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8_t as_bf16x8(const uint4& w) { return __builtin_bit_cast(bf16x8_t, w); }

// ------------------------------------------------------------- downdate ----

// Control scalars of the downdate (MERGE:148-176), fp32 as in the reference
// so that its branch decisions are reproduced.
struct Downdate {
  float lse;    // new natural-log lse (-inf: nothing left)
  float t;      // weight of the removed state
  float scale;  // renormalisation
};

__device__ __forceinline__ Downdate downdate_control(float l1, float l2) {
  const float diff = l2 - l1;
  const bool last_block = fabsf(expm1f(diff)) <= 1e-7f;
  const bool invalid = diff > 0.0f && !last_block;
  Downdate d;
  if (last_block) {
    d.lse = -INFINITY;
    d.t = 0.0f;
    d.scale = 0.0f;
  } else if (invalid) {
    d.lse = l1;
    d.t = 0.0f;
    d.scale = 1.0f;
  } else {
    d.lse = l1 + logf(fmaxf(1.0f - expf(diff) + 1e-7f, 1e-30f));
    d.t = expf(diff);
    d.scale = expf(l1 - d.lse);
  }
  return d;
}

__device__ __forceinline__ float load_lse(const void* p, int dtype, int64_t i) {
  if (dtype == MAC_DTYPE_F32) return static_cast<const float*>(p)[i];
  const uint16_t b = static_cast<const uint16_t*>(p)[i];
  if (dtype == MAC_DTYPE_BF16) return bf16_to_f32(b);
  return static_cast<float>(__builtin_bit_cast(_Float16, b));
}

__device__ __forceinline__ void store_lse(void* p, int dtype, int64_t i, float v) {
  if (dtype == MAC_DTYPE_F32) {
    static_cast<float*>(p)[i] = v;
  } else if (dtype == MAC_DTYPE_BF16) {
    static_cast<uint16_t*>(p)[i] = f32_to_bf16(v);
  } else {
    static_cast<uint16_t*>(p)[i] = __builtin_bit_cast(uint16_t, static_cast<_Float16>(v));
  }
}

// One 16-lane row group per row; 16 rows per 256-thread workgroup.  Every
// lane reads lse2 before the group's lane 0 overwrites it (same wave, program
// order), so no row reads a half-updated lse.
__global__ void __launch_bounds__(256) downdate_kernel(const uint16_t* __restrict__ out1,
                                                       const void* __restrict__ lse1, int dt1,
                                                       uint16_t* __restrict__ out2, void* __restrict__ lse2,
                                                       int dt2, int64_t rows, int D) {
  // Each 16-lane group takes kR rows at a time (rows g, g + 16, ... of the
  // workgroup's slab) with every load issued before the math; the rows are
  // read once, so o1 and o2 move with the non-temporal policy.
  constexpr int kR = 4;
  const int sub = threadIdx.x & 15;
  const int64_t step = static_cast<int64_t>(gridDim.x) * 16 * kR;
  for (int64_t row0 = static_cast<int64_t>(blockIdx.x) * 16 * kR + (threadIdx.x >> 4); row0 < rows; row0 += step) {
    Downdate c[kR];
#pragma unroll
    for (int k = 0; k < kR; ++k) {
      const int64_t row = min(row0 + 16 * k, rows - 1);
      c[k] = downdate_control(load_lse(lse1, dt1, row), load_lse(lse2, dt2, row));
    }
    if ((D & 7) == 0) {
      for (int e = sub * 8; e < D; e += 128) {
        uint4 wa[kR], wb[kR];
#pragma unroll
        for (int k = 0; k < kR; ++k) {
          const int64_t row = min(row0 + 16 * k, rows - 1);
          wa[k] = __builtin_bit_cast(uint4, __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(out1 + row * D + e)));
          wb[k] = __builtin_bit_cast(uint4, __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(out2 + row * D + e)));
        }
#pragma unroll
        for (int k = 0; k < kR; ++k) {
          if (row0 + 16 * k >= rows) break;
          float fa[8], fb[8];
          unpack8(wa[k], fa);
          unpack8(wb[k], fb);
          uint16_t r[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) r[i] = f32_to_bf16((fa[i] - c[k].t * fb[i]) * c[k].scale);
          u32x4_t w;
          w[0] = r[0] | (static_cast<uint32_t>(r[1]) << 16);
          w[1] = r[2] | (static_cast<uint32_t>(r[3]) << 16);
          w[2] = r[4] | (static_cast<uint32_t>(r[5]) << 16);
          w[3] = r[6] | (static_cast<uint32_t>(r[7]) << 16);
          __builtin_nontemporal_store(w, reinterpret_cast<u32x4_t*>(out2 + (row0 + 16 * k) * D + e));
        }
      }
    } else {
#pragma unroll
      for (int k = 0; k < kR; ++k) {
        const int64_t row = row0 + 16 * k;
        if (row >= rows) break;
        const uint16_t* a = out1 + row * D;
        uint16_t* b = out2 + row * D;
        for (int e = sub; e < D; e += 16)
          b[e] = f32_to_bf16((bf16_to_f32(a[e]) - c[k].t * bf16_to_f32(b[e])) * c[k].scale);
      }
    }
    if (sub == 0) {
#pragma unroll
      for (int k = 0; k < kR; ++k)
        if (row0 + 16 * k < rows) store_lse(lse2, dt2, row0 + 16 * k, c[k].lse);
    }
  }
}

// ------------------------------------------------------ window attention ----

constexpr int kMaxB = 4096;  // requests handled by the in-workgroup planner
constexpr int kTiles = 8;    // column tiles (16 query rows of one head) of a wide task

struct WindowParams {
  const uint16_t* q;  // attention queries [total_q, Hq, 128]
  const uint16_t* k;
  const uint16_t* v;
  const int32_t* qo_indptr;
  const int32_t* kv_indptr;
  const int32_t* kv_indices;
  // plain window attention
  uint16_t* out;
  float* out_lse;
  // split form: partial states of the pieces, the most pieces they hold and
  // the most row blocks that window_combine_kernel's grid covers
  float* part_o;
  float* part_ml;
  int max_pieces, max_blocks;
  // fused rectification
  const uint16_t* src_q;
  const uint16_t* o_full;
  const float* lse_full;
  uint16_t* q_cache;
  uint16_t* attn_cache;
  float* lse_cache;
  uint16_t* q_post_cache;
  const int32_t* request_length;
  const int32_t* req_ids;
  int64_t pool_tokens;
  int64_t total_q, kv_len_total;  // rows of q, entries of kv_indices
  int B, Hq, Hkv, R, M;
  int window_left;  // plain mode: keys [pos - window_left, pos]; < 0: [0, pos]
  int S, F, sink_mode;
  int rl_by_batch;
  float q_scale;  // sm_scale * log2(e)
};

enum WindowMode { kPlain = 0, kRectify = 1, kSplit = 2 };

// First row of request b that a kernel computes: 0 (every row), or the first
// of the last min(len, M) rows, which the ring keeps (fused form).
template <int kMode>
__device__ __forceinline__ int first_row(int len, int M) {
  return kMode == kRectify ? (len > M ? len - M : 0) : 0;
}

// Rows of request b the kernel computes; 0 for requests whose query or key
// ranges fall outside the buffers the caller described, or with fewer keys
// than queries.
template <int kMode>
__device__ __forceinline__ int request_rows(const WindowParams& p, int b) {
  const int q0 = p.qo_indptr[b], q1 = p.qo_indptr[b + 1];
  const int k0 = p.kv_indptr[b], k1 = p.kv_indptr[b + 1];
  const int len = q1 - q0, kvlen = k1 - k0;
  const bool ok = q0 >= 0 && q1 <= p.total_q && k0 >= 0 && k1 <= p.kv_len_total && len > 0 && kvlen >= len;
  return ok ? len - first_row<kMode>(len, p.M) : 0;
}

// Exclusive scan of one value per thread over a 256-thread workgroup; the
// total goes to `total`.  s_tmp: kWaves entries; ends with a barrier.
__device__ __forceinline__ int scan256(int v, int* s_tmp, int& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(x, off);
    if (lane >= off) x += y;
  }
  if (lane == 63) s_tmp[wave] = x;
  __syncthreads();
  int base = x - v;
  total = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    if (w < wave) base += s_tmp[w];
    total += s_tmp[w];
  }
  __syncthreads();
  return base;
}

// The plan of a batch, derived by every workgroup: s_boff[b] = pieces of the
// requests before b.  A piece is a block of kRowsT rows (plain and fused
// forms) or one key chunk of such a block (split form: ceil(kvlen / chunk)
// chunks per block).  Returns the chunk (split form).
//
// Split form: the number of key chunks must fit p.max_pieces partial states
// and follows from the batch: with W = sum of blocks x keys and NB blocks,
// chunk = W / (max_pieces - NB) rounded up to whole 64-key blocks gives at
// most W / chunk + NB <= max_pieces pieces.  Requests whose query ranges
// overlap can hold more row blocks than the caller's row count allows for
// (p.max_blocks), which is all the combining launch covers: the chunk is then
// kNoChunk, every piece is a whole block and writes its result itself.
constexpr int kNoChunk = 1 << 30;  // (a request has fewer keys)
constexpr int kMinSplitKeys = 256;  // smallest chunk: a piece's prologue and state cost about as much

template <int kMode, int kRowsT>
__device__ __forceinline__ int plan_pieces(const WindowParams& p, int* s_boff, int* s_tmp) {
  const int tid = threadIdx.x;
  const int B = p.B;
  const int per = ceil_div(B, 256);
  const int b0 = min(B, tid * per), b1 = min(B, b0 + per);
  int chunk = 0;
  if (kMode == kSplit) {
    int nb = 0;
    long long w = 0;
    for (int b = b0; b < b1; ++b) {
      const int n = ceil_div(request_rows<kMode>(p, b), kRowsT);
      nb += n;
      w += static_cast<long long>(n) * (p.kv_indptr[b + 1] - p.kv_indptr[b]);
    }
    int total_nb;
    scan256(nb, s_tmp, total_nb);
    __shared__ long long s_w[kWaves];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) w += __shfl_xor(w, off);
    if ((tid & 63) == 0) s_w[tid >> 6] = w;
    __syncthreads();
    w = 0;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) w += s_w[i];
    const int room = total_nb <= p.max_blocks ? p.max_pieces - total_nb : 0;
    const long long c = room > 0 ? ((w + room - 1) / room + 63) / 64 * 64 : kNoChunk;
    chunk = static_cast<int>(min(max(c, static_cast<long long>(kMinSplitKeys)), static_cast<long long>(kNoChunk)));
  }
  int sum = 0;
  for (int b = b0; b < b1; ++b) {
    int n = ceil_div(request_rows<kMode>(p, b), kRowsT);
    if (kMode == kSplit && n > 0) n *= ceil_div(p.kv_indptr[b + 1] - p.kv_indptr[b], chunk);
    s_boff[b] = n;  // the count until the prefix replaces it below
    sum += n;
  }
  int total;
  int acc = scan256(sum, s_tmp, total);
  for (int b = b0; b < b1; ++b) {
    const int n = s_boff[b];
    s_boff[b] = acc;
    acc += n;
  }
  if (tid == 0) s_boff[B] = total;
  __syncthreads();
  return chunk;
}

// Largest b < B with s_boff[b] <= piece.
__device__ __forceinline__ int request_of(const int* s_boff, int B, int piece) {
  int lo = 0, hi = B - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (s_boff[mid] <= piece) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Sliding-window attention for GQA groups of any size: the windowed
// FlashInfer pass (kPlain), the same over pieces of a row's keys with partial
// results (kSplit, for batches with too few row blocks to fill the GPU), or
// the fused rectification of the rows the ring keeps (kRectify: a window of S
// keys, optionally the front sink [0, min(F, E)) as a second key segment, P
// fed to the PV product as bf16 hi + lo, and the downdate and ring write as
// epilogue).
//
// A task is 4 kPer column tiles of one KV head: a tile is 16 consecutive query
// rows of one query head, each of the four waves owns kPer of them.  Wide tasks
// (kPer 2) are RT row tiles x 8 / RT heads, RT picked from the GQA group so
// that no tile is wasted on an absent head (G > 4: 16 rows x 8 heads; 3, 4: 32
// x 4; 2: 64 x 2; 1: 128 x 1), so that every K and V operand a wave reads from
// LDS feeds 32 columns whatever the group size.  Narrow tasks (kPer 1, RT 1: 16
// rows x 4 heads) have the shorter chain (see narrow_tasks).  K/V rows are
// staged in double-buffered LDS tiles of kBlk keys: 64 (one barrier and one
// round of address work per 64 keys), or 32 (fused form, whose epilogue also
// holds the full state's rows in LDS, narrow tasks, and see long_blocks).  Per
// wave and 32 keys:
//  * S^T = K Q^T: the A operand of score tile t, row m, is key 16 t + m; the
//    lane holding column col ends up with the scores of keys 16 t + 4 quad +
//    (0..3), quad = lane / 16.
//  * O^T += V^T P^T: V stays token-major in LDS; the A operand of each 16-dim
//    tile is two transposing LDS reads (ds_read_b64_tr_b16: in each 16-lane
//    group, lane i receives element i & 3 of the 4-element vectors of lanes
//    4e + (i >> 2), e < 4), the first of keys 4 quad + (0..3), the second of
//    keys 16 + 4 quad + (0..3): the same order of keys as P has in the lane's
//    B operand, so P goes from the score tiles to the PV product unmoved.
// LDS layouts: K chunk c (16 bytes) of key k at position c ^ (k & 15) of its
// 256-byte row; V row k at 288 k bytes.  A K read covers 16 consecutive keys
// on 16 different chunk positions, also where the hardware pairs lanes of two
// quads (rows padded to 272 bytes instead cost one conflict cycle per group
// of 16 lanes there: 23% of the LDS cycles), and the 8 keys of a V read (two
// quads) are 32 bytes apart in the banks.
// What bounds it: per wave and 32 keys, 32 MFMAs (512 clocks) and about 105
// other VALU instructions (670 clocks, the exponentials at a quarter of the
// rate) that the SIMD's two waves overlap only partly: 1500 clocks per wave
// and 32 keys, 800-850 TFLOP/s over long windows (a large bf16 matrix product
// reaches 1200 on the same card).  Before every wave had two tiles, groups of
// at most four heads read each operand for 16 columns only.  8 x 8192 rows,
// 32 query heads, window 256 / 2048 (us), one tile per wave -> two: 4 heads
// per group 655 / 3570 -> 577 / 2655; 1 head 1840 / 9470 -> 706 / 2930 (8
// heads had two before: 549 / 2600).  The fused form, 8 x 512 kept rows,
// 4 heads per group: 72 -> 62 us.
// The running maximum is moved lazily (only when a block exceeds it by 2^8),
// which leaves the result exact and skips most accumulator rescales.

constexpr int kKRow = 16;  // 16-byte units per staged K row
constexpr int kVRow = 18;  // per staged V row: 256 + 32

template <int RT, int kPer, int kMode, int kBlk>
__global__ void __launch_bounds__(256, (kPer == 1 && kMode == kPlain) ? 3 : 2) window_kernel(WindowParams p) {
  constexpr bool kFused = kMode == kRectify;
  constexpr int kTask = kWaves * kPer;  // column tiles of a task
  constexpr int kHeads = kTask / RT;    // query heads of a task
  constexpr int kRowsT = 16 * RT;       // query rows of a task
  constexpr bool kTrim = kMode == kPlain && kBlk == 32;  // no loads of 16-key groups past the keys' end
  constexpr int kSub = kBlk / 32;
  constexpr int kLd = kBlk / 16;  // keys each thread stages a chunk of
  // dynamic: s_boff[B + 1] piece offsets, s_qo[B + 1] / s_kv[B + 1] the
  // request offsets (copies of qo_indptr / kv_indptr)
  extern __shared__ int s_dyn[];
  int* s_boff = s_dyn;
  int* s_qo = s_dyn + (p.B + 1);
  int* s_kv = s_dyn + 2 * (p.B + 1);
  __shared__ int s_part[kWaves];
  __shared__ uint4 s_k[2][kBlk * kKRow];
  __shared__ uint4 s_v[2][kBlk * kVRow];
  __shared__ __align__(16) uint32_t s_bad[2][kWaves * kSub];  // per wave: its keys (of each 32) that have no pool row

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int quad = lane >> 4;
  const int col = lane & 15;
  const int B = p.B;
  for (int b = tid; b <= B; b += 256) {
    s_qo[b] = p.qo_indptr[b];
    s_kv[b] = p.kv_indptr[b];
  }
  const int chunk = plan_pieces<kMode, kRowsT>(p, s_boff, s_part);
  const int Hq = p.Hq, Hkv = p.Hkv;
  const int G = Hq / Hkv;
  // fused form: the full state's o rows of the task.  Pair e = row * kHeads +
  // head takes 16 16-byte units from unit 16 e + (e >> 2) on (the extra unit
  // per four pairs spreads the rows over the banks; a wave's direct copy
  // fills four pairs, one contiguous 1 KiB run)
  __shared__ uint4 s_of[kFused ? kTask * (16 * 16 + 4) : 1];
  const int nchunks = ceil_div(G, kHeads);
  const int per_piece = Hkv * nchunks;
  const int total_tasks = s_boff[B] * per_piece;
  const uint32_t row_bytes = static_cast<uint32_t>(Hkv) * kHeadDim * 2;  // one pool row of K or V
  const unsigned pool_rows = static_cast<unsigned>(min(p.pool_tokens, static_cast<int64_t>(INT_MAX)));
  // keys [pos - wl, pos] form a row's window (wl < 0: [0, pos])
  const int wl = kFused ? p.S - 1 : p.window_left;
  const bool sink = kFused && p.sink_mode == 1 && p.F > 0;  // the front sink [0, min(F, E)) as well
  // loader side: thread t stages 16-byte chunk t%16 of keys t/16 + 16 i
  const int ld_key = tid >> 4, ld_chunk = tid & 15;
  u32x4_t* const ld_k = reinterpret_cast<u32x4_t*>(&s_k[0][0]) + ld_key * kKRow + (ld_chunk ^ ld_key);
  u32x4_t* const ld_v = reinterpret_cast<u32x4_t*>(&s_v[0][0]) + ld_key * kVRow + ld_chunk;
  // compute side: this lane's K row (key col) and V^T read position (key 4
  // quad + (col >> 2), dims 4 (col & 3) ..)
  const uint4* rd_k[4];  // by k-step
#pragma unroll
  for (int s = 0; s < 4; ++s) rd_k[s] = &s_k[0][0] + col * kKRow + ((4 * s + quad) ^ col);
  const uint16_t* const rd_v =
      reinterpret_cast<const uint16_t*>(&s_v[0][0]) + (4 * quad + (col >> 2)) * (kVRow * 8) + 4 * (col & 3);
  // the wave's tiles c < kPer: task head and first row in the task
  int th[kPer], tr[kPer];
#pragma unroll
  for (int c = 0; c < kPer; ++c) {
    th[c] = (kPer * wave + c) / RT;
    tr[c] = 16 * ((kPer * wave + c) % RT);
  }

  // Task order, by form (measured at 64 requests x 8192 rows, S = 256):
  //  * windowed (plain, window_left >= 0): (KV head, head chunk) major, row
  //    block minor, and within each full round of the grid XCD x (the
  //    workgroups w with w % 8 == x, as the dispatcher deals them) takes the
  //    x-th contiguous eighth of the round's tasks: the row blocks sharing a
  //    K/V row run together under one L2 (row-block order dealt round-robin
  //    put them on different XCDs and fetched each K/V row about four times);
  //  * fused: row-block order (the KV heads of a row block together), XCD
  //    eighths as above (2-3% faster than round-robin; head-major was slower);
  //  * causal (window_left < 0) and split: row-block order dealt
  //    round-robin.  Causal tasks grow with the row block, and a workgroup
  //    would keep its offset within every round: with as many tasks per request
  //    as divide the grid (or nearly) some would take only the longest ones.
  //    So with as many row blocks in every request, where the offsets recur,
  //    every other round is dealt backwards (unsplit form: 8 x 1024 rows, 4
  //    heads per group, 168 us forwards, 111 back and forth; 2 x 2048 rows 139
  //    and 96), and so is a last, partial one (5 x 1037 rows 113 and 93).
  //    Ragged batches only gain and lose by it (5 x 765-1529 rows, 8 heads per
  //    group, 136 and 153).  Backwards in whole eights, which keeps an XCD's KV
  //    heads, gained nothing (8 heads per group and 4 KV heads, 5 x 1037 rows,
  //    96 and 118).
  const int grid = gridDim.x;
  const int eighth = grid / 8;
  const int npieces = s_boff[B];
  const bool head_major = kMode == kPlain && wl >= 0;
  const bool by_xcd = (kFused || (kMode == kPlain && wl >= 0)) && grid % 8 == 0;
  bool back_and_forth = false;
  if (kMode == kPlain && wl < 0) {
    int same = 1;
    for (int b = tid; b < B; b += 256) same &= s_boff[b + 1] - s_boff[b] == s_boff[1];
    back_and_forth = __syncthreads_and(same) != 0;
  }
  bool odd_round = true;
  for (int task = blockIdx.x; task < total_tasks; task += grid) {
    __syncthreads();  // the previous task's waves are done with the tiles
    const int round0 = task - static_cast<int>(blockIdx.x);
    odd_round = !odd_round;
    const bool backwards = back_and_forth && (odd_round || (round0 > 0 && round0 + grid > total_tasks));
    const int t = (by_xcd && round0 + grid <= total_tasks)
                      ? round0 + (static_cast<int>(blockIdx.x) % 8) * eighth + static_cast<int>(blockIdx.x) / 8
                      : (backwards ? round0 + min(grid, total_tasks - round0) - 1 - static_cast<int>(blockIdx.x) : task);
    int piece, hc;  // piece; KV head * nchunks + head chunk
    if (head_major) {
      hc = t / npieces;
      piece = t - hc * npieces;
    } else {
      piece = t / per_piece;
      hc = t - piece * per_piece;
    }
    const int hkv = hc / nchunks;
    const int hg0 = kHeads * (hc - hkv * nchunks);  // first head of the task in the group
    const int b = request_of(s_boff, B, piece);
    const int len = s_qo[b + 1] - s_qo[b];
    const int kvlen = s_kv[b + 1] - s_kv[b];
    const int64_t kv_begin = s_kv[b];
    int blk = piece - s_boff[b], key_lo = 0, key_hi = INT_MAX;  // row block and key chunk
    if (kMode == kSplit) {  // chunk-major: the row blocks that share a chunk's keys together
      const int nb = ceil_div(len, kRowsT);
      const int ch = blk / nb;
      blk -= ch * nb;
      key_lo = ch * chunk;
      key_hi = key_lo + min(chunk, kvlen - key_lo);
    }
    const int r_local = first_row<kMode>(len, p.M) + kRowsT * blk;
    const int nrows = min(kRowsT, len - r_local);
    const int pos0 = kvlen - len + r_local;
    const int pos_last = pos0 + nrows - 1;
    if (kMode == kSplit && key_lo > pos_last) continue;  // (past every row: the combine skips it too)
    // tile c of the wave: lane's row in the task, position, first key of its window
    bool live = false;
    int row[kPer], wlo[kPer];
    bool row_ok[kPer];
#pragma unroll
    for (int c = 0; c < kPer; ++c) {
      const bool live_c = hg0 + th[c] < G && tr[c] < nrows;
      live = live || live_c;
      row[c] = tr[c] + col;
      row_ok[c] = row[c] < nrows && live_c;
      wlo[c] = wl < 0 ? 0 : max(pos0 + row[c] - wl, 0);
    }
    // first and last row of the wave's tiles (uniform), for the mask-free test
    const int rf = min(tr[0], tr[kPer - 1]), rl = min(max(tr[0], tr[kPer - 1]) + 15, nrows - 1);
    const int wlo_f = wl < 0 ? 0 : max(pos0 + rf - wl, 0), wlo_l = wl < 0 ? 0 : max(pos0 + rl - wl, 0);
    // this request's kv_indices; entry offsets fit 32 bits (fewer than 2^30
    // entries, checked on the host), so a load is a uniform base plus a
    // 32-bit lane offset
    const char* kvi = reinterpret_cast<const char*>(p.kv_indices + kv_begin);
    const uint32_t last4 = 4u * static_cast<uint32_t>(kvlen - 1);
    auto index_at = [&](int key) -> int {  // entry of a key, clamped into the request
      return *reinterpret_cast<const int*>(kvi + min(static_cast<uint32_t>(key) * 4u, last4));
    };
    // The entries of the first segment's first two blocks (the loader's keys)
    // go out first, ahead of the Q rows and the epilogue's inputs: the first
    // K/V loads then wait for these entries only, not for everything issued
    // before them (the memory counter retires loads in order).
    const int seg_first = sink ? 0 : 1;
    const int lo_first = seg_first == 0 ? 0 : max(wl < 0 ? 0 : max(pos0 - wl, 0), key_lo);
    int pre_raw[2][kLd];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < kLd; ++i) pre_raw[u][i] = index_at(lo_first + u * kBlk + ld_key + 16 * i);
    __builtin_amdgcn_sched_barrier(0);  // (kept ahead of the loads below)
    // fused form: the epilogue's inputs that do not depend on the attention,
    // loaded now so that their latency hides behind it
    auto grow = [&](int r) { return static_cast<int64_t>(s_qo[b]) + r_local + (r < nrows ? r : 0); };
    int64_t grow_c[kPer];
#pragma unroll
    for (int c = 0; c < kPer; ++c) grow_c[c] = grow(row[c]);
    int req = 0, before = 0;
    float lse_full[kPer] = {};
    if (kFused) {
      req = p.req_ids[b];
      const bool req_ok = req >= 0 && req < p.R;
      before = p.rl_by_batch ? p.request_length[b] : p.request_length[req_ok ? req : 0];
#pragma unroll
      for (int c = 0; c < kPer; ++c) lse_full[c] = p.lse_full[grow_c[c] * Hq + hkv * G + min(hg0 + th[c], G - 1)];
    }
    // Fused form: the task's pre-RoPE query rows (copied into the ring with
    // the q_post NaN marker) and the full state's o rows (into s_of for the
    // epilogue) -- 16 kTask (row, head) pairs x 16 parts of 16 bytes, kTask
    // rounds of one part per thread -- move with the K/V stream, so that this traffic
    // overlaps the compute-bound key blocks instead of adding an HBM-bound
    // load round after them (every workgroup runs its task in step with the
    // others).  A round's loads go out behind a block's K/V loads; its query
    // part is stored when the next block is staged, and its o part is copied
    // straight into LDS (global_load_lds_dwordx4: no registers; waited for at
    // the next block's staging and barrier).  Round k, thread t: pair 16 k +
    // t / 16, part t % 16.
    constexpr int kCq = kTask;
    const int cq_part = tid & 15;
    const bool cq_req = kFused && req >= 0 && req < p.R;
    int cq = 0;               // rounds issued (uniform)
    bool cq_pending = false;  // round cq - 1 loaded, its query part not yet stored
    uint4 cq_src = make_uint4(0, 0, 0, 0);
    auto cq_issue = [&](int k) {
      const int e = 16 * k + (tid >> 4);
      const int r = min(e / kHeads, nrows - 1);  // (rows past the block: a valid address, not stored)
      const int64_t at = ((static_cast<int64_t>(s_qo[b]) + r_local + r) * Hq + hkv * G + min(hg0 + e % kHeads, G - 1)) *
                             kHeadDim + 8 * cq_part;
      cq_src = *reinterpret_cast<const uint4*>(p.src_q + at);
      uint4* run = &s_of[(16 * k + 4 * wave) * 16 + (16 * k + 4 * wave) / 4];  // the wave's four pairs
      __builtin_amdgcn_global_load_lds(static_cast<const void*>(p.o_full + at),
                                       (__attribute__((address_space(3))) void*)(run), 16, 0, 0);
    };
    auto cq_store = [&](int k) {
      const int e = 16 * k + (tid >> 4);
      const int r = e / kHeads, h = hg0 + e % kHeads;
      if (cq_req && r < nrows && h < G) {
        const int slot = static_cast<int>((static_cast<int64_t>(max(before, 0)) + r_local + r) % p.M);
        const int64_t at = ((static_cast<int64_t>(req) * p.M + slot) * Hq + hkv * G + h) * kHeadDim + 8 * cq_part;
        *reinterpret_cast<uint4*>(p.q_cache + at) = cq_src;
        if (p.q_post_cache != nullptr)
          *reinterpret_cast<uint4*>(p.q_post_cache + at) = make_uint4(0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u);
      }
    };

    // Q rows of the wave's tiles (B operands): lane (quad, col) holds
    // Q[row][8 (4s + quad) .. +8].  A lane past the task's rows reads its
    // first row and an absent head the group's last head (valid data, never
    // zeroed): such a lane's results are never stored, and each column keeps
    // its own softmax state.  With no select on the loaded values no wait
    // follows the loads: the Q rows and the first entries are one round.
    uint4 qreg[kPer][4];
#pragma unroll
    for (int c = 0; c < kPer; ++c) {
      const int h = hkv * G + min(hg0 + th[c], G - 1);
      const uint16_t* qp = p.q + (grow_c[c] * Hq + h) * kHeadDim;
#pragma unroll
      for (int s = 0; s < 4; ++s) qreg[c][s] = *reinterpret_cast<const uint4*>(qp + 8 * (4 * s + quad));
    }

    // l[c]: the softmax row sums.  Plain form: the lane's fp32 partial sums
    // in l[c][0] (reduced over the column's four lanes at the end).  Fused
    // form: accumulated by MFMAs with an all-ones A operand over P = hi + lo
    // (every element of the lane's l[c] then holds its column's sum), off the
    // VALU; the plain form cannot do that, since its P is bf16 hi alone and
    // the sum of that is ~2^-9 off per key, beyond what its lse output allows.
    // vt[c]: the scaled score past which m[c] moves (-inf: none seen yet).
    float m[kPer], vt[kPer];
    f32x4_t acc[kPer][8], l[kPer];
#pragma unroll
    for (int c = 0; c < kPer; ++c) {
      m[c] = kNegBig;
      vt[c] = -INFINITY;
      l[c] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) acc[c][dt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }

    const char* kbase = reinterpret_cast<const char*>(p.k + static_cast<int64_t>(hkv) * kHeadDim + ld_chunk * 8);
    const int64_t v_minus_k = reinterpret_cast<const char*>(p.v) - reinterpret_cast<const char*>(p.k);
    // the loader's K/V chunks of the block in flight (ok: bit i set if key i
    // has a row) and the raw indices of the block after it
    uint32_t ok = 0;
    int rn[kLd];
    u32x4_t kq[kLd], vq[kLd];
    auto load_block = [&](int base, int end, const int (&raw)[kLd]) {
      ok = 0;
#pragma unroll
      for (int i = 0; i < kLd; ++i) {
        if (kTrim && base + 16 * i >= end) continue;  // (uniform: none of these 16 keys exists)
        const bool in = base + ld_key + 16 * i < end && static_cast<unsigned>(raw[i]) < pool_rows;
        ok |= in ? 1u << i : 0u;
        const char* at = kbase + static_cast<uint64_t>(static_cast<uint32_t>(in ? raw[i] : 0)) * row_bytes;
        kq[i] = *reinterpret_cast<const u32x4_t*>(at);
        vq[i] = *reinterpret_cast<const u32x4_t*>(at + v_minus_k);
      }
    };
    {
      // the first segment's block 0 goes in flight here, right behind the Q
      // rows (issued in the segment loop, its loads would wait for every
      // load before them: the loop's entry joins the counts)
      const int hi_first = min(seg_first == 0 ? min(p.F, max(pos_last - wl, 0)) : pos_last + 1, key_hi);
      if (hi_first > lo_first) {
        load_block(lo_first, hi_first, pre_raw[0]);
#pragma unroll
        for (int i = 0; i < kLd; ++i) rn[i] = pre_raw[1][i];
      }
    }
    // segment 0: the front sink [0, min(F, w_lo)) of each row (fused form,
    // sink_mode 1); segment 1: the window [w_lo, pos]
    for (int seg = seg_first; seg < 2; ++seg) {
      const int seg_lo = seg == 0 ? 0 : max(wl < 0 ? 0 : max(pos0 - wl, 0), key_lo);
      const int seg_hi = min(seg == 0 ? min(p.F, max(pos_last - wl, 0)) : pos_last + 1, key_hi);
      const int nblk = seg_hi > seg_lo ? ceil_div(seg_hi - seg_lo, kBlk) : 0;
      // keys every row of the wave attends to, and keys any of them does
      const int all_lo = seg == 0 ? 0 : wlo_l, all_hi = seg == 0 ? min(p.F, wlo_f) : pos0 + rf + 1;
      const int any_lo = seg == 0 ? 0 : wlo_f, any_hi = seg == 0 ? min(p.F, wlo_l) : pos0 + rl + 1;
      if (seg != seg_first && nblk > 0) {  // (the first segment's block 0 is in flight)
        int raw[kLd];
#pragma unroll
        for (int i = 0; i < kLd; ++i) raw[i] = index_at(seg_lo + ld_key + 16 * i);
        load_block(seg_lo, seg_hi, raw);
#pragma unroll
        for (int i = 0; i < kLd; ++i) rn[i] = index_at(seg_lo + kBlk + ld_key + 16 * i);
      }
      for (int blk_i = 0; blk_i < nblk; ++blk_i) {
        const int buf = blk_i & 1;
        const int base = seg_lo + blk_i * kBlk;
        // stage the block: K and V rows (V of masked keys zeroed: P is 0 there, V may be NaN)
        {
          const bool all_ok = __all(ok == (1u << kLd) - 1u);
          if (!all_ok) {
#pragma unroll
            for (int i = 0; i < kLd; ++i) {
              const uint32_t z = (ok >> i) & 1 ? 0xffffffffu : 0u;
              vq[i] &= u32x4_t{z, z, z, z};
            }
          }
#pragma unroll
          for (int i = 0; i < kLd; ++i) {
            ld_k[buf * (kBlk * kKRow) + 16 * i * kKRow] = kq[i];
            ld_v[buf * (kBlk * kVRow) + 16 * i * kVRow] = vq[i];
          }
          if (kFused && cq_pending) {
            cq_store(cq - 1);
            cq_pending = false;
          }
          uint32_t bad[2] = {0, 0};  // lanes 16 r: key 16 i + 4 wave + r, bit 16 (i & 1) + 4 wave + r of word i / 2
          if (!all_ok) {
#pragma unroll
            for (int i = 0; i < kLd; ++i) {
              const uint64_t no = __ballot(((ok >> i) & 1) == 0);
#pragma unroll
              for (int r = 0; r < 4; ++r)
                bad[i >> 1] |= static_cast<uint32_t>((no >> (16 * r)) & 1) << (16 * (i & 1) + 4 * wave + r);
            }
          }
          if (lane == 0) {
#pragma unroll
            for (int h = 0; h < kSub; ++h) s_bad[buf][wave * kSub + h] = bad[h];
          }
        }
        __syncthreads();  // the block is visible; every wave is done with the block before last (same buffer)
        // the next block in flight while this one is computed
        if (blk_i + 1 < nblk) {
          load_block(base + kBlk, seg_hi, rn);
#pragma unroll
          for (int i = 0; i < kLd; ++i) rn[i] = index_at(base + 2 * kBlk + ld_key + 16 * i);  // (clamped)
        }
        if (kFused && cq < kCq) {
          cq_issue(cq);
          ++cq;
          cq_pending = true;
        }
        if (!live) continue;
        // sub-blocks of 32 keys that any of the wave's rows attends to
        const int s_lo = (any_lo - base) >> 5, s_hi = min(seg_hi, any_hi) - base;  // (s_lo: arithmetic shift)
#pragma unroll
        for (int sub = 0; sub < kSub; ++sub) {
          if (sub < s_lo || 32 * sub >= s_hi) continue;
          const int kb = base + 32 * sub;
          const int kt = buf * (kBlk * kKRow) + sub * (32 * kKRow);
          const uint16_t* vtile = rd_v + (buf * (kBlk * kVRow) + sub * (32 * kVRow)) * 8;
          uint32_t bad = 0;
#pragma unroll
          for (int w = 0; w < kWaves; ++w) bad |= s_bad[buf][w * kSub + sub];
          bad = __builtin_amdgcn_readfirstlane(bad);
          uint4 ka[2][4];
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int s = 0; s < 4; ++s) ka[t][s] = rd_k[s][kt + 16 * t * kKRow];
          bf16x8_t va[8];
#pragma unroll
          for (int dt = 0; dt < 8; ++dt)
            va[dt] = __builtin_shufflevector(lds_read_tr16(vtile + 16 * dt), lds_read_tr16(vtile + 16 * kVRow * 8 + 16 * dt),
                                             0, 1, 2, 3, 4, 5, 6, 7);
          // raw scores, the four accumulation chains interleaved (a tile
          // without rows is computed but never stored)
          f32x4_t c4[kPer][2];
#pragma unroll
          for (int c = 0; c < kPer; ++c)
#pragma unroll
            for (int t = 0; t < 2; ++t) c4[c][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
#pragma unroll
              for (int c = 0; c < kPer; ++c)
                c4[c][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(ka[t][s]), as_bf16x8(qreg[c][s]), c4[c][t], 0, 0, 0);
            }
          // keys inside every row's range, all present, need no masks
          if (kb < all_lo || kb + 32 > all_hi || bad != 0) {
#pragma unroll
            for (int c = 0; c < kPer; ++c) {
              // the row's keys [r_lo, r_hi) of the 32 as a bit mask: with two
              // comparisons per key instead, a short window's two masked
              // blocks cost a task 0.4 us
              const int r_lo = seg == 0 ? 0 : wlo[c], r_hi = seg == 0 ? min(p.F, wlo[c]) : pos0 + row[c] + 1;
              const int lo_k = min(max(r_lo - kb, 0), 32), hi_k = min(max(min(r_hi, seg_hi) - kb, 0), 32);
              const uint64_t range = ((1ull << hi_k) - 1) & ~((1ull << lo_k) - 1);
              const uint32_t keep = (static_cast<uint32_t>(range) & ~bad) >> (4 * quad);
#pragma unroll
              for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) c4[c][t][r] = (keep >> (16 * t + r)) & 1 ? c4[c][t][r] : -INFINITY;
            }
          }
          // lazy move of the reference point: p <= 2^8 stays exact in fp32.
          // The vote runs on each lane's own maximum (the four lanes of a
          // column share m[c], so any lane exceeding it is the column's
          // maximum exceeding it): the reduction over them is only needed
          // when the point moves.  The first key a column sees moves it (acc
          // and l are still zero, and the rescale by 2^(kNegBig - m_new) = 0
          // leaves them zero).  The softmax scale is applied inside exp2:
          // m[c] is a raw score, p = 2^(q_scale (s - m)).
          float bmax[kPer];
          bool past = false;
#pragma unroll
          for (int c = 0; c < kPer; ++c) {
            const float sv[8] = {c4[c][0][0], c4[c][0][1], c4[c][0][2], c4[c][0][3],
                                 c4[c][1][0], c4[c][1][1], c4[c][1][2], c4[c][1][3]};
            bmax[c] = max8_nonan(sv);
            past = past || bmax[c] * p.q_scale > vt[c];
          }
          if (__any(past)) {
#pragma unroll
            for (int c = 0; c < kPer; ++c) {
              const float bm = quad_max(bmax[c]);
              const float m_new = max3_nonan(m[c], bm, bm);
              const float alpha = fast_exp2((m[c] - m_new) * p.q_scale);
              m[c] = m_new;
              vt[c] = m_new > kNegBig ? m_new * p.q_scale + 8.0f : -INFINITY;
              if (kFused) l[c] *= alpha;
              else l[c][0] *= alpha;
#pragma unroll
              for (int dt = 0; dt < 8; ++dt) acc[c][dt] *= alpha;
            }
          }
          bf16x8_t pb[kPer], pl[kPer];
#pragma unroll
          for (int c = 0; c < kPer; ++c) {
            const float mo = -m[c] * p.q_scale;
            float psum = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float pe = fast_exp2(fmaf(c4[c][e >> 2][e & 3], p.q_scale, mo));
              if (!kFused) psum = e == 0 ? pe : psum + pe;  // (0 + pe = pe: no add)
              pb[c][e] = static_cast<__bf16>(pe);
              // The fused form also feeds the bf16 rounding residual of P
              // through a second MFMA (P = hi + lo, ~16 significant bits): the
              // downdate divides the window's contribution by the prefix's
              // share of the softmax mass, which amplifies any error of the
              // window state.
              if (kFused) pl[c][e] = static_cast<__bf16>(pe - static_cast<float>(pb[c][e]));
            }
            if (!kFused) l[c][0] += psum;
          }
          // O^T += V^T P^T (fused form: l += 1^T P^T as well)
          if (kFused) {
            const bf16x8_t ones = as_bf16x8(make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));
#pragma unroll
            for (int c = 0; c < kPer; ++c) {
              l[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[c], l[c], 0, 0, 0);
              l[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pl[c], l[c], 0, 0, 0);
            }
          }
#pragma unroll
          for (int dt = 0; dt < 8; ++dt)
#pragma unroll
            for (int c = 0; c < kPer; ++c) {
              acc[c][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[dt], pb[c], acc[c][dt], 0, 0, 0);
              if (kFused) acc[c][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[dt], pl[c], acc[c][dt], 0, 0, 0);
            }
        }
      }
      if (seg == 0) __syncthreads();  // the sink's last tiles are read before the window stages into them
    }
    if (kFused) {  // the rounds the blocks did not carry; then s_of is complete for every wave
      if (cq_pending) cq_store(cq - 1);
      for (; cq < kCq; ++cq) {
        cq_issue(cq);
        cq_store(cq);
      }
      __syncthreads();
    }
    if (!live) continue;

    if (kMode == kSplit && chunk < kNoChunk) {
      // the piece's unnormalised state: O^T accumulators as the lanes hold
      // them, and per column its reference point (log2 units) and sum
#pragma unroll
      for (int c = 0; c < kPer; ++c) {
        const int64_t tile = static_cast<int64_t>(t) * kTask + kPer * wave + c;
        const float lt = quad_sum(l[c][0]);
        f32x4_t* po = reinterpret_cast<f32x4_t*>(p.part_o) + tile * 8 * 64 + lane;
        if (!row_ok[c]) continue;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) po[dt * 64] = acc[c][dt];
        if (quad == 0) {
          p.part_ml[(tile * 16 + col) * 2] = m[c] * p.q_scale;
          p.part_ml[(tile * 16 + col) * 2 + 1] = lt;
        }
      }
      continue;
    }
    if (!kFused) {
#pragma unroll
      for (int c = 0; c < kPer; ++c) {
        const float lt = quad_sum(l[c][0]);
        if (!row_ok[c]) continue;
        const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
        const int64_t at = grow_c[c] * Hq + hkv * G + hg0 + th[c];
        uint16_t* op = p.out + at * kHeadDim + 4 * quad;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
          uint2 w;
          w.x = pack2_bf16(acc[c][dt][0] * inv, acc[c][dt][1] * inv);
          w.y = pack2_bf16(acc[c][dt][2] * inv, acc[c][dt][3] * inv);
          *reinterpret_cast<uint2*>(op + 16 * dt) = w;
        }
        if (quad == 0) p.out_lse[at] = lt > 0.0f ? (m[c] * p.q_scale + fast_log2(lt)) * kLn2 : -INFINITY;
      }
      continue;
    }

    // ---- fused: downdate the full state, store the ring row ----
    if (req < 0 || req >= p.R) continue;
    if (before < 0) before = 0;
    const uint2* of2 = reinterpret_cast<const uint2*>(s_of);
#pragma unroll
    for (int c = 0; c < kPer; ++c) {
      if (!row_ok[c]) continue;
      const int local = r_local + row[c];  // row index within the request
      const int slot = static_cast<int>((static_cast<int64_t>(before) + local) % p.M);
      const int64_t at = (static_cast<int64_t>(req) * p.M + slot) * Hq + hkv * G + hg0 + th[c];
      const bool empty = pos0 + row[c] + 1 - p.S <= (sink ? p.F : 0);  // nothing left after the downdate
      const float lt = l[c][0];
      const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
      const float lse_w = lt > 0.0f ? (m[c] * p.q_scale + fast_log2(lt)) * kLn2 : -INFINITY;
      Downdate d;
      if (empty) {
        d.lse = -INFINITY;
        d.t = 0.0f;
        d.scale = 0.0f;
      } else {
        d = downdate_control(lse_full[c], lse_w);
      }
      // the full state's o of the lane's row, dims 16 dt + 4 quad .. + 3, from s_of
      const int e = row[c] * kHeads + th[c];
      const uint2* of = of2 + 2 * (16 * e + (e >> 2)) + quad;
      uint16_t* ap = p.attn_cache + at * kHeadDim + 4 * quad;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        const uint2 f = of[4 * dt];
        const float fo[4] = {bf16_lo(f.x), bf16_hi(f.x), bf16_lo(f.y), bf16_hi(f.y)};
        float r[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = empty ? 0.0f : (fo[i] - d.t * (acc[c][dt][i] * inv)) * d.scale;
        uint2 w;
        w.x = pack2_bf16(r[0], r[1]);
        w.y = pack2_bf16(r[2], r[3]);
        *reinterpret_cast<uint2*>(ap + 16 * dt) = w;
      }
      if (quad == 0) p.lse_cache[at] = (p.sink_mode == 0 && p.F > 0) ? -INFINITY : d.lse;
      // (the pre-RoPE query row and the NaN marker of the unknown post-RoPE
      // row, PREFILL:251-262, went into the ring with the key blocks)
    }
  }
}

// Split form, second kernel: the states of a row block's pieces combined into
// out and out_lse.  One workgroup per (row block, head chunk, column tile);
// wave w sums the 16-dim tiles 2w, 2w + 1, lane for lane as window_kernel left
// them, each piece weighted by 2^(m - max m), eight pieces' loads in flight (a
// pass for the maxima first, one load at a time, took 70 of 206 us at one row
// over 127K keys).  The workgroups past the batch's row blocks return.
template <int RT>
__global__ void __launch_bounds__(256) window_combine_kernel(WindowParams p) {
  constexpr int kHeads = kTiles / RT;
  constexpr int kRowsT = 16 * RT;
  constexpr int kBatch = 8;
  extern __shared__ int s_dyn[];
  int* s_boff = s_dyn;               // [B + 1] pieces before a request
  int* s_rows = s_dyn + (p.B + 1);   // [B + 1] row blocks before it
  __shared__ int s_part[kWaves];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, quad = lane >> 4, col = lane & 15;
  const int chunk = plan_pieces<kSplit, kRowsT>(p, s_boff, s_part);
  if (chunk >= kNoChunk) return;  // window_kernel wrote the results
  const int Hq = p.Hq, Hkv = p.Hkv, G = Hq / Hkv, B = p.B;
  {
    const int per = ceil_div(B, 256), b0 = min(B, tid * per), b1 = min(B, b0 + per);
    int sum = 0, total;
    for (int i = b0; i < b1; ++i) sum += ceil_div(request_rows<kSplit>(p, i), kRowsT);
    int acc = scan256(sum, s_part, total);
    for (int i = b0; i < b1; ++i) {
      s_rows[i] = acc;
      acc += ceil_div(request_rows<kSplit>(p, i), kRowsT);
    }
    if (tid == 0) s_rows[B] = total;
    __syncthreads();
  }
  const int nchunks = ceil_div(G, kHeads);
  const int per_piece = Hkv * nchunks;
  const int tile = blockIdx.x % kTiles;
  const int item = blockIdx.x / kTiles;
  const int hc = item % per_piece;
  const int rb = item / per_piece;  // row block, numbered over the batch
  if (rb >= s_rows[B]) return;
  const int b = request_of(s_rows, B, rb);
  const int blk = rb - s_rows[b], nb = s_rows[b + 1] - s_rows[b];
  const int q0 = p.qo_indptr[b];
  const int len = p.qo_indptr[b + 1] - q0;
  const int kvlen = p.kv_indptr[b + 1] - p.kv_indptr[b];
  const int r_local = kRowsT * blk;
  const int nrows = min(kRowsT, len - r_local);
  const int pos_last = kvlen - len + r_local + nrows - 1;
  const int hkv = hc / nchunks;
  const int h = kHeads * (hc - hkv * nchunks) + tile / RT;  // head in the group
  const int r0 = 16 * (tile % RT);
  if (h >= G || r0 + col >= nrows) return;  // (window_kernel stored the lanes of whole rows only)
  const int n = __builtin_amdgcn_readfirstlane(ceil_div(pos_last + 1, chunk));  // pieces with keys of these rows
  auto slot = [&](int ch) {  // tile slot of chunk ch (window_kernel's task order)
    return (static_cast<int64_t>(s_boff[b] + ch * nb + blk) * per_piece + hc) * kTiles + tile;
  };
  float mx = kNegBig, lt = 0.0f;
  f32x4_t o[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
  for (int c0 = 0; c0 < n; c0 += kBatch) {
    f32x4_t a[kBatch][2];
    float w[kBatch], l[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int64_t t = slot(min(c0 + u, n - 1));
      const f32x4_t* po = reinterpret_cast<const f32x4_t*>(p.part_o) + t * 8 * 64 + (2 * wave) * 64 + lane;
      a[u][0] = po[0];
      a[u][1] = po[64];
      w[u] = p.part_ml[(t * 16 + col) * 2];
      l[u] = p.part_ml[(t * 16 + col) * 2 + 1];
    }
    float m_new = mx;
#pragma unroll
    for (int u = 0; u < kBatch; ++u) m_new = fmaxf(m_new, w[u]);
    const float keep = fast_exp2(mx - m_new);
    mx = m_new;
    lt *= keep;
    o[0] *= keep;
    o[1] *= keep;
    auto add = [&](int u) {
      const float f = fast_exp2(w[u] - mx);
      lt += f * l[u];
      o[0] += f * a[u][0];
      o[1] += f * a[u][1];
    };
    if (c0 + kBatch <= n) {
#pragma unroll
      for (int u = 0; u < kBatch; ++u) add(u);
    } else {  // (uniform) not the copies of the last piece, whose infinities a weight of 0 would keep
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
        if (c0 + u < n) add(u);
    }
  }
  const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
  const int64_t at = (static_cast<int64_t>(q0) + r_local + r0 + col) * Hq + hkv * G + h;
  uint16_t* op = p.out + at * kHeadDim + 4 * quad;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint2 v;
    v.x = pack2_bf16(o[i][0] * inv, o[i][1] * inv);
    v.y = pack2_bf16(o[i][2] * inv, o[i][3] * inv);
    *reinterpret_cast<uint2*>(op + 16 * (2 * wave + i)) = v;
  }
  if (quad == 0 && wave == 0) p.out_lse[at] = lt > 0.0f ? (mx + fast_log2(lt)) * kLn2 : -INFINITY;
}

// request_length[req] += len (indexed-by-request form, after the ring rows
// were addressed with the old value) for every request the window kernel
// wrote: the validity test of request_rows, a request it skipped is not bumped.
__global__ void bump_kernel(int32_t* request_length, const int32_t* req_ids, const int32_t* qo_indptr,
                            const int32_t* kv_indptr, int64_t total_q, int64_t kv_len_total, int B, int R) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  const int req = req_ids[b];
  const int q0 = qo_indptr[b], q1 = qo_indptr[b + 1];
  const int k0 = kv_indptr[b], k1 = kv_indptr[b + 1];
  const int len = q1 - q0;
  const bool ok = q0 >= 0 && q1 <= total_q && k0 >= 0 && k1 <= kv_len_total && len > 0 && k1 - k0 >= len;
  if (!ok || req < 0 || req >= R) return;
  atomicAdd(&request_length[req], len);
}

// Workgroups for `tasks` wave-sized units of work (4 per workgroup), at most
// as many as are resident at once (`kernel`'s occupancy on every CU), since
// the kernels loop over their tasks.
int grid_for(int64_t tasks, const void* kernel, size_t dyn_lds = 0) {
  int dev = 0, cus = 256, per_cu = 2;
  if (hipGetDevice(&dev) == hipSuccess) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0) cus = v;
    int occ = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, 256, dyn_lds) == hipSuccess && occ > 0) per_cu = occ;
  }
  const int64_t wgs = (tasks + 3) / 4;
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(wgs, static_cast<int64_t>(cus) * per_cu)));
}

// Row tiles of a task for a GQA group (window_kernel): 8 / RT heads cover it
// without absent heads up to the next power of two.
int row_tiles(int G) { return G > 4 ? 1 : (G > 2 ? 2 : (G > 1 ? 4 : 8)); }

int device_cus() {
  int dev = 0, v = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0)
    return 256;
  return v;
}

// Tasks that `rows` query rows of B requests of about equal length make in
// blocks of 16 rt rows and chunks of `heads` heads.
int64_t expected_tasks(int64_t rows, int B, int Hq, int Hkv, int rt, int heads) {
  const int64_t per_request = (rows + B - 1) / B;
  return B * ((per_request + 16 * rt - 1) / (16 * rt)) * Hkv * ceil_div(Hq / Hkv, heads);
}

// Split over keys (causal attention over whole prefixes, window_left < 0):
// pieces of the batch a split call plans for, or 0 where the row blocks alone
// give the GPU enough work.  A task per (row block, head chunk) streams its
// keys in one chain, so a batch with few of them leaves CUs idle; its keys
// are then cut so that there are up to two rounds of the resident workgroups
// (2 per CU) more tasks than row blocks.  Kept suffixes of long prompts are
// that case.  Unsplit, half a round, one, 1.5, two and three rounds of pieces
// took (us): 512 rows over 32K keys, 4 heads per group, 681, 430, 317, 329, 322
// and 331; 8 requests of 16-32 rows over 8K-64K keys, 8 heads per group, 1302,
// 253, 231, 203, 187 and 199; one row over 127K keys, 4 KV heads, 2768, 84, 80,
// 93, 104 and 124 (a piece's state is 64 KiB written and read once): one round
// leaves a ragged batch nothing to level it with.  From 3/4 of a round of tasks
// on the cut costs what it levels out (32 requests x 32 rows over 4K keys, 8
// heads per group: 129 unsplit, 141 split).
constexpr int64_t kSplitKeys = 1024;
struct Split {
  int64_t blocks = 0;  // bound on the batch's row blocks
  int pieces = 0;      // most (row block, key chunk) pieces; 0: no split
  size_t o_bytes = 0, bytes = 0;
};

Split split_plan(int B, int Hq, int Hkv, int64_t total_q, int64_t kv_len, int window_left) {
  Split sp;
  if (window_left >= 0 || B <= 0 || total_q <= 0 || Hkv <= 0 || Hq < Hkv) return sp;
  const int G = Hq / Hkv, rt = row_tiles(G);
  const int64_t per_piece = static_cast<int64_t>(Hkv) * ceil_div(G, kTiles / rt);
  // (a block holds at least one row, and every request but the first block of
  // each fills its blocks)
  sp.blocks = std::min<int64_t>(total_q, (total_q + 16 * rt - 1) / (16 * rt) + B);
  const int64_t grid = 2 * static_cast<int64_t>(device_cus());
  if (4 * sp.blocks * per_piece >= 3 * grid) return sp;
  if (kv_len < kSplitKeys * static_cast<int64_t>(B)) return sp;
  const int64_t pieces = sp.blocks + (2 * grid + per_piece - 1) / per_piece;
  sp.pieces = static_cast<int>(pieces);
  sp.o_bytes = static_cast<size_t>(pieces * per_piece) * kTiles * 8 * 64 * 16;
  sp.bytes = sp.o_bytes + static_cast<size_t>(pieces * per_piece) * kTiles * 16 * 2 * sizeof(float);
  return sp;
}

// Whether a call that split_plan allows is cut: the states and the second
// launch cost it 10-30 us, the more the more tasks it has (each in up to 5
// pieces already at 1024 keys), and what it saves is the part of a task's
// chain that idle CUs take over.  Keys per request from which it gains, in us
// unsplit / split (1-row requests over 4 or 8 KV heads): 96 tasks, 1100 keys
// 30.8 / 29.3; 128, 1100 keys 30 / 35, 1500 38 / 36; 160, 2000 keys 48 / 52, 3000
// 70 / 67; 192, 3000 keys 88 / 92, 4000 129 / 123; 256, 3000 keys 109 / 112, 4000
// 141 / 141, 8000 277 / 246; 1000 rows of one request (252), 3000 keys 84 / 86, 4000
// 110 / 104.
bool split_pays(const WindowParams& p) {
  const int64_t cus = device_cus();
  const int rt = row_tiles(p.Hq / p.Hkv);
  const int64_t tasks = expected_tasks(p.total_q, p.B, p.Hq, p.Hkv, rt, kTiles / rt);
  const int64_t line = (tasks - 68 * cus / 256) * 6400 / cus;  // 25 keys per task past 68 of 256 CUs
  return p.kv_len_total / p.B >= (tasks <= cus ? std::min<int64_t>(line, 4000) : line);
}

template <int RT>
void launch_split(const WindowParams& p, const Split& sp, hipStream_t stream) {
  const int64_t per_piece = static_cast<int64_t>(p.Hkv) * ceil_div(p.Hq / p.Hkv, kTiles / RT);
  const size_t lds = sizeof(int) * (static_cast<size_t>(p.B) + 1);  // of one array over the requests
  const void* kern = reinterpret_cast<const void*>(&window_kernel<RT, 2, kSplit, 64>);
  hipLaunchKernelGGL((window_kernel<RT, 2, kSplit, 64>), dim3(grid_for(4 * sp.pieces * per_piece, kern, 3 * lds)), dim3(256),
                     3 * lds, stream, p);
  hipLaunchKernelGGL((window_combine_kernel<RT>), dim3(static_cast<unsigned>(sp.blocks * per_piece * kTiles)), dim3(256),
                     2 * lds, stream, p);
}

template <int RT, int kPer, int kMode, int kBlk>
void launch_window_as(const WindowParams& p, int64_t rows, hipStream_t stream) {
  const int G = p.Hq / p.Hkv;
  const size_t lds = 3 * sizeof(int) * (static_cast<size_t>(p.B) + 1);
  const int64_t blocks = (rows + 16 * RT - 1) / (16 * RT) + p.B;  // (a bound)
  const void* kern = reinterpret_cast<const void*>(&window_kernel<RT, kPer, kMode, kBlk>);
  const int64_t tasks = blocks * p.Hkv * ceil_div(G, kWaves * kPer / RT);
  hipLaunchKernelGGL((window_kernel<RT, kPer, kMode, kBlk>), dim3(grid_for(4 * tasks, kern, lds)), dim3(256), lds, stream, p);
}

// Narrow tasks (16 rows x 4 heads, one column tile per wave) or wide ones
// (8 tiles, two per wave).  A narrow task's chain over its keys takes 25 us
// per 1000 keys where a wide one's takes 31, and more of them run side by
// side (three workgroups per CU); a wide task does twice the columns or more
// with the same reads.  So narrow tasks serve the calls that leave the GPU
// partly idle, where only the chain counts: as many narrow tasks as CUs, or
// two per CU where wide tasks would fill at most half of them (a quarter with
// a window: its wide chains are hardly longer).  And those whose requests
// have too few rows for a wide task's rows, at any batch.  Times in us,
// narrow / wide, 1000 keys or a window of 256, 4 heads per group but as said:
//   64 rows 27 / 33; 64 rows of 8 heads 28 / 33, of 1 head 26 / 31;
//   8 x 64 rows over 1500 keys (256 narrow) 40 / 49; 512 rows, window, 13 / 16;
//   64 x 4 rows (512, as many wide) 29 / 36; 1100 x 16 rows, 300 keys, 184 / 258;
//   16 x 64 rows (512, 256 wide) 38 / 36; window 19.8 / 19.2; 1 head 29 / 32
//   (128 wide) and 16.6 / 14.4; 4 x 256 rows of 1 head, window (512, 64 wide),
//   15.1 / 17.0; 64 x 64 rows 83 / 68.
// Fused form (two workgroups per CU either way): 8 x 100 rows (448 narrow) 19.4 /
// 22.6; 32 x 40 rows (768, 512 wide) 27.5 / 29.2, of 2 heads (256 wide) 25.9 /
// 23.0; 32 x 100 rows (1792) 64.7 / 63.8.
template <int kMode>
bool narrow_tasks(const WindowParams& p, int64_t rows) {
  const int64_t cus = device_cus();
  const int rt = row_tiles(p.Hq / p.Hkv);
  const int64_t narrow = expected_tasks(rows, p.B, p.Hq, p.Hkv, 1, kWaves);
  const int64_t wide = expected_tasks(rows, p.B, p.Hq, p.Hkv, rt, kTiles / rt);
  if (kMode == kRectify) return narrow <= 2 * cus || (narrow <= 3 * cus && 2 * narrow <= 3 * wide);
  return 4 * narrow <= 5 * wide || narrow <= cus ||
         (narrow <= 2 * cus && wide <= (p.window_left < 0 ? cus / 2 : cus / 4));
}

// Blocks of 32 or 64 keys for the wide tasks of 16-row blocks (plain form, 5
// or more heads per group).  64 (half of the barriers) pay where several row
// blocks share a request's keys: over whole prefixes, and with a window while
// the GPU has more than a round of tasks; and for single blocks over whole
// prefixes while it has at most one task per CU.  Elsewhere 32, whose window
// ends nearer to what it loads and which waits for fewer keys at a time.  32
// also for windows of up to 64 keys, windows over a K/V set that the caches do
// not hold (what is loaded past a window's end comes from HBM; counted as the
// index entries, at most the pool's rows), and batches whose request offsets
// leave a CU no room for two workgroups with 64.  Times in us, 64 / 32 (8 heads
// per group): 30 x 100 rows over 1500 keys 125 / 129; 8 x 200 over 200, 17.7 /
// 18.9; 1 row over 3000 keys 81 / 86; 96 requests of 1 row over 1500 keys (384
// tasks) 78 / 69; 500 x 16 rows over 300 keys 120 / 116; 16 x 64 rows, window 256,
// 19.0 / 18.0; 1100 x 16 over 300 keys 287 / 231.  N x 8192 rows, window 256, 16
// MiB of K/V each: 12, 815 / 820; 24, 1637 / 1639; 32, 2178 / 2174; 48, 3341 /
// 3285; 64, 4497 / 4367; window 64: 16, 729 / 709.
constexpr int64_t kFarBytes = 512ll << 20;  // twice the memory-side cache

bool long_blocks(const WindowParams& p, int64_t rows, size_t request_bytes) {
  const int64_t cus = device_cus();
  const int64_t tasks = expected_tasks(rows, p.B, p.Hq, p.Hkv, 1, kTiles);
  const int64_t far = std::min(p.kv_len_total, p.pool_tokens) * p.Hkv * (4 * kHeadDim);
  if (p.window_left >= 0 && (p.window_left < 64 || far > kFarBytes)) return false;
  int per_cu = 0;
  const void* kern = reinterpret_cast<const void*>(&window_kernel<1, 2, kPlain, 64>);
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, 256, request_bytes) != hipSuccess || per_cu < 2) return false;
  const bool shared = rows > 16 * static_cast<int64_t>(p.B);
  return p.window_left < 0 ? shared || tasks <= cus : shared && tasks > 2 * cus;
}

template <int RT, int kMode>
void launch_window_wide(const WindowParams& p, int64_t rows, hipStream_t stream) {
  if constexpr (kMode == kRectify) {
    launch_window_as<RT, 2, kMode, 32>(p, rows, stream);
  } else if constexpr (RT == 1) {
    if (long_blocks(p, rows, 3 * sizeof(int) * (static_cast<size_t>(p.B) + 1)))
      launch_window_as<RT, 2, kMode, 64>(p, rows, stream);
    else
      launch_window_as<RT, 2, kMode, 32>(p, rows, stream);
  } else {
    launch_window_as<RT, 2, kMode, 64>(p, rows, stream);
  }
}

// Launches the window kernel over at most `rows` query rows.
template <int kMode>
void launch_window(const WindowParams& p, int64_t rows, hipStream_t stream) {
  if (narrow_tasks<kMode>(p, rows)) return launch_window_as<1, 1, kMode, 32>(p, rows, stream);
  switch (row_tiles(p.Hq / p.Hkv)) {
    case 1: return launch_window_wide<1, kMode>(p, rows, stream);
    case 2: return launch_window_wide<2, kMode>(p, rows, stream);
    case 4: return launch_window_wide<4, kMode>(p, rows, stream);
    default: return launch_window_wide<8, kMode>(p, rows, stream);
  }
}

}  // namespace

#define REQUIRE(cond, ...) \
  do {                     \
    if (!(cond)) return mac::fail(MAC_ERR_INVALID_ARGUMENT, __VA_ARGS__); \
  } while (0)

#define HIP_OK(call)                                                                      \
  do {                                                                                    \
    hipError_t e_ = (call);                                                               \
    if (e_ != hipSuccess) return mac::fail(MAC_ERR_HIP, "%s: %s", #call, hipGetErrorString(e_)); \
  } while (0)

extern "C" int mac_update_then_downdate_bf16_inplace(const void* out1, const void* lse1, int32_t lse1_dtype,
                                                     void* out2, void* lse2, int32_t lse2_dtype, int64_t rows,
                                                     int32_t head_dim, void* stream) {
  REQUIRE(rows >= 0, "rows must be >= 0");
  REQUIRE(head_dim > 0, "head_dim must be > 0");
  REQUIRE(lse1_dtype >= MAC_DTYPE_F32 && lse1_dtype <= MAC_DTYPE_F16, "lse1 must be float32, bfloat16, or float16");
  REQUIRE(lse2_dtype >= MAC_DTYPE_F32 && lse2_dtype <= MAC_DTYPE_F16, "lse2 must be float32, bfloat16, or float16");
  if (rows == 0) return MAC_OK;
  REQUIRE(out1 && out2 && lse1 && lse2, "null pointer argument");
  if ((head_dim & 7) == 0)
    REQUIRE((reinterpret_cast<uintptr_t>(out1) & 15) == 0 && (reinterpret_cast<uintptr_t>(out2) & 15) == 0,
            "out tensors must be 16-byte aligned");
  const int64_t wgs = std::min<int64_t>((rows + 63) / 64, 65536);
  hipLaunchKernelGGL(downdate_kernel, dim3(static_cast<unsigned>(wgs)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(out1), lse1, lse1_dtype,
                     static_cast<uint16_t*>(out2), lse2, lse2_dtype, rows, head_dim);
  HIP_OK(hipGetLastError());
  return MAC_OK;
}

namespace {

// the kernels move bf16 rows with 16-byte vector accesses
bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }

int check_window_common(int B, int Hq, int Hkv, int D, int64_t total_q, int64_t pool, const void* q,
                        const void* k, const void* v, const int32_t* qo, const int32_t* kvp, const int32_t* kvi,
                        int64_t kv_len) {
  REQUIRE(D == kHeadDim, "head_dim must be 128 (got %d)", D);
  REQUIRE(Hq > 0 && Hkv > 0 && Hq % Hkv == 0, "Hq must be a positive multiple of Hkv");
  REQUIRE(B >= 0 && B <= kMaxB, "B must be in [0, %d] (got %d)", kMaxB, B);
  REQUIRE(total_q >= 0 && total_q <= INT_MAX && pool > 0, "bad total_q / pool_tokens");
  REQUIRE(total_q * Hq <= static_cast<int64_t>(INT_MAX) * 64, "total_q too large");
  REQUIRE(q && k && v && qo && kvp && kvi, "null pointer argument");
  REQUIRE(aligned16(q) && aligned16(k) && aligned16(v), "q, k and v must be 16-byte aligned");
  // the window kernel addresses a request's kv_indices with 32-bit byte offsets
  REQUIRE(kv_len >= 0 && kv_len < (int64_t{1} << 30), "kv_indices must hold fewer than 2^30 entries");
  return MAC_OK;
}

}  // namespace

namespace {

int check_window_args(const MacWindowAttentionArgs* a) {
  REQUIRE(a != nullptr, "args is NULL");
  REQUIRE(a->struct_size == sizeof(MacWindowAttentionArgs), "struct_size mismatch (%u vs %zu)", a->struct_size,
          sizeof(MacWindowAttentionArgs));
  REQUIRE(a->abi_version == MAC_ABI_VERSION, "abi_version mismatch");
  if (int rc = check_window_common(a->B, a->Hq, a->Hkv, a->D, a->total_q, a->pool_tokens, a->q, a->k_buffer,
                                   a->v_buffer, a->qo_indptr, a->kv_indptr, a->kv_indices, a->kv_indices_len))
    return rc;
  REQUIRE(a->out && a->out_lse, "out / out_lse must not be NULL");
  REQUIRE(aligned16(a->out), "out must be 16-byte aligned");
  return MAC_OK;
}

}  // namespace

extern "C" int64_t mac_prefill_window_attention_workspace(int32_t B, int32_t Hq, int32_t Hkv, int64_t total_q,
                                                          int64_t kv_indices_len, int32_t window_left) {
  return static_cast<int64_t>(split_plan(B, Hq, Hkv, total_q, kv_indices_len, window_left).bytes);
}

extern "C" int mac_prefill_window_attention_ws_bf16(const MacWindowAttentionArgs* a, void* workspace,
                                                    int64_t workspace_bytes, void* stream) {
  if (int rc = check_window_args(a)) return rc;
  REQUIRE(workspace_bytes >= 0 && aligned16(workspace), "workspace must be 16-byte aligned");
  if (a->B == 0 || a->total_q == 0) return MAC_OK;
  WindowParams p{};
  p.q = static_cast<const uint16_t*>(a->q);
  p.k = static_cast<const uint16_t*>(a->k_buffer);
  p.v = static_cast<const uint16_t*>(a->v_buffer);
  p.qo_indptr = a->qo_indptr;
  p.kv_indptr = a->kv_indptr;
  p.kv_indices = a->kv_indices;
  p.out = static_cast<uint16_t*>(a->out);
  p.out_lse = a->out_lse;
  p.pool_tokens = a->pool_tokens;
  p.total_q = a->total_q;
  p.kv_len_total = a->kv_indices_len;
  p.B = a->B;
  p.Hq = a->Hq;
  p.Hkv = a->Hkv;
  p.M = 1;
  p.window_left = a->window_left;
  p.q_scale = static_cast<float>(a->sm_scale * 1.4426950408889634);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const Split sp = workspace != nullptr
                       ? split_plan(a->B, a->Hq, a->Hkv, a->total_q, a->kv_indices_len, a->window_left)
                       : Split{};
  if (sp.pieces > 0 && static_cast<int64_t>(sp.bytes) <= workspace_bytes && split_pays(p)) {
    p.part_o = static_cast<float*>(workspace);
    p.part_ml = reinterpret_cast<float*>(static_cast<char*>(workspace) + sp.o_bytes);
    p.max_pieces = sp.pieces;
    p.max_blocks = static_cast<int>(sp.blocks);
    switch (row_tiles(p.Hq / p.Hkv)) {
      case 1: launch_split<1>(p, sp, s); break;
      case 2: launch_split<2>(p, sp, s); break;
      case 4: launch_split<4>(p, sp, s); break;
      default: launch_split<8>(p, sp, s); break;
    }
  } else {
    launch_window<kPlain>(p, a->total_q, s);
  }
  HIP_OK(hipGetLastError());
  return MAC_OK;
}

extern "C" int mac_prefill_window_attention_bf16(const MacWindowAttentionArgs* a, void* stream) {
  return mac_prefill_window_attention_ws_bf16(a, nullptr, 0, stream);
}

extern "C" int mac_prefill_rectify_update_cache_bf16(const MacRectifyArgs* a, void* stream) {
  REQUIRE(a != nullptr, "args is NULL");
  REQUIRE(a->struct_size == sizeof(MacRectifyArgs), "struct_size mismatch (%u vs %zu)", a->struct_size,
          sizeof(MacRectifyArgs));
  REQUIRE(a->abi_version == MAC_ABI_VERSION, "abi_version mismatch");
  if (int rc = check_window_common(a->B, a->Hq, a->Hkv, a->D, a->total_q, a->pool_tokens, a->q_post, a->k_buffer,
                                   a->v_buffer, a->qo_indptr, a->kv_indptr, a->kv_indices, a->kv_indices_len))
    return rc;
  REQUIRE(a->M > 0, "capacity (M) must be > 0");
  REQUIRE(a->R > 0, "R must be > 0");
  REQUIRE(a->semantic_pos_ahead >= 1, "semantic_pos_ahead must be >= 1 (the window is S keys)");
  REQUIRE(a->front_sink_tokens >= 0, "front_sink_tokens must be >= 0");
  REQUIRE(a->sink_mode == 0 || a->sink_mode == 1, "sink_mode must be 0 or 1");
  REQUIRE(a->request_length_len == a->R || a->request_length_len == a->B, "request_length must be [R] or [B]");
  REQUIRE(a->src_q && a->o_full && a->lse_full && a->q_cache && a->attn_cache && a->lse_cache &&
              a->request_length && a->req_ids,
          "null pointer argument");
  REQUIRE(aligned16(a->src_q) && aligned16(a->o_full) && aligned16(a->q_cache) && aligned16(a->attn_cache) &&
              (a->q_post_cache == nullptr || aligned16(a->q_post_cache)),
          "src_q, o_full, q_cache, attn_cache and q_post_cache must be 16-byte aligned");
  if (a->B == 0 || a->total_q == 0) return MAC_OK;
  WindowParams p{};
  p.q = static_cast<const uint16_t*>(a->q_post);
  p.k = static_cast<const uint16_t*>(a->k_buffer);
  p.v = static_cast<const uint16_t*>(a->v_buffer);
  p.qo_indptr = a->qo_indptr;
  p.kv_indptr = a->kv_indptr;
  p.kv_indices = a->kv_indices;
  p.src_q = static_cast<const uint16_t*>(a->src_q);
  p.o_full = static_cast<const uint16_t*>(a->o_full);
  p.lse_full = a->lse_full;
  p.q_cache = static_cast<uint16_t*>(a->q_cache);
  p.attn_cache = static_cast<uint16_t*>(a->attn_cache);
  p.lse_cache = a->lse_cache;
  p.q_post_cache = static_cast<uint16_t*>(a->q_post_cache);
  p.request_length = a->request_length;
  p.req_ids = a->req_ids;
  p.pool_tokens = a->pool_tokens;
  p.total_q = a->total_q;
  p.kv_len_total = a->kv_indices_len;
  p.B = a->B;
  p.Hq = a->Hq;
  p.Hkv = a->Hkv;
  p.R = a->R;
  p.M = a->M;
  p.S = a->semantic_pos_ahead;
  p.F = a->front_sink_tokens;
  p.sink_mode = a->sink_mode;
  // the by-batch form wins when R == B, as in mac_prefill_update_cache
  p.rl_by_batch = a->request_length_len == a->B;
  p.q_scale = static_cast<float>(a->sm_scale * 1.4426950408889634);
  const int64_t kept = std::min<int64_t>(a->total_q, static_cast<int64_t>(a->B) * a->M);
  hipStream_t s = static_cast<hipStream_t>(stream);
  launch_window<kRectify>(p, kept, s);
  HIP_OK(hipGetLastError());
  if (!p.rl_by_batch) {
    hipLaunchKernelGGL(bump_kernel, dim3((a->B + 255) / 256), dim3(256), 0, s, a->request_length, a->req_ids,
                       a->qo_indptr, a->kv_indptr, p.total_q, p.kv_len_total, a->B, a->R);
    HIP_OK(hipGetLastError());
  }
  return MAC_OK;
}
