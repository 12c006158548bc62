// Router scoring: pre-summed query tiles against the HBM-resident pooled K_r bank.
//
// score[b, c] = max over scored tokens t of (scale / Hq) * sum_h q'[b,t,h] . kr[c, h / G]
//             = max_t (scale / Hq) * Qs[b,t,:] . kr[c,:]        with Qs[b,t,g,:] = sum_{h in g} q'[b,t,h,:]
// (the mean over heads is linear, so the G query heads of one KV group are summed first).  That is
// an NT GEMM  [B*S_pad, Hkv*D] x [C, Hkv*D]^T  whose output is never written: each 32-row MFMA
// block is reduced to a column max over its scored rows in registers.  For routing the column maxima
// of a query are folded further, across the chunks of one document, and merged with atomicMax into
// doc_key[B, n_docs] (order-preserving uint32 keys): the max over a document's chunks happens in the
// scoring epilogue and no per-chunk plane exists.  msa_chunk_scores keeps the per-chunk form.
#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

#include "gather_device.h"
#include "route_internal.h"

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16_t;
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------------------------------
// Prologue: normalise (cosine mode), sum the G heads of each KV group, cast, build row masks, clear the key plane.
// One workgroup of Hkv*16 lanes per (b, padded token); lane (g, j) owns 8 contiguous d of group g.
// A row that is not scored (a masked token, or the padding of a query to a multiple of 32 rows) repeats the query's
// first scored row: a repeated row changes no maximum, so the scoring epilogues fold whole 32-row blocks without
// per-row tests.  A query without any scored token keeps rows of zeros and mask words of zero: its row blocks are
// skipped and its keys stay 0.  The workgroup of every 32nd row writes the mask word of its 32 rows (all ones or
// zero), workgroup 0 the zero words that pad the mask to whole M tiles, and all workgroups together clear the
// `clear_words` key words the scoring kernel merges into with atomicMax.
// Short queries of a batch share row blocks (RowPacking): then the word of a row block tells every row's own query, rows behind the last
// query are zero, and the scan's large tiles have a block's rows in the order of its units (unit_row).
// ------------------------------------------------------------------------------------------
// Words behind the persistent scan's tile pool: the pool's counter, on a cache line of its own, then one word per
// workgroup through which the wavefront that drew a tile tells the workgroup's others.
constexpr int kSchedCounterWords = 32;
constexpr int kSchedMaxWorkgroups = 1024;
constexpr size_t kSchedBytes = (size_t)(kSchedCounterWords + kSchedMaxWorkgroups) * sizeof(uint32_t);

// Eight fp32 values as three bf16 operands whose sum they are, each the rest rounded: up to 2^-8 and 2^-17 of the value behind the first.
// kInfinite: a first part that would round to an infinity is cut off instead, and nothing is left of an infinity; without it either leaves a NaN.
template <bool kInfinite>
__device__ __forceinline__ void split_three(const float (&x)[8], uint4 (&part)[3]) {
  uint32_t w[3][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = x[2 * i], b = x[2 * i + 1];
    w[0][i] = pack_bf16x2(a, b);
    if constexpr (kInfinite) {
      if ((w[0][i] & 0x7f80u) == 0x7f80u) w[0][i] = (w[0][i] & 0xffff0000u) | __float_as_uint(a) >> 16;
      if ((w[0][i] & 0x7f800000u) == 0x7f800000u) w[0][i] = (w[0][i] & 0xffffu) | (__float_as_uint(b) & 0xffff0000u);
    }
    const float a1 = bf16lo(w[0][i]), b1 = bf16hi(w[0][i]);
    const float ra = kInfinite && a == a1 ? 0.f : a - a1, rb = kInfinite && b == b1 ? 0.f : b - b1;
    w[1][i] = pack_bf16x2(ra, rb);
    w[2][i] = pack_bf16x2(ra - bf16lo(w[1][i]), rb - bf16hi(w[1][i]));
  }
#pragma unroll
  for (int p = 0; p < 3; ++p) part[p] = make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]);
}
// Where score_parts_kernel's operands of the queries lie: 32 rows x 16 values of K, a part each, in the order of a wavefront's lanes.
constexpr int kPartBytes = 1024, kPartStep = 3 * kPartBytes;
__device__ __forceinline__ int64_t part_at(int row, int k, int K) {
  return ((int64_t)(row >> 5) * (K / 16) + k / 16) * kPartStep + (row & 31) * 16 + (k & 8) * 64;
}

// Where the large-tile scan has row `row` of a block of four units of eight rows: unit u in rows 4 u .. 4 u + 3 of either sixteen.
__device__ __forceinline__ int unit_row(int row) { return (row & ~31) | (row & 4) << 2 | (row & 24) >> 1 | (row & 3); }

template <typename TIn, typename TOut, bool kParts = false>
__global__ void presum_queries_kernel(const TIn* __restrict__ q, const uint8_t* __restrict__ qmask, int32_t B,
                                      int32_t S, int32_t S_pad, int32_t Hq, int32_t Hkv, int32_t normalize,
                                      TOut* __restrict__ qs, uint32_t* __restrict__ row_bits, int32_t mask_words,
                                      uint32_t* __restrict__ key_plane, int64_t clear_words, uint32_t* __restrict__ sched,
                                      int32_t packed, int32_t by_units) {
  const int row = blockIdx.x;              // b * S_pad + s
  const int b = row / S_pad;
  int s = row % S_pad;
  const int G = Hq / Hkv;
  const int g = threadIdx.x >> 4, j = threadIdx.x & 15;
  const bool behind = b >= B;              // (packed: the last block's rows behind the last query)
  bool valid = !behind && s < S && (qmask == nullptr || qmask[(int64_t)b * S + s] != 0);
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < clear_words; i += (int64_t)gridDim.x * blockDim.x)
    key_plane[i] = 0u;
  const bool writes_word = (row & 31) == 0;           // rows are padded per query to a multiple of 32, or packed
  if (packed && writes_word) {
    __shared__ uint32_t scored_rows;
    if (threadIdx.x == 0) scored_rows = 0u;
    __syncthreads();
    const int tokens = (min((row + 31) / S_pad, B - 1) - b + 1) * S;      // of the block's queries, which lie side by side
    for (int i = (int)threadIdx.x; i < tokens; i += blockDim.x)
      if (qmask == nullptr || qmask[(int64_t)b * S + i] != 0) {
        const int first = (b + i / S) * S_pad - row, lo = max(first, 0), hi = min(first + S_pad, 32);
        atomicOr(&scored_rows, (hi < 32 ? (1u << hi) - 1u : 0xffffffffu) & (0xffffffffu << lo));
      }
    __syncthreads();
    if (threadIdx.x == 0) row_bits[row >> 5] = scored_rows;
  }
  if (!behind && (!valid || (writes_word && !packed))) {      // (uniform over the workgroup)
    // the query's first scored token, found by the workgroup's first wavefront
    __shared__ int first_scored;
    if (threadIdx.x < 64) {
      const int nl = min((int)blockDim.x, 64);
      int found = qmask == nullptr ? 0 : -1;
      for (int base = 0; base < S && found < 0; base += nl) {
        const int t = base + (int)threadIdx.x;
        const bool v = (int)threadIdx.x < nl && t < S && qmask[(int64_t)b * S + t] != 0;
        const uint64_t m = __ballot(v);
        if (m != 0) found = base + __builtin_ctzll(m);
      }
      if (threadIdx.x == 0) {
        first_scored = found;
        if (writes_word && !packed) row_bits[row >> 5] = found >= 0 ? 0xffffffffu : 0u;
      }
    }
    __syncthreads();
    if (!valid && first_scored >= 0) {
      s = first_scored;
      valid = true;
    }
  }
  if (blockIdx.x == 0) {
    for (int w = (int)(gridDim.x >> 5) + (int)threadIdx.x; w < mask_words; w += blockDim.x) row_bits[w] = 0u;
    if (threadIdx.x == 0) sched[0] = 0u;        // the scan's pool counter
  }
  float acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = 0.f;
  if (valid) {
    const TIn* p0 = q + (((int64_t)b * S + s) * Hq + g * G) * kHeadDim + 8 * j;
    for (int h0 = 0; h0 < G; h0 += 4) {          // four heads' loads in flight before the first is normalised
      float x[4][8];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const TIn* p = p0 + (int64_t)min(h0 + u, G - 1) * kHeadDim;
        if constexpr (sizeof(TIn) == 2) {
          const uint4 w = *reinterpret_cast<const uint4*>(p);
          x[u][0] = bf16lo(w.x); x[u][1] = bf16hi(w.x); x[u][2] = bf16lo(w.y); x[u][3] = bf16hi(w.y);
          x[u][4] = bf16lo(w.z); x[u][5] = bf16hi(w.z); x[u][6] = bf16lo(w.w); x[u][7] = bf16hi(w.w);
        } else {
          const float4 lo = *reinterpret_cast<const float4*>(p);
          const float4 hi = *reinterpret_cast<const float4*>(p + 4);
          x[u][0] = lo.x; x[u][1] = lo.y; x[u][2] = lo.z; x[u][3] = lo.w;
          x[u][4] = hi.x; x[u][5] = hi.y; x[u][6] = hi.z; x[u][7] = hi.w;
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        float inv = h0 + u < G ? 1.f : 0.f;      // a clamped repeat of the last head adds nothing
        if (normalize) {
          float ssq = 0.f;
#pragma unroll
          for (int i = 0; i < 8; ++i) ssq += x[u][i] * x[u][i];
          ssq += __shfl_xor(ssq, 1); ssq += __shfl_xor(ssq, 2);     // the 16 lanes of one group
          ssq += __shfl_xor(ssq, 4); ssq += __shfl_xor(ssq, 8);
          inv *= 1.0f / fmaxf(sqrtf(ssq), 1e-12f);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] += x[u][i] * inv;
      }
    }
  }
  if constexpr (kParts) {
    uint4 part[3];
    split_three<true>(acc, part);
    char* to = reinterpret_cast<char*>(qs) + part_at(row, g * kHeadDim + 8 * j, Hkv * kHeadDim);
#pragma unroll
    for (int p = 0; p < 3; ++p) *reinterpret_cast<uint4*>(to + p * kPartBytes) = part[p];
    return;
  }
  TOut* o = qs + ((int64_t)(by_units ? unit_row(row) : row) * Hkv + g) * kHeadDim + 8 * j;
  if constexpr (sizeof(TOut) == 2) {
    uint4 w;
    w.x = pack_bf16x2(acc[0], acc[1]); w.y = pack_bf16x2(acc[2], acc[3]);
    w.z = pack_bf16x2(acc[4], acc[5]); w.w = pack_bf16x2(acc[6], acc[7]);
    *reinterpret_cast<uint4*>(o) = w;
  } else {
    *reinterpret_cast<float4*>(o) = make_float4(acc[0], acc[1], acc[2], acc[3]);
    *reinterpret_cast<float4*>(o + 4) = make_float4(acc[4], acc[5], acc[6], acc[7]);
  }
}

// ------------------------------------------------------------------------------------------
// The other reductions over a query's tokens (src/msa_service.py:751-780): "mean" (sum over the scored tokens / their
// number) and "last" (the token at position count - 1, count = scored tokens).  Both are linear in the query row, or
// pick one, so they collapse the query to ONE pre-summed row before the scan: mean_t (q_t . k) = (mean_t q_t) . k.
// The scan and its max over rows then run unchanged on one row block per query whose 32 rows all hold that row.
//
// collapse_queries_kernel: one workgroup per (query, KV group); its 16 slots of 16 lanes take tokens slot, slot + 16,
// ...; a slot sums, over its tokens that count, the group's (normalised, in cosine mode) heads; the slots meet in LDS in
// a fixed order.  Writes the fp32 row and, from group 0, the number of tokens that counted.
// ------------------------------------------------------------------------------------------
constexpr int kQueryMax = MSA_QUERY_MAX, kQueryMean = MSA_QUERY_MEAN, kQueryLast = MSA_QUERY_LAST;

template <typename TIn>
__global__ __launch_bounds__(256) void collapse_queries_kernel(const TIn* __restrict__ q, const uint8_t* __restrict__ qmask,
                                                               int32_t S, int32_t Hq, int32_t Hkv, int32_t normalize,
                                                               int32_t query_reduce, float* __restrict__ rows,
                                                               int32_t* __restrict__ counts) {
  __shared__ float part[16][kHeadDim];
  __shared__ int n_scored;
  const int b = blockIdx.x, g = blockIdx.y;
  const int G = Hq / Hkv;
  const int slot = threadIdx.x >> 4, j = threadIdx.x & 15;
  // scored tokens of the query (every wavefront counts them: the result is needed by all)
  int count = 0;
  if (qmask == nullptr) {
    count = S;
  } else {
    const int lane = threadIdx.x & 63;
    for (int base = 0; base < S; base += 64) {
      const int t = base + lane;
      count += __builtin_popcountll(__ballot(t < S && qmask[(int64_t)b * S + t] != 0));
    }
  }
  const int last = max(count - 1, 0);
  auto counts_in = [&](int t) {
    const bool scored = qmask == nullptr || qmask[(int64_t)b * S + t] != 0;
    return query_reduce == kQueryLast ? (t == last && scored) : scored;
  };
  float acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = 0.f;
  int used = 0;
  for (int t = slot; t < S; t += 16) {
    if (!counts_in(t)) continue;                       // (uniform over the slot's 16 lanes)
    ++used;
    const TIn* p0 = q + (((int64_t)b * S + t) * Hq + g * G) * kHeadDim + 8 * j;
    for (int h = 0; h < G; ++h) {
      float x[8];
      const TIn* p = p0 + (int64_t)h * kHeadDim;
      if constexpr (sizeof(TIn) == 2) {
        const uint4 w = *reinterpret_cast<const uint4*>(p);
        x[0] = bf16lo(w.x); x[1] = bf16hi(w.x); x[2] = bf16lo(w.y); x[3] = bf16hi(w.y);
        x[4] = bf16lo(w.z); x[5] = bf16hi(w.z); x[6] = bf16lo(w.w); x[7] = bf16hi(w.w);
      } else {
        const float4 lo = *reinterpret_cast<const float4*>(p);
        const float4 hi = *reinterpret_cast<const float4*>(p + 4);
        x[0] = lo.x; x[1] = lo.y; x[2] = lo.z; x[3] = lo.w; x[4] = hi.x; x[5] = hi.y; x[6] = hi.z; x[7] = hi.w;
      }
      float inv = 1.f;
      if (normalize) {
        float ssq = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) ssq += x[i] * x[i];
        inv = 1.0f / fmaxf(sqrtf(row16_sum(ssq)), 1e-12f);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] += x[i] * inv;
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) part[slot][8 * j + i] = acc[i];
  if (threadIdx.x == 0) n_scored = 0;
  __syncthreads();
  if (j == 0 && used) atomicAdd(&n_scored, used);
  __syncthreads();
  if (threadIdx.x < kHeadDim) {
    float sum = 0.f;
    for (int s2 = 0; s2 < 16; ++s2) sum += part[s2][threadIdx.x];
    const int n = n_scored;
    rows[((int64_t)b * Hkv + g) * kHeadDim + threadIdx.x] = n > 0 ? sum / (float)n : 0.f;
    if (g == 0 && threadIdx.x == 0) counts[b] = n;
  }
}

// One row block (32 rows) per query, every row the collapsed row; mask words, padding words, the key plane and the
// tile pool's counter as presum_queries_kernel leaves them.  One workgroup per row.
template <typename TOut>
__global__ void broadcast_rows_kernel(const float* __restrict__ rows, const int32_t* __restrict__ counts, int32_t Hkv,
                                      TOut* __restrict__ qs, uint32_t* __restrict__ row_bits, int32_t mask_words,
                                      uint32_t* __restrict__ key_plane, int64_t clear_words, uint32_t* __restrict__ sched) {
  const int row = blockIdx.x, b = row >> 5;
  const int K = Hkv * kHeadDim;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < clear_words; i += (int64_t)gridDim.x * blockDim.x)
    key_plane[i] = 0u;
  const bool any = counts[b] > 0;
  if ((row & 31) == 0 && threadIdx.x == 0) row_bits[row >> 5] = any ? 0xffffffffu : 0u;
  if (blockIdx.x == 0) {
    for (int w = (int)(gridDim.x >> 5) + (int)threadIdx.x; w < mask_words; w += blockDim.x) row_bits[w] = 0u;
    if (threadIdx.x == 0) sched[0] = 0u;
  }
  for (int c = threadIdx.x; c < K; c += blockDim.x) {
    const float x = any ? rows[(int64_t)b * K + c] : 0.f;
    if constexpr (sizeof(TOut) == 2) qs[(int64_t)row * K + c] = f32_to_bf16(x);
    else qs[(int64_t)row * K + c] = x;
  }
}

// ------------------------------------------------------------------------------------------
// MFMA operand traits.  LDS rows hold 128 bytes of K (64 bf16 or 32 fp32) plus 16 bytes of pad,
// which makes the 16-byte / 4-byte operand reads of a 32-row block bank-conflict free.
// ------------------------------------------------------------------------------------------
constexpr int kRowBytes = 128;
constexpr int kRowStride = kRowBytes + 16;

template <typename T>
struct Mma;
template <>
struct Mma<bf16_t> {
  typedef bf16x8_t Frag;
  static constexpr int kSub = 4;   // 32x32x16 steps per 64-element K tile
  static __device__ __forceinline__ Frag load(const char* row, int sub, int half) {
    return *reinterpret_cast<const Frag*>(row + sub * 32 + half * 16);
  }
  static __device__ __forceinline__ floatx16_t mma(Frag a, Frag b, floatx16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mma<float> {
  typedef float Frag;
  static constexpr int kSub = 16;  // 32x32x2 steps per 32-element K tile
  static __device__ __forceinline__ Frag load(const char* row, int sub, int half) {
    return *reinterpret_cast<const Frag*>(row + sub * 8 + half * 4);
  }
  static __device__ __forceinline__ floatx16_t mma(Frag a, Frag b, floatx16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
  }
};

// The HBM-bound form for up to 128 query rows (bf16, 128 x 256, streaming over N tiles) stages its operand tiles with
// buffer loads that write LDS directly (no staging registers, no ds_write; un-padded 128-byte rows whose 16-byte units
// are XOR-swizzled by (row >> 1) & 7: a direct load cannot pad, its 64 lanes fill 1 KB of LDS in lane order, so the
// swizzle is applied to the global address each lane fetches), three
// stages of each operand (3 x 16 KB + 3 x 32 KB = 144 KB): both operands are requested two K steps ahead, which keeps
// 96 KB per compute unit in flight (returns are in order, so the query tile has to run as far ahead as the K_r tile for
// the K_r tile's lead to count).
constexpr int kDtlStreamLdsBytes = 3 * (128 + 256) * 128;

// Chunks of a document are adjacent columns: a segmented max-scan over the 32 lanes of each half of a wavefront leaves a document's maximum
// in the last lane of its run, which alone touches memory (about two atomics per 32 chunks instead of 32 stores, and no per-chunk plane
// to read back).  What a lane may take in a step of the scan depends on the documents alone, so it is found once for all queries that are
// folded over them: four shifts inside the rows of 16 lanes, then lane 15 of the lower row joins the runs that cross into the upper one.
// Lanes that a shift cannot reach read 0, the identity of max over keys.
struct DocRuns {
  int doc;
  uint32_t take[5];      // all ones where the lane's run reaches as far
  bool last;             // the run's last lane, inside the bank
};
__device__ __forceinline__ DocRuns doc_runs(int doc, bool inside, int half, int l32) {
  DocRuns r;
  r.doc = doc;
  const int prev = __builtin_amdgcn_update_dpp(doc, doc, 0x138, 0xF, 0xF, false);      // wave_shr:1
  const uint64_t heads64 = __ballot(l32 == 0 || prev != doc);
  const uint32_t heads = half ? (uint32_t)(heads64 >> 32) : (uint32_t)heads64;
  const uint32_t upto = heads & ((2u << l32) - 1u);                  // heads at or below this lane (never empty)
  const int dist = l32 - (31 - __builtin_clz(upto));                 // from the first lane of the run
#pragma unroll
  for (int k = 0; k < 4; ++k) r.take[k] = dist >= 1 << k ? 0xffffffffu : 0u;
  r.take[4] = dist > (l32 & 15) ? 0xffffffffu : 0u;
  r.last = inside && (l32 == 31 || ((heads >> (l32 + 1)) & 1u));
  return r;
}
// The lanes' keys folded over the runs, into the query's row of the key plane.
__device__ __forceinline__ void merge_runs(const DocRuns& r, float run, uint32_t* row, bool scored) {
  uint32_t m = f32_to_key(run);
#define MSA_SCAN_STEP(K, CTRL, ROWS) \
  m = max(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, CTRL, ROWS, 0xF, ROWS == 0xF) & r.take[K]);
  MSA_SCAN_STEP(0, 0x111, 0xF)   // row_shr:1
  MSA_SCAN_STEP(1, 0x112, 0xF)
  MSA_SCAN_STEP(2, 0x114, 0xF)
  MSA_SCAN_STEP(3, 0x118, 0xF)
  MSA_SCAN_STEP(4, 0x142, 0xA)   // row_bcast:15 into rows 1, 3
#undef MSA_SCAN_STEP
  if (r.last && scored) atomicMax(row + r.doc, m);
}
template <typename T, int BM, int BN, int kSets, bool kStream>
constexpr bool score_tile_is_direct_stream() {
  return sizeof(T) == 2 && BM == 128 && BN == 256 && kSets == 1 && kStream;
}

// Workgroup tile BM x BN, WAVES_M x WAVES_N wavefronts, each owning TM x TN blocks of 32 x 32.
// kSets: register sets of global loads, i.e. K tiles in flight ahead of the one being multiplied.  One is enough when
// a tile's MFMA work outlasts a load's latency (the MFMA-bound shapes); the HBM-bound shapes (few query rows) need
// more bytes in flight per compute unit than one tile holds.
// kDocMax: keys are folded over the chunks of a document (chunk_doc) and merged into out_key[B, n_docs];
// otherwise one key per (query, chunk) is merged into out_key[B, C].
// kUnit: rows a query is a multiple of.  32: one that is scored counts whole.  8 and 4: short queries share a row block, whose word tells
// the rows that count; a query of units of 4 is one unit.
// kStream: one workgroup per compute-unit slot walks N tiles blockIdx.x, blockIdx.x + gridDim.x, ... (one M tile
// only) with the load / store / multiply pipeline running across tile boundaries: the first K tiles of the next N
// tile are already in flight while the last ones of the current tile are multiplied and its epilogue runs, so the
// HBM stream never drains between tiles.  That is what the HBM-bound shapes need; the fp32 form keeps one
// workgroup per tile.
template <typename T, int BM, int BN, int WAVES_M, int WAVES_N, int kSets, bool kDocMax, bool kStream, int kUnit = 32>
__global__ __launch_bounds__(WAVES_M* WAVES_N * 64) void score_gemm_kernel(
    const T* __restrict__ qs,            // [M_rows, K]  pre-summed queries, M_rows = B * S_pad
    const T* __restrict__ kr,            // [C, K]
    const uint32_t* __restrict__ row_bits,  // [ceil(M_alloc / 32)] scored-row bitmask
    uint32_t* __restrict__ out_key,      // [B, n_docs] or [B, C], zeroed
    const int32_t* __restrict__ chunk_doc,  // [C] document of every chunk (kDocMax)
    int32_t M_rows, int32_t C, int32_t K, int32_t units_per_query, int32_t tiles_m, int32_t tiles_n,
    int32_t m_group, int32_t n_docs) {
  static_assert(kUnit == 32 || (kDocMax && (kUnit == 8 || kUnit == 4)), "packed queries are folded over documents");
  constexpr int kThreads = WAVES_M * WAVES_N * 64;
  constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  constexpr int TM = WM / 32, TN = WN / 32;
  constexpr int kVecA = BM * 8 / kThreads, kVecB = BN * 8 / kThreads;   // 16-byte vectors per thread per tile
  static_assert(BM * 8 % kThreads == 0 && BN * 8 % kThreads == 0, "tile/threads mismatch");

  extern __shared__ __align__(16) char lds[];
  constexpr int kBufBytes = (BM + BN) * kRowStride;   // [A tile | B tile] per buffer, two buffers
  constexpr bool kDtlStream = score_tile_is_direct_stream<T, BM, BN, kSets, kStream>();

  // XCD-aware tile order: workgroups are dealt round-robin to the 8 XCDs, so each XCD gets one
  // contiguous range of K_r tiles.  Inside it the M tiles are walked in groups of m_group: a group's
  // query rows stay in that XCD's L2 while its K_r tiles stream past once per group.
  int tile_n, tile_m;
  if constexpr (kStream) {
    tile_n = blockIdx.x;
    tile_m = 0;
  }
  // Position `vb` of the XCD-aware tile order -> (M tile, N tile); false for the padding positions of the order.
  const int n_per_xcd = (tiles_n + 7) / 8, per_group = n_per_xcd * m_group;
  auto decode_tile = [&](int vb, int& tm, int& tn) -> bool {
    const int within = vb / 8;
    const int rem = within % per_group;
    tn = (vb % 8) * n_per_xcd + rem / m_group;
    tm = (within / per_group) * m_group + rem % m_group;
    return tn < tiles_n && tm < tiles_m;
  };
  if constexpr (!kStream) {
    if (!decode_tile(blockIdx.x, tile_m, tile_n)) return;
  }
  if (tile_n >= tiles_n || tile_m >= tiles_m) return;
  int m0 = tile_m * BM, n0 = tile_n * BN;

  const int tid = threadIdx.x, lane = tid & 63;
  // (wave-uniform by construction; said so, the LDS addresses of the direct loads stay in scalar registers instead of
  // being read back from a lane in front of every load: 1.9 % on the large-tile scan)
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  const int half = lane >> 5, l32 = lane & 31;

  const int64_t row_bytes_g = (int64_t)K * sizeof(T);
  const char* ga = reinterpret_cast<const char*>(qs);
  const char* gb = reinterpret_cast<const char*>(kr);

  // Global -> register staging through buffer loads: one resource per operand tile whose extent is
  // the valid part of the tile, so rows past M_rows / C read as zero in hardware (no branches, no
  // clamps).  The range check is defined on the vector offset, so the row displacement of a thread's
  // vectors rides there; the K-tile displacement (which stays inside the row, so it can never carry a
  // load past the extent) is scalar.
  const int rows_a = min(BM, M_rows - m0);
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(ga) + (int64_t)m0 * row_bytes_g, 0, (int)(rows_a * row_bytes_g), 0x00020000);
  const int rows_b = min(BN, C - n0);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(gb) + (int64_t)n0 * row_bytes_g, 0, (int)(rows_b * row_bytes_g), 0x00020000);
  __amdgpu_buffer_rsrc_t rsrc_ld = rsrc_b;      // kStream: the N tile the loads have reached
  const int voff = (tid >> 3) * (int)row_bytes_g + (tid & 7) * 16;
  const int vec_stride = (kThreads / 8) * (int)row_bytes_g;     // rows between a thread's vectors
  static_assert(kSets == 1 || kSets == 2, "one or two K tiles in flight");
  u32x4_t ra[kSets][kVecA], rb[kSets][kVecB];
  // K_r streams through once per M tile group while the query matrix is re-read by every workgroup of an XCD: the
  // non-temporal hint on the K_r loads keeps the queries in the 4 MiB L2 (traffic past L2 9.9 -> 6.9 GB per launch
  // at the 100M-token bank, 1.5 % faster).
  constexpr int kStreamHint = 2;
  constexpr int kPastEnd = 0x40000000;   // vector offset beyond any tile's extent: the load returns zeros, no traffic
  const int k_tiles = (int)(row_bytes_g / kRowBytes);
  auto load_tile = [&](auto set_tag, int kt) {
    constexpr int set = decltype(set_tag)::value;
    const int vo = kt < k_tiles ? voff : kPastEnd;   // a tile past the row is never fetched (keeps the loop branch-free)
#pragma unroll
    for (int i = 0; i < kVecA; ++i)
      ra[set][i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, vo + i * vec_stride, kt * kRowBytes, 0);
#pragma unroll
    for (int i = 0; i < kVecB; ++i) {
      if constexpr (kStream)
        rb[set][i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_ld, vo + i * vec_stride, kt * kRowBytes, kStreamHint);
      else
        rb[set][i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, vo + i * vec_stride, kt * kRowBytes, kStreamHint);
    }
  };
  // kStream: the loads walk the workgroup's whole sequence of (N tile, K tile) steps; past its last tile they
  // fetch nothing.
  int ld_n0 = n0, ld_kt = 0;
  auto load_next = [&](auto set_tag) {
    load_tile(set_tag, ld_n0 < C ? ld_kt : k_tiles);
    if (++ld_kt == k_tiles) {
      ld_kt = 0;
      ld_n0 = (int)min((int64_t)ld_n0 + (int64_t)gridDim.x * BN, (int64_t)C);
      rsrc_ld = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(gb) + (int64_t)ld_n0 * row_bytes_g, 0,
                                                  (int)(min(BN, C - ld_n0) * row_bytes_g), 0x00020000);
    }
  };
  auto store_tile = [&](auto set_tag, int buf) {
    constexpr int set = decltype(set_tag)::value;
#pragma unroll
    for (int i = 0; i < kVecA; ++i) {
      const int v = tid + i * kThreads, r = v >> 3, c = v & 7;
      *reinterpret_cast<u32x4_t*>(lds + buf * kBufBytes + r * kRowStride + c * 16) = ra[set][i];
    }
#pragma unroll
    for (int i = 0; i < kVecB; ++i) {
      const int v = tid + i * kThreads, r = v >> 3, c = v & 7;
      *reinterpret_cast<u32x4_t*>(lds + buf * kBufBytes + (BM + r) * kRowStride + c * 16) = rb[set][i];
    }
  };
  typedef std::integral_constant<int, 0> Set0;
  typedef std::integral_constant<int, 1 % kSets> Set1;

  floatx16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // Software pipeline over K tiles.  While tile kt is multiplied out of LDS buffer kt&1:
  //   - tile kt+1 (already in registers) is written to the other buffer during sub-step 1, and the
  //     global loads of tile kt+2 are issued right behind it (a whole iteration to land);
  //   - operand fragments are double-buffered in registers, one sub-step ahead of the MFMAs;
  //   - the single barrier per tile sits before the LAST sub-step's MFMAs, after that sub-step's
  //     fragments were read, so the first fragments of tile kt+1 are fetched under those MFMAs.
  // Hazards: buffer (kt+1)&1 held tile kt-1, whose last fragment reads were issued before the
  // barrier of iteration kt-1; the writes of tile kt+1 are complete at the barrier of iteration kt.
  typedef typename Mma<T>::Frag Frag;
  constexpr int kSub = Mma<T>::kSub;
  const int a_row = (wm * WM + l32) * kRowStride, b_row = (BM + wn * WN + l32) * kRowStride;
  Frag fa[2][TM], fb[2][TN];
  auto load_frags = [&](int buf, int sub, int slot) {
    const char* pa = lds + buf * kBufBytes + a_row;
    const char* pb = lds + buf * kBufBytes + b_row;
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[slot][i] = Mma<T>::load(pa + i * 32 * kRowStride, sub, half);
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[slot][j] = Mma<T>::load(pb + j * 32 * kRowStride, sub, half);
  };

  // One K tile out of LDS buffer `step & 1`; kMore says a next step exists (the steady-state loop is
  // compiled without that condition so the wait counters around the barrier stay exact).  Tile t travels in
  // register set t % kSets; `set_tag` names the set that holds the next step's tile, which is stored and then
  // refilled with the tile kSets steps further on.
  auto k_tile = [&](auto more_tag, auto set_tag, int step) {
    constexpr bool kMore = decltype(more_tag)::value;
    const int buf = step & 1;
#pragma unroll
    for (int sub = 0; sub < kSub; ++sub) {
      if (sub + 1 < kSub) {
        load_frags(buf, sub + 1, (sub + 1) & 1);
      } else if (kMore) {
        __syncthreads();
        load_frags(buf ^ 1, 0, 0);
        __builtin_amdgcn_sched_barrier(0);   // keep the last sub-step's MFMAs behind these reads
      }
      if (sub == 1 && kMore) {
        store_tile(set_tag, buf ^ 1);
        if constexpr (kStream) {
          __builtin_amdgcn_sched_barrier(0);   // the refill reuses the registers the stores above read
          load_next(set_tag);
        } else if constexpr (kSets > 1) {
          __builtin_amdgcn_sched_barrier(0);
          load_tile(set_tag, step + 1 + kSets);
        } else if (step + 2 < k_tiles) {
          load_tile(set_tag, step + 2);
        }
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = Mma<T>::mma(fa[sub & 1][i], fb[sub & 1][j], acc[i][j]);
    }
  };

  // ---- direct-to-LDS form (see score_tile_is_direct_stream) ----
  // A wavefront's load instruction covers 8 rows of the operand tile: lane l lands in LDS at byte 16 * l of that 1 KB
  // block, i.e. row l / 8, unit slot l % 8, and fetches the unit that belongs there.
  const int dtl_row = (lane >> 3), dtl_slot = lane & 7;

  // Epilogue of the N tile starting at chunk `tile_n0`.  acc[i][j][e] is row 8*(e/4) + 4*half + e%4, column l32 of
  // its 32x32 block.  Consecutive row blocks of one query are folded into `run` (each half of the wavefront over its
  // own rows); emit() joins the halves and merges the query's column maxima of both blocks into the key plane.
  // Several wavefronts and workgroups hold parts of a query (and of a document), so the merge is an atomicMax into
  // a zeroed plane.  emit() is reached by whole wavefronts (q and any are uniform).
  //
  // With one workgroup per compute unit nothing else runs while an epilogue waits, so it must not wait on memory:
  // the scored-row words of the wavefront's row blocks and the documents of its columns are requested ahead (before
  // the K loop / a tile ahead) and only consumed here, and the lane exchanges of the document fold are row moves.
  const int n_queries = M_rows / (units_per_query * kUnit);
  uint32_t rbits[TM];                                   // scored-row word of each row block (same in every lane)
  // query of the wavefront's first row block (unit) and its place in the query: later ones follow by counting
  // (one division per wavefront, under the first tile's load latency, instead of one per block in the epilogue)
  int q_first = 0, r_first = 0;
  auto fetch_rows = [&]() {
#pragma unroll
    for (int i = 0; i < TM; ++i) rbits[i] = row_bits[(m0 + wm * WM + i * 32) >> 5];   // 0 past M_rows (buffer is padded)
    const int blk0 = (m0 + wm * WM) / kUnit;
    q_first = blk0 / units_per_query;
    r_first = blk0 - q_first * units_per_query;
  };
  int cdoc[TN];                                         // document of each column; lanes past the bank never join a run
  auto fetch_docs = [&](int tile_n0) {
    if constexpr (kDocMax) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = tile_n0 + wn * WN + j * 32 + l32;
        cdoc[j] = n < C ? chunk_doc[n] : -1 - l32;
      }
    }
  };
  // Both column blocks of the wavefront at once: after the halves are joined (one half-wave swap: the upper half of
  // block 0's partial maxima against the lower half of block 1's) the lower 32 lanes hold block 0's 32 column maxima
  // and the upper 32 lanes block 1's, so the segmented scan and the atomics below run once per query for the
  // wavefront's 64 columns instead of once per block with half the lanes idle.
  static_assert(TN == 2, "the epilogue pairs the two column blocks of a wavefront");
  DocRuns runs[kUnit == 4 ? 2 : 1];      // of the wavefront's 64 columns, half a half; of either 32, in both halves, where a half has queries of its own
  auto find_runs = [&](int tile_n0) {
    if constexpr (kDocMax && kUnit == 4) {
#pragma unroll
      for (int j = 0; j < TN; ++j) runs[j] = doc_runs(cdoc[j], tile_n0 + wn * WN + j * 32 + l32 < C, half, l32);
    } else if constexpr (kDocMax) {
      runs[0] = doc_runs(half ? cdoc[1] : cdoc[0], tile_n0 + wn * WN + half * 32 + l32 < C, half, l32);
    }
  };
  auto emit = [&](int q, int tile_n0, const float (&run_half)[TN], bool any) {
    if (!any || q >= n_queries) return;
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(run_half[0]), __float_as_uint(run_half[1]), false, false);
    const float run = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    if constexpr (kDocMax) {
      merge_runs(runs[0], run, out_key + (int64_t)q * n_docs, true);
    } else {
      const int n = tile_n0 + wn * WN + half * 32 + l32;
      if (n < C) atomicMax(&out_key[(int64_t)q * C + n], f32_to_key(run));
    }
  };
  auto four = [&](const floatx16_t& a, int g) { return fmaxf(fmaxf(a[4 * g], a[4 * g + 1]), fmaxf(a[4 * g + 2], a[4 * g + 3])); };
  auto epilogue = [&](int tile_n0) {
    find_runs(tile_n0);
    if constexpr (kUnit == 4) {
      // registers 4 g .. 4 g + 3 of a block are rows of two queries, one a half of the wavefront: nothing to join.  A maximum of what is no
      // number counts for nothing, as in the forms that join some with -inf: its key would be in front of every score's.
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const uint32_t bits = __builtin_amdgcn_readfirstlane(rbits[i]);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          if ((bits >> (8 * g) & 0xffu) == 0u) continue;
          const bool scored = bits >> (8 * g + 4 * half) & 1u;
          uint32_t* const row = out_key + (int64_t)(q_first + 8 * i + 2 * g + half) * n_docs;
#pragma unroll
          for (int j = 0; j < TN; ++j) merge_runs(runs[j], fmaxf(-INFINITY, four(acc[i][j], g)), row, scored);
        }
      }
      return;
    }
    float run[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) run[j] = -INFINITY;
    bool any = false;
    int run_q = q_first, r = r_first;                      // query of row block i, its block index inside the query
    if constexpr (kUnit == 8) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const uint32_t bits = __builtin_amdgcn_readfirstlane(rbits[i]);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          if (r == units_per_query) {                      // the unit opens the next query
            emit(run_q, tile_n0, run, any);
#pragma unroll
            for (int j = 0; j < TN; ++j) run[j] = -INFINITY;
            any = false; ++run_q; r = 0;
          }
          ++r;
          if ((bits >> (8 * g) & 0xffu) == 0u) continue;
#pragma unroll
          for (int j = 0; j < TN; ++j) run[j] = fmaxf(run[j], four(acc[i][j], g));
          any = true;
        }
      }
      emit(run_q, tile_n0, run, any);
      return;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const uint32_t bits = __builtin_amdgcn_readfirstlane(rbits[i]);
      if (r == units_per_query) {                          // row block i opens the next query
        emit(run_q, tile_n0, run, any);
#pragma unroll
        for (int j = 0; j < TN; ++j) run[j] = -INFINITY;
        any = false; ++run_q; r = 0;
      }
      ++r;
      if (bits == 0xffffffffu) {                            // every row scored: no per-row tests
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          float mx = acc[i][j][0];
#pragma unroll
          for (int e = 1; e < 16; ++e) mx = fmaxf(mx, acc[i][j][e]);
          run[j] = fmaxf(run[j], mx);
        }
        any = true;
      } else if (bits != 0) {
        const uint32_t mine = bits >> (4 * half);           // this half's rows: bit 8*(e/4) + e%4
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          float mx = -INFINITY;
#pragma unroll
          for (int e = 0; e < 16; ++e)
            if (mine & (1u << (8 * (e >> 2) + (e & 3)))) mx = fmaxf(mx, acc[i][j][e]);
          run[j] = fmaxf(run[j], mx);
        }
        any = true;
      }
    }
    emit(run_q, tile_n0, run, any);
  };

  if constexpr (kDtlStream) {
    static_assert(kThreads == 512 && kSub == 4 && TM == 2 && TN == 2, "laid out for 8 wavefronts of 64 x 64");
    constexpr int kAStage = BM * 128, kBStage = BN * 128, kStages = 3;
    constexpr int kALoads = BM / 64, kBLoads = BN / 64;      // 1 KB blocks (8 rows) per wavefront and stage
    constexpr int kWaitAllButNewestStep = 0x0F70 + kALoads + kBLoads, kWaitAll = 0x0F70;
    char* const lds_a = lds;
    char* const lds_b = lds + kStages * kAStage;
    auto dtl_barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    auto voff_of = [&](int row) { return row * (int)row_bytes_g + ((dtl_slot ^ ((row >> 1) & 7)) * 16); };
    auto load_a = [&](int stage, int kt) {
#pragma unroll
      for (int i = 0; i < kALoads; ++i) {
        const int blk = wave * kALoads + i;
        MSA_LOAD_TO_LDS(rsrc_a, lds_a + stage * kAStage + blk * 1024, voff_of(blk * 8 + dtl_row), kt * kRowBytes, 0);
      }
    };
    auto load_b = [&](int stage, int kt) {
#pragma unroll
      for (int i = 0; i < kBLoads; ++i) {
        const int blk = wave * kBLoads + i;
        MSA_LOAD_TO_LDS(rsrc_ld, lds_b + stage * kBStage + blk * 1024, voff_of(blk * 8 + dtl_row), kt * kRowBytes,
                        kStreamHint);
      }
    };
    auto frags = [&](int stage, int sub, int slot) {
      const int unit = sub * 2 + half;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int row = wm * WM + i * 32 + l32;
        fa[slot][i] = *reinterpret_cast<const Frag*>(lds_a + stage * kAStage + row * 128 + ((unit ^ ((row >> 1) & 7)) * 16));
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int row = wn * WN + j * 32 + l32;
        fb[slot][j] = *reinterpret_cast<const Frag*>(lds_b + stage * kBStage + row * 128 + ((unit ^ ((row >> 1) & 7)) * 16));
      }
    };
    // The workgroup's N tiles (blockIdx.x, blockIdx.x + gridDim.x, ...) form one sequence of K steps; the loads run two
    // steps ahead of the MFMAs across tile boundaries.
    const int my_tiles = (tiles_n - tile_n + (int)gridDim.x - 1) / (int)gridDim.x;
    int t_ld = 0, kt_ld = 0;                       // tile and K tile the loads have reached
    auto advance_ld = [&]() {
      if (++kt_ld == k_tiles) {
        kt_ld = 0;
        if (++t_ld < my_tiles) {
          const int tn = tile_n + t_ld * (int)gridDim.x;
          rsrc_ld = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(gb) + (int64_t)tn * BN * row_bytes_g, 0,
                                                      (int)(min(BN, C - tn * BN) * row_bytes_g), 0x00020000);
        }
      }
    };
    fetch_rows();                                  // one M tile: the scored-row words serve every N tile
    fetch_docs(n0);
    load_a(0, 0);
    load_b(0, 0);
    advance_ld();
    if (t_ld < my_tiles) {
      load_a(1, kt_ld);
      load_b(1, kt_ld);
      advance_ld();
      __builtin_amdgcn_s_waitcnt(kWaitAllButNewestStep);
    } else {
      __builtin_amdgcn_s_waitcnt(kWaitAll);
    }
    dtl_barrier();
    frags(0, 0, 0);
    int st = 0, t = 0, kt = 0;
    for (;;) {
      const int st1 = st == 2 ? 0 : st + 1, st2 = st1 == 2 ? 0 : st1 + 1;
      const bool more = !(t == my_tiles - 1 && kt == k_tiles - 1);    // a next step exists
      const bool more2 = t_ld < my_tiles;                              // the step behind it exists
      if (more2) {
        load_a(st2, kt_ld);      // stage of the step before this one: its last reads were behind the previous barrier
        load_b(st2, kt_ld);
        advance_ld();
      }
      auto substep = [&](auto sub_tag, auto fresh_tag) {
        constexpr int sub = decltype(sub_tag)::value;
        constexpr bool fresh = decltype(fresh_tag)::value;
        if constexpr (sub + 1 < kSub) {
          frags(st, sub + 1, (sub + 1) & 1);
        } else {
          if (more) {
            if (more2) __builtin_amdgcn_s_waitcnt(kWaitAllButNewestStep);
            else __builtin_amdgcn_s_waitcnt(kWaitAll);
            dtl_barrier();
            frags(st1, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            if constexpr (fresh) acc[i][j] = Mma<T>::mma(fa[sub & 1][i], fb[sub & 1][j], floatx16_t{});
            else acc[i][j] = Mma<T>::mma(fa[sub & 1][i], fb[sub & 1][j], acc[i][j]);
          }
        if constexpr (sub + 1 < kSub) {
#pragma unroll
          for (int g = 0; g < TM + TN; ++g) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // one LDS read
          }
        }
      };
      if (kt == 0) substep(std::integral_constant<int, 0>{}, std::true_type{});
      else substep(std::integral_constant<int, 0>{}, std::false_type{});
      substep(std::integral_constant<int, 1>{}, std::false_type{});
      substep(std::integral_constant<int, 2>{}, std::false_type{});
      substep(std::integral_constant<int, 3>{}, std::false_type{});
      st = st1;
      if (++kt == k_tiles) {
        epilogue(n0);
        if (!more) break;
        kt = 0;
        ++t;
        n0 += (int)gridDim.x * BN;
        fetch_docs(n0);
      }
    }
  } else if constexpr (kStream) {
    // The workgroup's tiles form one sequence of steps (K tiles are even in number, so set tags and LDS buffers
    // alternate the same way in every tile); an epilogue sits where a tile's last step ends, with the next tile's
    // first operand fragments already in registers and its loads in flight.
    const int my_tiles = (tiles_n - tile_n + (int)gridDim.x - 1) / (int)gridDim.x;
    const int steps = my_tiles * k_tiles;
    load_next(Set0{});
    store_tile(Set0{}, 0);
    load_next(Set1{});
    if constexpr (kSets == 2) load_next(Set0{});
    __syncthreads();
    load_frags(0, 0, 0);
    fetch_rows();
    fetch_docs(n0);
    int done_n0 = n0, in_tile = 0;
    for (int step = 0; step + 2 < steps; step += 2) {
      k_tile(std::true_type{}, Set1{}, step);
      k_tile(std::true_type{}, Set0{}, step + 1);
      in_tile += 2;
      if (in_tile == k_tiles) {
        epilogue(done_n0);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
        in_tile = 0;
        done_n0 += (int)gridDim.x * BN;
        fetch_docs(done_n0);
      }
    }
    k_tile(std::true_type{}, Set1{}, steps - 2);
    k_tile(std::false_type{}, Set0{}, steps - 1);
    epilogue(done_n0);
  } else {
    if constexpr (kSets == 2) {
      // tile t travels in register set (t & 1): iteration kt stores tile kt+1 and refills its set with tile kt+3
      load_tile(Set0{}, 0);
      store_tile(Set0{}, 0);
      load_tile(Set1{}, 1);
      load_tile(Set0{}, 2);
      __syncthreads();
      load_frags(0, 0, 0);
      fetch_rows();
      fetch_docs(n0);
      int kt = 0;
      for (; kt + 2 < k_tiles; kt += 2) {
        k_tile(std::true_type{}, Set1{}, kt);
        k_tile(std::true_type{}, Set0{}, kt + 1);
      }
      if (kt + 1 < k_tiles) {
        k_tile(std::true_type{}, Set1{}, kt);
        k_tile(std::false_type{}, Set0{}, kt + 1);
      } else {
        k_tile(std::false_type{}, Set1{}, kt);
      }
    } else {
      load_tile(Set0{}, 0);
      store_tile(Set0{}, 0);
      if (k_tiles > 1) load_tile(Set0{}, 1);
      __syncthreads();
      load_frags(0, 0, 0);
      fetch_rows();
      fetch_docs(n0);
      for (int kt = 0; kt + 1 < k_tiles; ++kt) k_tile(std::true_type{}, Set0{}, kt);
      k_tile(std::false_type{}, Set0{}, k_tiles - 1);
    }
    epilogue(n0);
  }
}

// ------------------------------------------------------------------------------------------
// The MFMA-bound form (bf16, more than 128 query rows): 256 x 256 tile, four wavefronts (one per SIMD) of 128 x 128,
// a wavefront's 8 x 8 blocks of 16 x 16 in the 256 accumulation registers, and the K step written at the
// instruction level (scan_asm.inc, generated by gen_scan_asm.py, which describes the schedule and the registers the
// asm statements own: v128 - v255 and a0 - a255; the compiler-allocated code of this kernel is held below v128 by the
// register limit on its declaration and uses no accumulation registers, which the build checks).  One wavefront per
// SIMD has nobody to cover a wait, so every wait the step contains is met long before it is reached: operand
// fragments are read a sub-step ahead, the query and K_r tiles are requested two K steps ahead (LDS: two stages of the
// query tile, three of the K_r tile, filled by buffer loads that write LDS directly), and the one barrier per step
// stands behind an MFMA.  128 x 128 wavefront tiles read a third less from LDS per product than a 2 x 4 layout of eight
// wavefronts.
//
// What bounds it is power: the clock falls until the chip is inside its budget (matrix cores busy 0.84 of the cycles at 1.5 - 1.75 GHz,
// of 2.4), so what counts is energy per product.  v_mfma_f32_16x16x32_bf16 passes an accumulator half as often for the same products as
// v_mfma_f32_32x32x16_bf16: 1.605M chunks x 2048 query rows take 4.25 ms here, 4.66 with the 32 x 32 x 16 form (1.58 and 1.45
// PFLOP/s).  A loop of nothing but MFMAs (msa_diag_mfma_loop) shows part of that: 1953 TFLOP/s against 1886 with operands that
// change; on zeros, which cost little power, the larger form is the faster one (2213 and 2449).
//
// Persistent: one workgroup per compute unit walks its share of the tile list (scan_walk.h) as one sequence of K
// steps, the loads two steps ahead across tile boundaries.  With a gather job attached the last workgroup of the
// launch copies the K / V rows of an earlier selection instead (gather_device.h).  The last pool_n N tiles are handed
// out one at a time to workgroups that have finished their own share: during the first K steps of the tile in front of
// a pool tile one lane draws a position from the pool's counter (an atomic that returns), publishes it through the
// workgroup's claim word (an exchange that returns, so its arrival says the word is in L2) and every wavefront reads
// it back, one hop per K step, each issued in front of the step's tile loads so that the step's own wait (all but the
// eight newest loads) covers it.  The hops' values live in v217 - v219.
// ------------------------------------------------------------------------------------------
#include "scan_asm.inc"
#include "scan_walk.h"

constexpr int kScan4CompilerVgprs = 128;     // the compiler's share of the vector registers in score_scan4_kernel
constexpr int kScan4UnitsVgprs = 96;         // and in score_scan4_units_kernel, whose statements own v96 - v127 too
constexpr int kScan4LdsBytes = 5 * 256 * 128;

// kUnits: short queries share row blocks in units of eight rows (RowPacking), up to four queries a block.  A block's word tells the units
// that count, the reduction leaves a maximum per unit, and all of a tile's maxima are folded between two of the next tile's steps.
template <bool kDocMax, bool kUnits>
__device__ __forceinline__ void scan4_body(
    const bf16_t* __restrict__ qs,          // [M_rows, K]  pre-summed queries, M_rows = B * S_pad
    const bf16_t* __restrict__ kr,          // [C, K]
    const uint32_t* __restrict__ row_bits,  // [ceil(M_alloc / 32)] scored-row bitmask
    uint32_t* __restrict__ out_key,         // [B, n_docs] or [B, C], zeroed
    const int32_t* __restrict__ chunk_doc,  // [C] document of every chunk (kDocMax)
    int32_t M_rows, int32_t C, int32_t K, int32_t blocks_per_query, int32_t tiles_m, int32_t tiles_n, int32_t m_group,
    int32_t n_docs, const GatherJob& job, uint32_t* __restrict__ sched, int32_t pool_n) {      // (kUnits: units per query)
  [[maybe_unused]] constexpr int kUnit = kUnits ? 8 : 32;
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int kThreads = 256, BM = 256, BN = 256;
  extern __shared__ __align__(16) char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (job.active && (int)blockIdx.x == (int)gridDim.x - 1) {
    // plan (sorted, de-duplicated selection -> copy entries), host rows, then the documents an earlier sample already
    // fetched; the workgroup barriers order the three steps' memory
    msa_gather::plan_body(job.doc_sel, job.doc_chunk_off, job.n_docs, job.B, job.k,
                          (int32_t)min(job.capacity_rows, (int64_t)0x7fffffff), job.dedup, job.cu_sel, job.plan,
                          reinterpret_cast<int32_t*>(lds), tid, kThreads);
    __syncthreads();
    const int groups = kThreads / msa_gather::kCopyRowLanes;
    const int group = tid / msa_gather::kCopyRowLanes, lane_in_row = tid % msa_gather::kCopyRowLanes;
    msa_gather::copy_body<false, 8>(job.k_src, job.v_src, job.plan, job.B * job.k, job.row_vecs, job.capacity_rows,
                                    job.k_dst, job.v_dst, 0, 1, group, groups, lane_in_row);
    __syncthreads();
    if (job.dedup)
      msa_gather::copy_body<true, 8>(nullptr, nullptr, job.plan, job.B * job.k, job.row_vecs, job.capacity_rows, job.k_dst,
                                     job.v_dst, 0, 1, group, groups, lane_in_row);
    return;
  }
  const ScanWalk walk = scan_walk_init((int)blockIdx.x, (int)gridDim.x, job.active ? 1 : 0, tiles_m, tiles_n, m_group, pool_n);
  if (walk.own_count == 0) return;

  const int wm = wave >> 1, wn = wave & 1;
  const int half = lane >> 5, l32 = lane & 31;
  const int row_bytes = K * (int)sizeof(bf16_t);
  const int k_tiles = row_bytes / kRowBytes;
  {
    // per-lane constants of the asm statements: LDS offsets of the operand fragments of the two sub-steps (the rows of a
    // wavefront's blocks are 16 apart, which leaves the swizzle term alone) and the global offsets of the lanes' 16
    // bytes in the wavefront's eight 1 KB blocks of a tile (lane l lands at byte 16 * l of its block, i.e. row l / 8,
    // unit slot l % 8, and fetches the unit that belongs there)
    int aa[2], ab[2], vo[8];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int sw = ((s * 4 + (lane >> 4)) ^ (((lane & 15) >> 1) & 7)) * 16;
      aa[s] = (wm * 128 + (lane & 15)) * 128 + sw;
      ab[s] = (wn * 128 + (lane & 15)) * 128 + sw;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = (wave * 8 + i) * 8 + (lane >> 3);
      vo[i] = row * row_bytes + (((lane & 7) ^ ((row >> 1) & 7)) * 16);
    }
    asm volatile(MSA_SCAN4_SET_ADDR ::"v"(aa[0]), "v"(aa[1]), "v"(ab[0]), "v"(ab[1]) : MSA_SCAN4_CLOBBERS);
    asm volatile(MSA_SCAN4_SET_VOFF ::"v"(vo[0]), "v"(vo[1]), "v"(vo[2]), "v"(vo[3]), "v"(vo[4]), "v"(vo[5]), "v"(vo[6]), "v"(vo[7])
                 : MSA_SCAN4_CLOBBERS);
    // v222: byte offset of a lane's column in a run of 64 document ids; v223: the pool counter's increment
    asm volatile("v_lshlrev_b32 v222, 2, %0\n\tv_mov_b32 v223, 1" ::"v"(lane) : MSA_SCAN4_CLOBBERS);
    asm volatile(MSA_SCAN4_SET_FOLD ::"v"(l32) : MSA_SCAN4_CLOBBERS);
  }
  const char* ga = reinterpret_cast<const char*>(qs);
  const char* gb = reinterpret_cast<const char*>(kr);
  // One resource per operand tile whose extent is the valid part of the tile: rows past M_rows / C read as zero in
  // hardware (the range check is on the vector offset, where the row displacement rides; the K displacement is
  // scalar and stays inside the row).  A tile that does not exist gets an empty extent: its loads fetch nothing.
  auto make_a = [&](int tm, bool valid) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(ga) + (valid ? (int64_t)tm * BM * row_bytes : 0), 0,
                                             valid ? min(BM, M_rows - tm * BM) * row_bytes : 0, 0x00020000);
  };
  auto make_b = [&](int tn, bool valid) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(gb) + (valid ? (int64_t)tn * BN * row_bytes : 0), 0,
                                             valid ? min(BN, C - tn * BN) * row_bytes : 0, 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t rsrc_docs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(kDocMax ? chunk_doc : nullptr), 0, kDocMax ? C * 4 : 0, 0x00020000);

  // The workgroup's tiles: `cur` is multiplied, `nxt` is the one behind it (the loads enter it two K steps before the
  // MFMAs do).  Own tiles first, then pool draws.
  int tm_c, tn_c, tm_n = 0, tn_n = 0, own_idx = 0;
  ScanWalkCursor cursor = scan_walk_cursor(walk);
  scan_walk_cursor_tile(walk, cursor, tm_c, tn_c);
  __amdgpu_buffer_rsrc_t ra_c = make_a(tm_c, true), rb_c = make_b(tn_c, true), ra_n, rb_n;
  bool nxt_valid = false, nxt_pending = false;
  auto plan_next = [&]() {
    nxt_valid = own_idx + 1 < walk.own_count;
    nxt_pending = !nxt_valid && pool_n > 0;
    if (nxt_valid) {
      ++own_idx;
      scan_walk_cursor_next(walk, cursor);
      scan_walk_cursor_tile(walk, cursor, tm_n, tn_n);
    }
    ra_n = make_a(tm_n, nxt_valid);
    rb_n = make_b(tn_n, nxt_valid);
  };
  plan_next();
  uint32_t* const pool_counter = sched;
  uint32_t* const my_claim = sched + kSchedCounterWords + blockIdx.x;
  const bool drawer = wave == 0;
  const uint32_t zero_off = 0;

  // ---- epilogue state: see score_gemm_kernel's epilogue, of which this is the form with four row blocks ----
  const int n_queries = M_rows / (blocks_per_query * kUnit);
  typedef const __attribute__((address_space(4))) uint32_t* const_words_t;      // scalar loads
  const const_words_t row_bits_c = (const_words_t)row_bits;
  // floor(2^32 / d) + 1 divides exactly while n * d < 2^32 (row blocks < 2^19, blocks per query <= 2^11; units < 2^21, a query's <= 2^7)
  const uint32_t bpq_magic = (uint32_t)(0x100000000ull / (uint32_t)blocks_per_query) + 1u;
  uint32_t rbits[4] = {0u, 0u, 0u, 0u};
  int q_first = 0, r_first = 0;
  auto fetch_rows = [&](int m0) {
    const int blk0 = (m0 + wm * 128) >> 5;
#pragma unroll
    for (int i = 0; i < 4; ++i) rbits[i] = row_bits_c[blk0 + i];          // 0 past M_rows (the buffer is padded)
    const int first = (m0 + wm * 128) / kUnit;
    q_first = blocks_per_query == 1 ? first : (int)__umulhi((uint32_t)first, bpq_magic);     // first / blocks_per_query
    r_first = first - q_first * blocks_per_query;
  };
  // the documents of the wavefront's 128 columns, 64 per load, into v220 / v221 (v216: their offsets): requested in
  // front of a K step (whose waits cover them), read when the tile's maxima are folded; columns past the bank read 0
  // and are masked below
  auto fetch_docs = [&](int n0) {
    if constexpr (kDocMax) {
      const int first = (n0 + wn * 128) * 4;      // (in the vector offset, which is what the extent is checked against)
      asm volatile("s_nop 4\n\tv_add_u32 v216, %1, v222\n\tbuffer_load_dword v220, v216, %0, 0 offen\n\t"
                   "buffer_load_dword v221, v216, %0, 0 offen offset:256"
                   ::"s"(rsrc_docs), "s"(first) : MSA_SCAN4_CLOBBERS);
    }
  };
  // Folds the finished tile's block maxima (v224 - v239, left by the reduction that rides in the next tile's first K
  // step or by the stand-alone one): row blocks of one query are joined, and at a query's end the two pairs of column
  // blocks are merged into the key plane.  Every row of a scored block counts (the prologue kernel made unscored rows
  // repeat a scored one); a block whose mask word is zero belongs to a query without scored tokens or to the padding
  // past M_rows and is skipped.
  auto fold_tile = [&](int n0) {
    float mx[8];
#define MSA_SCAN4_READ8(TEXT)                                                                                                     \
    asm volatile(TEXT : "=v"(mx[0]), "=v"(mx[1]), "=v"(mx[2]), "=v"(mx[3]), "=v"(mx[4]), "=v"(mx[5]), "=v"(mx[6]), "=v"(mx[7]))
    const int n_first = n0 + wn * 128 + lane;      // the lane's columns: this one and the 64th behind it
    DocRuns runs[2];
    if constexpr (kDocMax) {
      int doc0, doc1;
      asm volatile("v_mov_b32 %0, v220\n\tv_mov_b32 %1, v221" : "=v"(doc0), "=v"(doc1));
      runs[0] = doc_runs(n_first < C ? doc0 : -1 - l32, n_first < C, half, l32);
      runs[1] = doc_runs(n_first + 64 < C ? doc1 : -1 - l32, n_first + 64 < C, half, l32);
    }
    float run[2] = {-INFINITY, -INFINITY};
    bool any = false;
    int run_q = q_first, r = r_first;
    auto emit = [&]() {
      if (!any || run_q >= n_queries) return;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        if constexpr (kDocMax) merge_runs(runs[p], run[p], out_key + (int64_t)run_q * n_docs, true);
        else if (n_first + 64 * p < C) atomicMax(&out_key[(int64_t)run_q * C + n_first + 64 * p], f32_to_key(run[p]));
      }
    };
    if constexpr (kUnits) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (i == 0) MSA_SCAN4_READ8(MSA_SCAN4_UNIT_READ_0);
        if (i == 1) MSA_SCAN4_READ8(MSA_SCAN4_UNIT_READ_1);
        if (i == 2) MSA_SCAN4_READ8(MSA_SCAN4_UNIT_READ_2);
        if (i == 3) MSA_SCAN4_READ8(MSA_SCAN4_UNIT_READ_3);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (r == blocks_per_query) {                     // the unit opens the next query
            emit();
            run[0] = run[1] = -INFINITY;
            any = false; ++run_q; r = 0;
          }
          ++r;
          if (rbits[i] >> (8 * u) & 0xffu) {
            any = true;
            run[0] = fmaxf(run[0], mx[u]);
            run[1] = fmaxf(run[1], mx[4 + u]);
          }
        }
      }
      emit();
      return;
    }
    MSA_SCAN4_READ8(MSA_SCAN4_MAX_READ);
#undef MSA_SCAN4_READ8
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (r == blocks_per_query) {                         // row block i opens the next query
        emit();
        run[0] = run[1] = -INFINITY;
        any = false; ++run_q; r = 0;
      }
      ++r;
      if (rbits[i] != 0) {
        any = true;
        run[0] = fmaxf(run[0], mx[2 * i]);
        run[1] = fmaxf(run[1], mx[2 * i + 1]);
      }
    }
    emit();
  };

  // ---- prologue: the first two K tiles of the first tile, the first fragments ----
  const int woff = wave * 8192;
  int sa = 0, sb = 0x10000;
  asm volatile(MSA_SCAN4_LOAD8_NT ::[dst] "s"(0x10000 + woff), [r] "s"(rb_c), [k] "s"(0) : MSA_SCAN4_CLOBBERS);
  asm volatile(MSA_SCAN4_LOAD8 ::[dst] "s"(0 + woff), [r] "s"(ra_c), [k] "s"(0) : MSA_SCAN4_CLOBBERS);
  asm volatile(MSA_SCAN4_LOAD8_NT ::[dst] "s"(0x18000 + woff), [r] "s"(rb_c), [k] "s"(kRowBytes) : MSA_SCAN4_CLOBBERS);
  asm volatile(MSA_SCAN4_LOAD8 ::[dst] "s"(0x8000 + woff), [r] "s"(ra_c), [k] "s"(kRowBytes) : MSA_SCAN4_CLOBBERS);
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  asm volatile(MSA_SCAN4_FRAGS0 ::[sa] "s"(sa), [sb] "s"(sb) : MSA_SCAN4_CLOBBERS);

  // A tile's accumulators are reduced inside the next tile's first K step and folded right behind it, so the fold of
  // tile t uses the row words and the documents fetched for t; those of t + 1 are requested once it is done.
  bool have_prev = false;
  int prev_n0 = 0;
  for (;;) {
    // Step kt requests K tile kt + 2: of this tile while it has one, of the next tile after that.  The steps are laid
    // out so that between two of them the scalar unit has next to nothing to do (a wavefront that is alone on its SIMD
    // pays for every instruction between two MFMAs): the resources a step reads are fixed per loop, and the tile
    // pool's hops ride in front of four peeled steps.
#define MSA_SCAN4_STEP_CLOBBERS(TEXT, RA, RB, KOFF, ...)                                                     \
    asm volatile(TEXT : [sa] "+s"(sa), [sb] "+s"(sb)                                                         \
                 : [ra] "s"(RA), [rb] "s"(RB), [k] "s"(KOFF), [woff] "s"(woff) : __VA_ARGS__)
#define MSA_SCAN4_STEP(TEXT, RA, RB, KOFF) MSA_SCAN4_STEP_CLOBBERS(TEXT, RA, RB, KOFF, MSA_SCAN4_CLOBBERS)
    const bool pending = nxt_pending;      // the tile behind this one comes from the pool (k_tiles >= 6 then)
    if (pending && drawer && lane == 0)    // v217 = counter++
      asm volatile("s_nop 4\n\tglobal_atomic_add v217, %0, v223, %1 sc0" ::"v"(zero_off), "s"(pool_counter) : "memory");
    // What the finished tile left is reduced inside this tile's first step.  Usually the wavefront's four row blocks
    // are one query whose rows all count (blocks_per_query a multiple of 4: queries of 128, 256, ... padded tokens) and
    // the tile lies inside the bank: then the step also folds the maxima into the key plane.  Otherwise it leaves one
    // maximum per block and fold_tile() does the rest; a wavefront whose rows are all padding has nothing to fold.
    const bool fold_any = have_prev && (rbits[0] | rbits[1] | rbits[2] | rbits[3]) != 0;
    const bool fold_fast = kDocMax && !kUnits && fold_any && (blocks_per_query & 3) == 0 && rbits[0] != 0 && prev_n0 + BN <= C;
    if (fold_fast) {
      const uint32_t* okey = out_key + (int64_t)q_first * n_docs;
      if (k_tiles > 2)
        asm volatile(MSA_SCAN4_KSTEP_FRESH_FOLD : [sa] "+s"(sa), [sb] "+s"(sb)
                     : [ra] "s"(ra_c), [rb] "s"(rb_c), [k] "s"(2 * kRowBytes), [woff] "s"(woff), [okey] "s"(okey) : MSA_SCAN4_CLOBBERS);
      else
        asm volatile(MSA_SCAN4_KSTEP_FRESH_FOLD : [sa] "+s"(sa), [sb] "+s"(sb)
                     : [ra] "s"(ra_n), [rb] "s"(rb_n), [k] "s"(0), [woff] "s"(woff), [okey] "s"(okey) : MSA_SCAN4_CLOBBERS);
    } else if (kUnits && fold_any) {
      if (k_tiles > 2) MSA_SCAN4_STEP_CLOBBERS(MSA_SCAN4_KSTEP_FRESH_UNITS, ra_c, rb_c, 2 * kRowBytes, MSA_SCAN4_UNITS_CLOBBERS);
      else MSA_SCAN4_STEP_CLOBBERS(MSA_SCAN4_KSTEP_FRESH_UNITS, ra_n, rb_n, 0, MSA_SCAN4_UNITS_CLOBBERS);
      fold_tile(prev_n0);
    } else if (fold_any) {
      if (k_tiles > 2) MSA_SCAN4_STEP(MSA_SCAN4_KSTEP_FRESH_REDUCE, ra_c, rb_c, 2 * kRowBytes);
      else MSA_SCAN4_STEP(MSA_SCAN4_KSTEP_FRESH_REDUCE, ra_n, rb_n, 0);
      fold_tile(prev_n0);
    } else {
      if (k_tiles > 2) MSA_SCAN4_STEP(MSA_SCAN4_KSTEP_FRESH, ra_c, rb_c, 2 * kRowBytes);
      else MSA_SCAN4_STEP(MSA_SCAN4_KSTEP_FRESH, ra_n, rb_n, 0);
    }
    const int n0 = tn_c * BN;
    fetch_rows(tm_c * BM);
    fetch_docs(n0);
    int kt = 1;
    if (pending) {
      if (drawer && lane == 0)           // claim word = v217; its old value comes back in v218
        asm volatile("s_nop 4\n\tglobal_atomic_swap v218, %0, v217, %1 sc0" ::"v"(zero_off), "s"(my_claim) : "memory");
      MSA_SCAN4_STEP(MSA_SCAN4_KSTEP, ra_c, rb_c, 3 * kRowBytes);
      // every wavefront reads the word back (past the L1: device scope)
      asm volatile("s_nop 4\n\tglobal_load_dword v219, %0, %1 sc1" ::"v"(zero_off), "s"(my_claim) : "memory");
      MSA_SCAN4_STEP(MSA_SCAN4_KSTEP, ra_c, rb_c, 4 * kRowBytes);
      int p_next;                        // complete since the last step's wait
      asm volatile("v_readfirstlane_b32 %0, v219" : "=s"(p_next));
      nxt_pending = false;
      nxt_valid = p_next < walk.pool_total;
      if (nxt_valid) scan_walk_pool(walk, p_next, tm_n, tn_n);
      ra_n = make_a(tm_n, nxt_valid);
      rb_n = make_b(tn_n, nxt_valid);
      MSA_SCAN4_STEP(MSA_SCAN4_KSTEP, ra_c, rb_c, 5 * kRowBytes);
      kt = 4;
    }
    for (int k_l = (kt + 2) * kRowBytes; k_l < row_bytes; k_l += kRowBytes) MSA_SCAN4_STEP(MSA_SCAN4_KSTEP, ra_c, rb_c, k_l);
    for (int k_l = k_tiles > 2 ? 0 : kRowBytes; k_l < 2 * kRowBytes; k_l += kRowBytes) MSA_SCAN4_STEP(MSA_SCAN4_KSTEP, ra_n, rb_n, k_l);
#undef MSA_SCAN4_STEP
#undef MSA_SCAN4_STEP_CLOBBERS
    have_prev = true;
    prev_n0 = n0;
    if (!nxt_valid) break;
    tm_c = tm_n; tn_c = tn_n;
    ra_c = ra_n; rb_c = rb_n;
    plan_next();
  }
  if constexpr (kUnits) asm volatile(MSA_SCAN4_REDUCE_UNITS ::: MSA_SCAN4_UNITS_CLOBBERS);
  else asm volatile(MSA_SCAN4_REDUCE ::: MSA_SCAN4_CLOBBERS);
  fold_tile(prev_n0);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#endif
}

#define MSA_SCAN4_PARAMS                                                                                                          \
  const bf16_t *__restrict__ qs, const bf16_t *__restrict__ kr, const uint32_t *__restrict__ row_bits, uint32_t *__restrict__ out_key, \
      const int32_t *__restrict__ chunk_doc, int32_t M_rows, int32_t C, int32_t K, int32_t per_query, int32_t tiles_m, int32_t tiles_n, \
      int32_t m_group, int32_t n_docs, GatherJob job, uint32_t *__restrict__ sched, int32_t pool_n
template <bool kDocMax>
__global__ __launch_bounds__(256) __attribute__((amdgpu_num_vgpr(kScan4CompilerVgprs))) void score_scan4_kernel(MSA_SCAN4_PARAMS) {
  scan4_body<kDocMax, false>(qs, kr, row_bits, out_key, chunk_doc, M_rows, C, K, per_query, tiles_m, tiles_n, m_group, n_docs, job, sched, pool_n);
}
__global__ __launch_bounds__(256) __attribute__((amdgpu_num_vgpr(kScan4UnitsVgprs))) void score_scan4_units_kernel(MSA_SCAN4_PARAMS) {
  scan4_body<true, true>(qs, kr, row_bits, out_key, chunk_doc, M_rows, C, K, per_query, tiles_m, tiles_n, m_group, n_docs, job, sched, pool_n);
}
#undef MSA_SCAN4_PARAMS

// chunk_key -> fp32 scores (times scale / Hq); key 0 (query without a scored token) -> -inf.
__global__ void decode_scores_kernel(const uint32_t* __restrict__ key, int64_t n, float mul,
                                     float* __restrict__ out) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const uint32_t k = key[i];
    out[i] = k == 0 ? -INFINITY : key_to_f32(k) * mul;
  }
}

// ------------------------------------------------------------------------------------------
// fp32 banks of few chunks, or few query rows.  Tiles of 128 x 128 give a bank of 8000 chunks to 63 workgroups, each of which
// multiplies 1024-deep products at a compute unit's fp32 rate alone (57 us a tile, also where half of its rows are padding).  Here
// a workgroup owns 32 chunks and its four wavefronts a quarter of K each: a wavefront's share of the K_r rows stays in 128 of its
// registers for the whole launch, the query rows follow a 32-row block at a time, and the four partial blocks meet in LDS behind one
// barrier per block, where the rows' maximum is taken.  Column maxima of a query wait in LDS and are merged into the key plane at the end.
// K_r and query rows come through a ring of stages of a cache line of 32 rows, direct loads of eight whole lines: an MFMA operand
// loaded from memory touches 32 lines an instruction, 32 bytes each, and the address unit takes four times as long over it.  What
// bounds it: the matrix cores' fp32 rate (256 FLOP a cycle and compute unit) and, with few rows, the launch and the first loads.
// Whole routing calls, us, operands from memory and through the ring: 8000 chunks x 64 rows 30.7 and 26.4, 512 x 64 20.4 and 17.9,
// 64000 x 64 123 and 106, 128000 x 32 178 and 157, 8000 x 512 85 and 83.
// ------------------------------------------------------------------------------------------
constexpr int kSplitK = 1024, kSplitWaves = 4, kSplitCols = 32, kSplitMaxBlocks = 32;
constexpr int kSplitSlab = 32 * 128;           // a stage of a wavefront's ring: 32 rows, a cache line (32 values of K) each
constexpr int split_lds_bytes(int ring) {
  return kSplitWaves * ring * kSplitSlab + (2 * kSplitWaves * 32 + kSplitMaxBlocks) * kSplitCols * 4;
}
static_assert(split_lds_bytes(6) <= 160 * 1024 && 2 * split_lds_bytes(2) <= 160 * 1024);

// Four 1 KB blocks straight into LDS, as an asm statement so that the compiler does not drain what is in flight in front of its own LDS
// reads; the kernel counts.  M0 is put back as it was.
__device__ __forceinline__ void request_slab(__amdgpu_buffer_rsrc_t rsrc, uint32_t lds_dst, const int (&at)[4], int soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  uint32_t saved_m0;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 4\n\t"
      "buffer_load_dwordx4 %2, %6, %7 offen lds\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %3, %6, %7 offen lds\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %4, %6, %7 offen lds\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %5, %6, %7 offen lds\n\ts_mov_b32 m0, %0"
      : "=&s"(saved_m0) : "s"(lds_dst), "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "s"(rsrc), "s"(soff) : "scc", "memory");
#endif
}

// The maxima `best` of `queries` queries from q0 on, in the columns from n0 on, into the key plane.
template <bool kDocMax>
__device__ __forceinline__ void merge_best(uint32_t (*best)[kSplitCols], int queries, int q0, int n0, int C, int n_docs, int wave, int waves,
                                           uint32_t* __restrict__ out_key, int32_t own_doc) {
  const int lane = threadIdx.x & 63, l32 = lane & 31;
  for (int base = wave * 64; base < queries * kSplitCols; base += waves * 64) {              // 32 lanes a query
    const int i = base + lane, n = n0 + l32;
    const bool in = i < queries * kSplitCols && n < C;
    uint32_t key = in ? best[i / kSplitCols][l32] : 0u;
    const int64_t row = q0 + i / kSplitCols;
    if constexpr (kDocMax) {
      // a document's chunks are neighbours: the first of its columns here takes their maximum (one atomic each would queue up where a
      // few long documents meet many row blocks: 500 chunks of 16 documents x 1000 rows 215 us instead of 41)
      const int32_t doc = in ? own_doc : -1;
#pragma unroll
      for (int o = 1; o < kSplitCols; o <<= 1) {
        const uint32_t other = __shfl_down(key, o, kSplitCols);
        const int32_t other_doc = __shfl_down(doc, o, kSplitCols);
        if (l32 + o < kSplitCols && other_doc == doc) key = max(key, other);
      }
      const bool first = __shfl_up(doc, 1, kSplitCols) != doc || l32 == 0;
      if (in && first && key != 0) atomicMax(&out_key[row * n_docs + doc], key);
    } else {
      if (in && key != 0) atomicMax(&out_key[row * C + n], key);
    }
  }
}

template <bool kDocMax, int kRing>
__global__ __launch_bounds__(kSplitWaves * 64, 2) void score_split_kernel(const float* __restrict__ qs, const float* __restrict__ kr,
                                                                        const uint32_t* __restrict__ row_bits,
                                                                        uint32_t* __restrict__ out_key,
                                                                        const int32_t* __restrict__ chunk_doc, int32_t M_rows,
                                                                        int32_t C, int32_t blocks_per_query, int32_t n_docs,
                                                                        int32_t blocks_per_wg) {
  constexpr int kRow = kSplitK * (int)sizeof(float), kSlice = kRow / kSplitWaves, kStages = kSlice / 128;
  static_assert(kStages == 8, "stages alternate between two register buffers");
  extern __shared__ __align__(16) char lds[];
  char* const shared = lds + kSplitWaves * kRing * kSplitSlab;
  float(*part)[kSplitWaves][32 * kSplitCols] = reinterpret_cast<float(*)[kSplitWaves][32 * kSplitCols]>(shared);
  uint32_t(*best)[kSplitCols] = reinterpret_cast<uint32_t(*)[kSplitCols]>(shared + 2 * kSplitWaves * 32 * kSplitCols * 4);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int n0 = blockIdx.x * kSplitCols, blocks = M_rows >> 5;
  if (n0 >= C) return;                                   // (the grid's columns are a multiple of eight)
  const int b0 = blockIdx.y * blocks_per_wg, b1 = min(blocks, b0 + blocks_per_wg);
  char* const ring = lds + wave * kRing * kSplitSlab;
  const uint32_t ring_at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)ring);
  // a load's lanes take eight rows, eight 16-byte units each; unit u of row r lies at u ^ (r & 7)
  int at[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) at[i] = (8 * i + (lane >> 3)) * kRow + wave * kSlice + (((lane & 7) ^ (lane >> 3)) * 16);
  // what is requested next: stage `stage` of the K_r rows, then of one block of query rows after another (behind the last, zeros
  // through an empty extent)
  int stage = 0, req_blk = b0 - 1, req_slot = 0, slot = 0;
  __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(reinterpret_cast<const char*>(kr)) + (int64_t)n0 * kRow, 0, min(kSplitCols, C - n0) * kRow, 0x00020000);
  auto request = [&]() {
    request_slab(rs, ring_at + req_slot * kSplitSlab, at, stage * 128);
    req_slot = req_slot + 1 == kRing ? 0 : req_slot + 1;
    if (++stage == kStages) {
      stage = 0;
      ++req_blk;
      rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(qs)) + (int64_t)min(req_blk, blocks - 1) * 32 * kRow,
                                             0, req_blk < b1 ? 32 * kRow : 0, 0x00020000);
    }
  };
  auto wait_for = [&](auto younger_tag) {        // all stages but the `younger` newest have arrived
    constexpr int n = 4 * decltype(younger_tag)::value;
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
    asm volatile("" ::: "memory");
  };
  int unit[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) unit[c] = l32 * 128 + (((2 * c + half) ^ (l32 & 7)) * 16);
  auto read = [&](u32x4_t* to) {
#pragma unroll
    for (int c = 0; c < 4; ++c) to[c] = *reinterpret_cast<const u32x4_t*>(ring + slot * kSplitSlab + unit[c]);
    slot = slot + 1 == kRing ? 0 : slot + 1;
  };
  u32x4_t k[4 * kStages], q[2][4];
#pragma unroll
  for (int i = 0; i < kRing; ++i) request();
  const int q0 = b0 / blocks_per_query;
  const int32_t own_doc = kDocMax ? chunk_doc[min(n0 + l32, C - 1)] : 0;
  for (int i = tid; i < kSplitMaxBlocks * kSplitCols; i += kSplitWaves * 64) best[i / kSplitCols][i % kSplitCols] = 0u;
#pragma unroll
  for (int i = 0; i < kStages; ++i) {
    wait_for(std::integral_constant<int, kRing - 1>{});
    read(k + 4 * i);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // the slot may be requested again
    request();
  }
  wait_for(std::integral_constant<int, kRing - 1>{});
  read(q[0]);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  request();
  int query = q0, in_query = b0 - q0 * blocks_per_query;
  for (int blk = b0; blk < b1; ++blk) {
    const uint32_t bits = row_bits[blk];                 // all rows of a block are scored, or none (presum_queries_kernel)
    floatx16_t acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.f;
#pragma unroll
    for (int i = 0; i < kStages; ++i) {                  // stage i's products beside the reads of the one behind it
      wait_for(std::integral_constant<int, kRing - 1>{});
      read(q[(i + 1) & 1]);
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int x = 0; x < 4; ++x)
          acc = Mma<float>::mma(__uint_as_float(q[i & 1][c][x]), __uint_as_float(k[4 * i + c][x]), acc);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      request();
    }
    // acc[e] is (row 8 * (e / 4) + 4 * half + e % 4, column l32) over this wavefront's quarter of K
    float(*p)[32 * kSplitCols] = part[blk & 1];
#pragma unroll
    for (int e = 0; e < 16; ++e) p[wave][(8 * (e >> 2) + 4 * half + (e & 3)) * kSplitCols + l32] = acc[e];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    float top = -INFINITY;                               // of four rows; the other half of the wavefront has four more
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = ((tid >> 5) * 4 + r) * kSplitCols + l32;
      top = fmaxf(top, (p[0][i] + p[1][i]) + (p[2][i] + p[3][i]));
    }
    top = fmaxf(top, __shfl_xor(top, 32));
    if (bits != 0 && half == 0) atomicMax(&best[query - q0][l32], f32_to_key(top));
    if (++in_query == blocks_per_query) {
      in_query = 0;
      ++query;
    }
  }
  __builtin_amdgcn_s_waitcnt(0);                         // (nothing in flight when the workgroup ends)
  __syncthreads();
  merge_best<kDocMax>(best, b1 > b0 ? (b1 - 1) / blocks_per_query - q0 + 1 : 0, q0, n0, C, n_docs, wave, kSplitWaves, out_key, own_doc);
}

// ------------------------------------------------------------------------------------------
// fp32 banks of up to 32 chunks a compute unit: the same split of the work, the products on the bf16 matrix cores.  An fp32 value is
// three bf16 ones exactly, and of the nine products of two values the six largest are formed: 192 cycles where the fp32 form takes 512.  What
// is left out is up to 2^-24 of a product (the second parts times the third ones), 2^-27 in the mean: with its own rounding a product is within
// 2^-23 where the fp32 instruction gives 2^-24.  (First parts cut off instead of rounded: 2^-21.8.  Eight products, 2^-24: 8192 chunks x 1024
// rows 127 -> 141 us, 1000 x 64 16.6 -> 17.1.)  Values below 2^-109 lose their last parts.  Errors of 8000 chunks x 64 rows against float64, all scores: 5.8e-8 of
// their norm, 1.7e-7 there.  Eight wavefronts hold an eighth of K each, of their 32 chunks in three parts in 96 registers; the
// queries come as operands from the prologue (part_at), a kilobyte a load, four steps of K ahead.  The first parts' products and the
// others' have sums of their own, so that small ones are not rounded away one by one.  What bounds it: K_r from memory with few rows
// (8000 chunks x 64 rows 15.6 -> 13.5 us, the first block multiplied as it arrives; 13.9 with all four slabs requested at once), and
// the operands' way from the L2 with many, 196 KB a block, which takes twice the 1.4 us that the products do (half of it would want
// 64 chunks a workgroup, whose parts the registers do not hold).  An infinity among the values makes NaN where parts of different
// sign meet, so a sum that is NaN is formed again value by value, by a whole wavefront: once a NaN chunk or query row, which end there, once a
// row for a chunk with an infinity.  Calls of 8000 chunks x 64 rows, one chunk with a NaN, with an infinity, all queries NaN: 28, 40 and 49 us, 26 without
// (a lane for each sum, value after value: 206, 212 and 328).
// ------------------------------------------------------------------------------------------
constexpr int kPartsWaves = 8, kPartsSlabs = 4, kPartsMaxRows = 1024;
constexpr int kPartsLds = kPartsWaves * kPartsSlabs * kSplitSlab + kSplitMaxBlocks * kSplitCols * 4;
static_assert(kPartsLds <= 160 * 1024 && 2 * kPartsWaves * 32 * kSplitCols * 4 <= kPartsWaves * kPartsSlabs * kSplitSlab, "partial sums take the slabs' place");

// Sixteen values of a query, put together from their parts, times as many of a chunk: a lane's share of a sum that is formed again.
struct ValuesDot {
  float sum = 0.f;
  bool query_nan = false, key_nan = false;
  __device__ __forceinline__ ValuesDot(const char* qp, const float* kr) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint4 w[3];
#pragma unroll
      for (int n = 0; n < 3; ++n) w[n] = *reinterpret_cast<const uint4*>(qp + h * 512 + n * kPartBytes);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        auto piece = [&](int n) {
          const uint32_t u = e < 2 ? w[n].x : e < 4 ? w[n].y : e < 6 ? w[n].z : w[n].w;
          return e & 1 ? bf16hi(u) : bf16lo(u);
        };
        const float x = piece(0) + (piece(1) + piece(2)), y = kr[8 * h + e];
        query_nan |= x != x;
        key_nan |= y != y;
        sum += x * y;
      }
    }
  }
};

template <bool kDocMax>
__global__ __launch_bounds__(kPartsWaves * 64) void score_parts_kernel(const char* __restrict__ qs, const float* __restrict__ kr,
                                                                      const uint32_t* __restrict__ row_bits, uint32_t* __restrict__ out_key,
                                                                      const int32_t* __restrict__ chunk_doc, int32_t M_rows, int32_t C,
                                                                      int32_t blocks_per_query, int32_t n_docs, int32_t blocks_per_wg) {
  typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 operand_t;
  constexpr int kRow = kSplitK * (int)sizeof(float), kSlice = kRow / kPartsWaves, kSteps = kSplitK / kPartsWaves / 16, kAhead = 4;
  static_assert(kSlice == kPartsSlabs * 128 && kSteps == 2 * kPartsSlabs && kSteps % kAhead == 0 && kPartsSlabs == 4, "a wavefront's share of K");
  extern __shared__ __align__(16) char lds[];
  float(*part)[kPartsWaves][32 * kSplitCols] = reinterpret_cast<float(*)[kPartsWaves][32 * kSplitCols]>(lds);
  uint32_t(*best)[kSplitCols] = reinterpret_cast<uint32_t(*)[kSplitCols]>(lds + kPartsWaves * kPartsSlabs * kSplitSlab);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int n0 = blockIdx.x * kSplitCols, blocks = M_rows >> 5;
  if (n0 >= C) return;                                   // (the grid's columns are a multiple of eight)
  const int b0 = blockIdx.y * blocks_per_wg, b1 = min(blocks, b0 + blocks_per_wg);
  const int32_t own_doc = kDocMax ? chunk_doc[min(n0 + l32, C - 1)] : 0;

  // The first operands, then the chunks' rows, a slab of every wavefront before the next ones: the requests are taken up as fast as memory
  // answers, and the last wavefront's first slab would come behind all of the others'.
  const __amdgpu_buffer_rsrc_t rs_q = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(qs) + (int64_t)b0 * (kSplitK / 16) * kPartStep, 0,
                                                                        (b1 - b0) * (kSplitK / 16) * kPartStep, 0x00020000);
  u32x4_t q[kAhead][3];
  auto request_q = [&](u32x4_t (&to)[3], int blk, int step) {          // (of a block behind the last: zeros)
#pragma unroll
    for (int p = 0; p < 3; ++p)
      to[p] = __builtin_amdgcn_raw_buffer_load_b128(rs_q, lane * 16 + ((blk - b0) * (kSplitK / 16) + wave * kSteps + step) * kPartStep + p * kPartBytes, 0, 0);
  };
#pragma unroll
  for (int i = 0; i < kAhead; ++i) request_q(q[i], b0, i);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  char* const slabs = lds + wave * kPartsSlabs * kSplitSlab;
  const uint32_t slabs_at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)slabs);
  int at[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) at[i] = (8 * i + (lane >> 3)) * kRow + wave * kSlice + (((lane & 7) ^ (lane >> 3)) * 16);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(reinterpret_cast<const char*>(kr)) + (int64_t)n0 * kRow, 0, min(kSplitCols, C - n0) * kRow, 0x00020000);
  auto request_k = [&](int i) { request_slab(rs, slabs_at + i * kSplitSlab, at, i * 128); };
  request_k(0);
  __builtin_amdgcn_s_barrier();
  request_k(1);
  __builtin_amdgcn_s_barrier();
  request_k(2);
  const int q0 = b0 / blocks_per_query;
  for (int i = tid; i < kSplitMaxBlocks * kSplitCols; i += kPartsWaves * 64) best[i / kSplitCols][i % kSplitCols] = 0u;

  u32x4_t k[kSteps][3];
  floatx16_t big, small;
  auto clear = [&]() {
#pragma unroll
    for (int e = 0; e < 16; ++e) big[e] = small[e] = 0.f;
  };
  auto multiply = [&](int i, int blk) {                  // a step of K; what is kAhead steps on takes its operands' registers
    u32x4_t(&a)[3] = q[i % kAhead];
    auto mul = [&](int x, int y, floatx16_t c) {
      return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(operand_t, a[x]), __builtin_bit_cast(operand_t, k[i][y]), c, 0, 0, 0);
    };
    small = mul(0, 1, small);
    big = mul(0, 0, big);
    small = mul(1, 0, small);
    small = mul(1, 1, small);
    small = mul(0, 2, small);
    small = mul(2, 0, small);
    request_q(a, blk + (i + kAhead) / kSteps, (i + kAhead) % kSteps);
  };
  clear();
  auto take = [&](auto slab) {                           // once what is younger than the slab alone is outstanding: other slabs, operands
    constexpr int i = decltype(slab)::value, kOps = 6;
    constexpr int kYounger = i == 0 ? 8 : i == 1 ? 8 + kOps : i == 2 ? 4 + 2 * kOps : 2 * kOps;
    __builtin_amdgcn_s_waitcnt((kYounger & 15) | (kYounger >> 4 << 14) | (7 << 4) | (15 << 8));
    asm volatile("" ::: "memory");
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float x[8];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const u32x4_t w = *reinterpret_cast<const u32x4_t*>(slabs + i * kSplitSlab + l32 * 128 + (((4 * h + 2 * half + c) ^ (l32 & 7)) * 16));
#pragma unroll
        for (int e = 0; e < 4; ++e) x[4 * c + e] = __uint_as_float(w[e]);
      }
      uint4 parts[3];
      split_three<false>(x, parts);
#pragma unroll
      for (int p = 0; p < 3; ++p) k[2 * i + h][p] = __builtin_bit_cast(u32x4_t, parts[p]);
      multiply(2 * i + h, b0);
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);                   // (the operands' requests are counted)
  };
  take(std::integral_constant<int, 0>{});
  request_k(3);
  take(std::integral_constant<int, 1>{});
  take(std::integral_constant<int, 2>{});
  take(std::integral_constant<int, 3>{});
  __syncthreads();                                       // partial sums lie where the slabs were
  uint32_t nan_columns = 0;                              // chunks found to hold a NaN
  // sum e is (row 8 * (e / 4) + 4 * half + e % 4, column l32) over this wavefront's eighth of K
  for (int blk = b0; blk < b1; ++blk) {
    if (blk > b0) {
      clear();
#pragma unroll
      for (int i = 0; i < kSteps; ++i) multiply(i, blk);
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) part[(blk - b0) & 1][wave][(8 * (e >> 2) + 4 * half + (e & 3)) * kSplitCols + l32] = big[e] + small[e];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const uint32_t bits = row_bits[blk];                 // all rows of a block are scored, or none (presum_queries_kernel)
    const float(*p)[32 * kSplitCols] = part[(blk - b0) & 1];
    float top = -INFINITY;                               // of two rows; the other half of the wavefront has two more
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int row = (tid >> 5) * 2 + r, i = row * kSplitCols + l32;
      float v = ((p[0][i] + p[1][i]) + (p[2][i] + p[3][i])) + ((p[4][i] + p[5][i]) + (p[6][i] + p[7][i]));
      for (uint64_t again = __ballot(v != v && n0 + l32 < C && (nan_columns >> l32 & 1) == 0); again != 0;) {
        const int at = __builtin_ctzll(again);             // the lane whose sum is formed
        const ValuesDot dot(qs + part_at(32 * blk + wave * 4 + (at >> 5) * 2 + r, lane * 16, kSplitK), kr + (int64_t)(n0 + (at & 31)) * kSplitK + lane * 16);
        const float sum = lanes_sum(row16_sum(dot.sum));
        v = lane == at ? sum : v;
        again &= again - 1;
        if (__any(dot.query_nan)) again &= at < 32 ? ~0ull << 32 : 0ull;           // none of the row's sums is a number
        if (__any(dot.key_nan)) {
          nan_columns |= 1u << (at & 31);
          again &= ~(0x100000001ull << (at & 31));
        }
      }
      top = fmaxf(top, v);
    }
    top = fmaxf(top, __shfl_xor(top, 32));
    if (bits != 0 && half == 0) atomicMax(&best[blk / blocks_per_query - q0][l32], f32_to_key(top));
  }
  __syncthreads();
  merge_best<kDocMax>(best, b1 > b0 ? (b1 - 1) / blocks_per_query - q0 + 1 : 0, q0, n0, C, n_docs, wave, kPartsWaves, out_key, own_doc);
}

// Optional timing of the scoring kernel alone: event pairs recorded around its launch.  The lock makes the record
// list safe against concurrent callers; while timing is off a launch only reads one atomic flag.
struct KernelTimer {
  std::mutex mu;
  std::atomic<int> on{0};
  hipEvent_t* start = nullptr;
  hipEvent_t* stop = nullptr;
  int cap = 0;
  int n = 0;
} g_timer;

constexpr size_t kLdsPerCu = 160 * 1024;

// Compute units of the current device (asked once; the library drives one device per process).
int compute_units() {
  static const int n = [] {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      cus = 256;
    return cus;
  }();
  return n;
}

template <typename T, int BM, int BN, int WAVES_M, int WAVES_N, int kSets, bool kDocMax, bool kStream, int kUnit = 32>
int launch_gemm(const void* qs, const void* kr, const uint32_t* row_bits, uint32_t* out_key, const int32_t* chunk_doc,
                int32_t M_rows, int32_t C, int32_t K, int32_t units_per_query, int32_t n_docs, hipStream_t st) {
  const size_t lds = score_tile_is_direct_stream<T, BM, BN, kSets, kStream>() ? (size_t)kDtlStreamLdsBytes
                                                                               : (size_t)2 * (BM + BN) * kRowStride;
  const int tiles_m = (M_rows + BM - 1) / BM;
  const int tiles_n = (C + BN - 1) / BN;
  // M tiles are walked in groups of 8 per K_r tile: a group's query rows (4 MiB in bf16) are what an XCD's L2
  // holds.  At 8 M tiles that is all of them (groups of 1, 2, 4 lose 2-14 % there); with 16 M tiles groups of 8
  // measured 1.4 % faster than one group, with 256 (a 64k-row prefill batch) 4 %.
  const int m_group = std::min(tiles_m, 8);
  const int m_groups = (tiles_m + m_group - 1) / m_group;
  int grid = 8 * ((tiles_n + 7) / 8) * m_groups * m_group;
  if (kStream) {      // one workgroup per slot the compute units offer (LDS decides how many fit), each walking several tiles
    if (tiles_m != 1) {
      msa_set_error("score_gemm: the streaming form takes one M tile, got %d", tiles_m);
      return MSA_EINVAL;
    }
    grid = std::min(tiles_n, compute_units() * std::max<int>(1, (int)(kLdsPerCu / lds)));
  }
  auto kern = score_gemm_kernel<T, BM, BN, WAVES_M, WAVES_N, kSets, kDocMax, kStream, kUnit>;
  static std::atomic<int> lds_limit_raised{0};
  MSA_HIP(raise_dynamic_lds_limit(lds_limit_raised, reinterpret_cast<const void*>(kern), (int)lds));
  int slot = -1;
  if (g_timer.on.load(std::memory_order_acquire)) {
    std::lock_guard<std::mutex> lock(g_timer.mu);
    if (g_timer.n < g_timer.cap) slot = g_timer.n++;
  }
  if (slot >= 0) MSA_HIP(hipEventRecord(g_timer.start[slot], st));
  kern<<<grid, WAVES_M * WAVES_N * 64, lds, st>>>(static_cast<const T*>(qs), static_cast<const T*>(kr), row_bits, out_key,
                                                  chunk_doc, M_rows, C, K, units_per_query, tiles_m, tiles_n, m_group,
                                                  n_docs);
  MSA_LAUNCH_CHECK();
  if (slot >= 0) MSA_HIP(hipEventRecord(g_timer.stop[slot], st));
  return MSA_OK;
}

// As many workgroups along the query blocks as give every compute unit two, at most kSplitMaxBlocks blocks each.  Those of a column come
// a multiple of the XCDs behind one another, so that one L2 has its K_r rows for all of them; the columns that this adds end at once.  us a
// call, one workgroup a column and two: 8000 chunks x 64 rows 24.4 and 23.1, x 256 54.2 and 48.9, 6112 x 64 25.4 and 24.0 (two of 250 or
// 191 columns that meet in different L2s: 30.5, 55.1 and 27.4).
struct SplitGrid {
  int cols, per_wg, x, y;       // columns, blocks a workgroup; the grid
};
SplitGrid split_grid(int32_t C, int32_t M_rows) {
  const int cols = (C + kSplitCols - 1) / kSplitCols, blocks = M_rows / 32;
  const int want = std::min(blocks, std::max((blocks + kSplitMaxBlocks - 1) / kSplitMaxBlocks, 2 * compute_units() / cols));
  const int per_wg = (blocks + want - 1) / want;
  return {cols, per_wg, (cols + 7) / 8 * 8, (blocks + per_wg - 1) / per_wg};
}
template <bool kDocMax>
int launch_split(const void* qs, const void* kr, const uint32_t* row_bits, uint32_t* out_key, const int32_t* chunk_doc,
                 int32_t M_rows, int32_t C, int32_t blocks_per_query, int32_t n_docs, hipStream_t st) {
  const SplitGrid plan = split_grid(C, M_rows);
  const int cols = plan.cols, per_wg = plan.per_wg;
  const dim3 grid((unsigned)plan.x, (unsigned)plan.y);
  int slot = -1;
  if (g_timer.on.load(std::memory_order_acquire)) {
    std::lock_guard<std::mutex> lock(g_timer.mu);
    if (g_timer.n < g_timer.cap) slot = g_timer.n++;
  }
  if (slot >= 0) MSA_HIP(hipEventRecord(g_timer.start[slot], st));
  // one workgroup a compute unit: the deep ring; more: two of them with two slots a wavefront
  const bool one = (int64_t)cols * grid.y <= compute_units();
  const auto kern = one ? score_split_kernel<kDocMax, 6> : score_split_kernel<kDocMax, 2>;
  const int lds = split_lds_bytes(one ? 6 : 2);
  static std::atomic<int> lds_limit_raised[2] = {{0}, {0}};
  MSA_HIP(raise_dynamic_lds_limit(lds_limit_raised[one], reinterpret_cast<const void*>(kern), lds));
  kern<<<grid, kSplitWaves * 64, lds, st>>>(static_cast<const float*>(qs), static_cast<const float*>(kr), row_bits,
                                            out_key, chunk_doc, M_rows, C, blocks_per_query, n_docs, per_wg);
  MSA_LAUNCH_CHECK();
  if (slot >= 0) MSA_HIP(hipEventRecord(g_timer.stop[slot], st));
  return MSA_OK;
}

// Up to one workgroup a compute unit, those of a column a multiple of the XCDs behind one another (the columns that this adds count: 85
// columns in three rows of 88 leave five XCDs with a workgroup more than they have compute units).
SplitGrid parts_grid(int32_t C, int32_t M_rows) {
  const int cols = (C + kSplitCols - 1) / kSplitCols, blocks = M_rows / 32, x = (cols + 7) / 8 * 8;
  const int want = std::min(blocks, std::max(1, compute_units() / x)), per_wg = (blocks + want - 1) / want;
  return {cols, per_wg, x, (blocks + per_wg - 1) / per_wg};
}
// The line between the other fp32 forms: launch_gemm_for has its figures.
bool split_ok(int32_t C, int32_t M_rows) { return M_rows <= 64 || (int64_t)C * M_rows <= (int64_t)1 << 21; }
// Whether a call of fp32 queries takes score_parts_kernel.  A block costs a compute unit about 3.2 us there and 3.7 in score_split_kernel, which has
// two workgroups a unit and starts 1.3 us later; parts of queries are written in pieces of 16 bytes, some 7.5 us for a thousand rows.  Whole
// calls, us, score_split_kernel (from 2^21 on tiles) and here: chunks x rows 300 x 64 17.4 and 16.3, 2000 x 128 18.1 and 17.8, 3300 x 192 29.7
// and 23.8, 5500 x 512 82.8 and 64.8, 8192 x 64 24.2 and 22.0, x 1024 144 and 115; not taken: 300 x 512 20.5 and 22.5, 2700 x 512 41.0 and 43.8,
// 4200 x 384 47.5 and 51.6 (132 workgroups of twelve blocks).
bool takes_parts(int32_t dtype, int64_t C, int32_t K, int32_t M_rows, int32_t query_reduce) {
  const int units = compute_units();
  if (dtype != MSA_F32 || K != kSplitK || M_rows > kPartsMaxRows || query_reduce != kQueryMax || C > (int64_t)kSplitCols * units) return false;
  const SplitGrid here = parts_grid((int32_t)C, M_rows), there = split_grid((int32_t)C, M_rows);
  if (here.x > units) return false;
  if (!split_ok((int32_t)C, M_rows)) return true;
  const int share = there.per_wg * ((there.x * there.y + units - 1) / units);
  return 3.2f * (float)here.per_wg + 0.0075f * (float)M_rows < 3.7f * (float)share + 1.3f;
}
template <bool kDocMax>
int launch_parts(const void* qs, const void* kr, const uint32_t* row_bits, uint32_t* out_key, const int32_t* chunk_doc,
                 int32_t M_rows, int32_t C, int32_t blocks_per_query, int32_t n_docs, hipStream_t st) {
  const SplitGrid grid = parts_grid(C, M_rows);
  static std::atomic<int> lds_limit_raised{0};
  MSA_HIP(raise_dynamic_lds_limit(lds_limit_raised, reinterpret_cast<const void*>(score_parts_kernel<kDocMax>), kPartsLds));
  int slot = -1;
  if (g_timer.on.load(std::memory_order_acquire)) {
    std::lock_guard<std::mutex> lock(g_timer.mu);
    if (g_timer.n < g_timer.cap) slot = g_timer.n++;
  }
  if (slot >= 0) MSA_HIP(hipEventRecord(g_timer.start[slot], st));
  score_parts_kernel<kDocMax><<<dim3((unsigned)grid.x, (unsigned)grid.y), kPartsWaves * 64, kPartsLds, st>>>(
      static_cast<const char*>(qs), static_cast<const float*>(kr), row_bits, out_key, chunk_doc, M_rows, C, blocks_per_query, n_docs, grid.per_wg);
  MSA_LAUNCH_CHECK();
  if (slot >= 0) MSA_HIP(hipEventRecord(g_timer.stop[slot], st));
  return MSA_OK;
}

// Launch of the MFMA-bound form (score_scan4_kernel): one workgroup per compute unit, persistent.
std::atomic<int> g_tile_pool_enabled{1};

template <bool kDocMax, bool kUnits = false>
int launch_scan4(const void* qs, const void* kr, const uint32_t* row_bits, uint32_t* out_key, const int32_t* chunk_doc,
                 int32_t M_rows, int32_t C, int32_t K, int32_t blocks_per_query, int32_t n_docs, hipStream_t st,
                 const GatherJob* job, bool* job_taken, uint32_t* sched) {
  constexpr int BM = 256, BN = 256;
  const int tiles_m = (M_rows + BM - 1) / BM;
  const int tiles_n = (C + BN - 1) / BN;
  const int k_tiles = K * (int)sizeof(bf16_t) / kRowBytes;
  // the loop requests K tiles two steps ahead: at least two K tiles per tile
  if (K * (int)sizeof(bf16_t) % kRowBytes != 0 || k_tiles < 2) {
    msa_set_error("score_scan4: K=%d is not a multiple of 64 of at least 128", K);
    return MSA_EINVAL;
  }
  // M tiles are walked in groups of 8 per K_r tile: a group's query rows (4 MiB in bf16) are what an XCD's L2 holds.
  // At 8 M tiles that is all of them (groups of 1, 2, 4 lose 2-14 % there); with 16 M tiles groups of 8 measured
  // 1.4 % faster than one group, with 256 (a 64k-row prefill batch) 4 %.
  const int m_group = std::min(tiles_m, 8);
  const int grid = std::min(kSchedMaxWorkgroups, std::max(16, compute_units() / 8 * 8));
  // The XCDs do not run at one speed (their ends lay up to 6 % apart with fixed ranges, in an order that changes from
  // launch to launch): the last eighth of the N tiles is a pool the workgroups draw from one tile at a time once
  // their own share is done.  Worth it when a workgroup has tiles enough for the pool to even the ends out, and
  // possible when a tile is deep enough for a draw to come back in time (three hops, one per K step, in front of the
  // step in which the loads leave the tile).
  int pool_n = 0;
  if (g_tile_pool_enabled.load(std::memory_order_relaxed) && (int64_t)tiles_m * tiles_n >= (int64_t)16 * grid && k_tiles >= 6)
    pool_n = tiles_n / 8;
  GatherJob no_job{};
  const GatherJob* the_job = &no_job;
  if (job != nullptr && job->active) {
    the_job = job;
    if (job_taken) *job_taken = true;
  }
  auto kern = score_scan4_kernel<kDocMax>;
  if constexpr (kUnits) kern = score_scan4_units_kernel;
  static std::atomic<int> lds_limit_raised{0}, resources_checked{0};
  if (const int rc = check_asm_kernel_resources(resources_checked, reinterpret_cast<const void*>(kern), kUnits ? "score_scan4_units_kernel" : "score_scan4_kernel",
                                                nullptr, nullptr))
    return rc;
  MSA_HIP(raise_dynamic_lds_limit(lds_limit_raised, reinterpret_cast<const void*>(kern), kScan4LdsBytes));
  int slot = -1;
  if (g_timer.on.load(std::memory_order_acquire)) {
    std::lock_guard<std::mutex> lock(g_timer.mu);
    if (g_timer.n < g_timer.cap) slot = g_timer.n++;
  }
  if (slot >= 0) MSA_HIP(hipEventRecord(g_timer.start[slot], st));
  kern<<<grid, 256, kScan4LdsBytes, st>>>(static_cast<const bf16_t*>(qs), static_cast<const bf16_t*>(kr), row_bits, out_key,
                                          chunk_doc, M_rows, C, K, blocks_per_query, tiles_m, tiles_n, m_group, n_docs,
                                          *the_job, sched, pool_n);
  MSA_LAUNCH_CHECK();
  if (slot >= 0) MSA_HIP(hipEventRecord(g_timer.stop[slot], st));
  return MSA_OK;
}

// Tile choice by query rows.  Up to 64 rows: narrow M tile, two workgroups per compute unit, two K tiles of global
// loads ahead (3 % faster than one).  Up to 128 rows: 128 x 256 with both operands loaded straight into LDS two K steps
// ahead (1.5 % faster than the register-staged 128 x 384 it replaced, which beat register-staged 128 x 256 by 3 % and
// 128 x 128 by 8 %; more register sets of loads in flight or 16 wavefronts measured 0-6 % slower: the bytes in flight
// are not what limits this shape, the query tile's own traffic and the MFMA work are - with a query tile of zeros the
// same launch streams at the rate of the 64-row form).  More rows are MFMA-bound: the 256 x 256 tile of
// score_scan4_kernel, which is also the form that can carry a gather job.
template <bool kDocMax>
int launch_gemm_for(int32_t dtype, const void* qs, const void* kr, const uint32_t* row_bits, uint32_t* out_key,
                    const int32_t* chunk_doc, int32_t M_rows, int32_t C, int32_t K, int32_t bpq, int32_t n_docs,
                    hipStream_t st, const GatherJob* job, bool* job_taken, uint32_t* sched, int unit, bool by_units) {
  if constexpr (kDocMax) {
    if (by_units) return launch_scan4<true, true>(qs, kr, row_bits, out_key, chunk_doc, M_rows, C, K, bpq, n_docs, st, job, job_taken, sched);
    if (unit == 8 && M_rows <= 64)
      return launch_gemm<bf16_t, 64, 128, 2, 2, 2, true, true, 8>(qs, kr, row_bits, out_key, chunk_doc, M_rows, C, K, bpq, n_docs, st);
    if (unit == 8)
      return launch_gemm<bf16_t, 128, 256, 2, 4, 1, true, true, 8>(qs, kr, row_bits, out_key, chunk_doc, M_rows, C, K, bpq, n_docs, st);
    if (unit == 4 && M_rows <= 64)
      return launch_gemm<bf16_t, 64, 128, 2, 2, 2, true, true, 4>(qs, kr, row_bits, out_key, chunk_doc, M_rows, C, K, bpq, n_docs, st);
    if (unit == 4)
      return launch_gemm<bf16_t, 128, 256, 2, 4, 1, true, true, 4>(qs, kr, row_bits, out_key, chunk_doc, M_rows, C, K, bpq, n_docs, st);
  }
  // The line between the fp32 forms: above it the tiles' reuse of both operands is worth more than the even split (16384 chunks x
  // 128 rows: 61 us in the split form, 84 in tiles; x 256 rows 95 and 88; 65536 x 128: 190 and 151), except that the tiles pad up
  // to 64 rows to 128 (65536 x 64: 123 and 142).
  if (dtype != MSA_BF16 && K == kSplitK && split_ok(C, M_rows))
    return launch_split<kDocMax>(qs, kr, row_bits, out_key, chunk_doc, M_rows, C, bpq, n_docs, st);
  if (dtype != MSA_BF16)
    return launch_gemm<float, 128, 128, 2, 2, 1, kDocMax, false>(qs, kr, row_bits, out_key, chunk_doc, M_rows, C, K, bpq, n_docs, st);
  if (M_rows <= 64)
    return launch_gemm<bf16_t, 64, 128, 2, 2, 2, kDocMax, true>(qs, kr, row_bits, out_key, chunk_doc, M_rows, C, K, bpq, n_docs, st);
  if (M_rows <= 128)
    return launch_gemm<bf16_t, 128, 256, 2, 4, 1, kDocMax, true>(qs, kr, row_bits, out_key, chunk_doc, M_rows, C, K, bpq, n_docs, st);
  return launch_scan4<kDocMax>(qs, kr, row_bits, out_key, chunk_doc, M_rows, C, K, bpq, n_docs, st, job, job_taken, sched);
}

}  // namespace

// ------------------------------------------------------------------------------------------
// Workspace layout (shared with topk.hip through route_internal.h)
// ------------------------------------------------------------------------------------------

RouteWorkspace route_workspace_layout(int32_t B, int32_t S, int32_t Hkv, int32_t D, int64_t plane_cols, int64_t n_docs,
                                      int32_t dtype, bool parts, int32_t unit) {
  RouteWorkspace w{};
  w.S_pad = (S + unit - 1) / unit * unit;
  w.M_rows = (B * w.S_pad + 31) / 32 * 32;
  const int64_t m_alloc = ((int64_t)w.M_rows + 255) / 256 * 256;   // every M tile may read whole mask words
  w.mask_words = (int32_t)(m_alloc / 32);
  size_t off = 0;
  w.off_qs = off;       off = align_up(off + (size_t)w.M_rows * Hkv * D * (parts ? 3 * sizeof(bf16_t) : elem_bytes(dtype)), 256);
  w.off_row_bits = off; off = align_up(off + (size_t)w.mask_words * sizeof(uint32_t), 256);
  w.off_key = off;      off = align_up(off + (size_t)B * plane_cols * sizeof(uint32_t), 256);
  w.topk_blocks = topk_blocks_for(n_docs);
  w.off_cand = off;     off = align_up(off + (size_t)B * w.topk_blocks * kTopkMax * sizeof(uint64_t), 256);
  w.off_sched = off;    off = align_up(off + kSchedBytes, 256);
  w.off_collapsed = off; off = align_up(off + (size_t)B * Hkv * D * sizeof(float) + (size_t)B * sizeof(int32_t), 256);
  w.bytes = off;
  return w;
}

namespace {
// How the rows of a batch of queries lie in the scan (bf16, maxima over tokens and chunks).  A query has row blocks of 32 of its own, or,
// where that asks for a smaller form of the scan or fewer of its large tiles, queries are padded to units of 8 or 4 rows and share
// blocks: the padding is multiplied like the rest, 4 tokens in 32 rows eight times over.  What it costs is a fold per query in place of
// one per block, and in the large tiles a fold between two steps (16 queries of 104 rows 4129 -> 3930 us where one tile row in eight goes).
// Whole calls, us, row blocks of their own and shared ones, 1.6M chunks: 28 queries x 2 tokens 2059 -> 597, 22 x 4 1550 -> 574, 10 x 3
// 1118 -> 525, 7 x 5 599 -> 510, 16 x 8 1114 -> 580, 32 x 8 2078 -> 760 (one row of large tiles: every step waits for K_r), 6 x 37 1192 ->
// 703, 32 x 37 4118 -> 2928, 5 x 20 613 -> 547; 160,000 chunks: 28 x 2 230 -> 86, 32 x 37 426 -> 326.  Where all tiles are one round
// anyway the blocks stay apart (20,000 chunks, 9 x 37: 35.9 and 37.9).  A scan that carries a gather stays one that can.
struct RowPacking {
  int32_t unit;
  bool by_units;      // the large tiles, rows in the order of their units
};
RowPacking row_packing(int32_t B, int32_t S, int64_t C, bool gathers) {
  auto rows = [&](int unit) { return (int64_t)B * ((S + unit - 1) / unit * unit); };
  const int64_t whole = rows(32);
  if (!gathers || whole <= 128)
    for (const int64_t most : {64, 128}) {
      if (whole <= most) return {32, false};
      if (rows(8) <= most) return {8, false};
      if (S <= 4 && rows(4) <= most) return {4, false};
    }
  // rounds of tiles that the compute units have to multiply
  auto rounds = [&](int64_t m) { return ((m + 255) / 256 * ((C + 255) / 256) + compute_units() - 1) / compute_units(); };
  if (S <= 1024 && rounds(rows(8)) < rounds(whole)) return {8, true};
  return {32, false};
}

// Whether some bank's fp32 queries of these sizes come in parts.
bool may_take_parts(int32_t B, int32_t S, int32_t Hkv, int32_t D) { return (int64_t)B * ((S + 31) / 32 * 32) <= kPartsMaxRows && Hkv * D == kSplitK; }
}  // namespace

// Host-side replay of the large-tile scan's tile order (scan_walk.h): every scoring workgroup walks its own tiles
// with the cursor the kernel uses, then the workgroups draw the pool's tiles in turn from one counter.
extern "C" int msa_diag_scan_walk(int32_t tiles_m, int32_t tiles_n, int32_t grid, int32_t has_copy_workgroup,
                                  int32_t pool_n, int32_t* visits) {
  MSA_REQUIRE(visits != nullptr, "msa_diag_scan_walk: null output");
  MSA_REQUIRE(tiles_m > 0 && tiles_n > 0 && grid >= 16 && grid <= kSchedMaxWorkgroups && pool_n >= 0 && pool_n <= tiles_n,
              "msa_diag_scan_walk: tiles %d x %d, grid %d, pool %d out of range", tiles_m, tiles_n, grid, pool_n);
  const int m_group = std::min(tiles_m, 8);
  for (int64_t i = 0; i < (int64_t)tiles_m * tiles_n; ++i) visits[i] = 0;
  const int scoring = grid - (has_copy_workgroup ? 1 : 0);
  std::vector<int> draws;
  for (int b = 0; b < scoring; ++b) {
    const ScanWalk w = scan_walk_init(b, grid, has_copy_workgroup, tiles_m, tiles_n, m_group, pool_n);
    if (w.own_count == 0) continue;
    ScanWalkCursor c = scan_walk_cursor(w);
    for (int idx = 0; idx < w.own_count; ++idx) {
      int tm, tn, tm2, tn2;
      scan_walk_cursor_tile(w, c, tm, tn);
      scan_walk_own(w, idx, tm2, tn2);
      if (tm != tm2 || tn != tn2 || tm < 0 || tm >= tiles_m || tn < 0 || tn >= tiles_n) {
        msa_set_error("msa_diag_scan_walk: workgroup %d tile %d: cursor (%d, %d), closed form (%d, %d)", b, idx, tm, tn, tm2, tn2);
        return MSA_ESTATE;
      }
      ++visits[(int64_t)tm * tiles_n + tn];
      if (idx + 1 < w.own_count) scan_walk_cursor_next(w, c);
    }
    draws.push_back(b);
  }
  int counter = 0;
  while (pool_n > 0 && !draws.empty()) {
    std::vector<int> still;
    for (int b : draws) {
      const ScanWalk w = scan_walk_init(b, grid, has_copy_workgroup, tiles_m, tiles_n, m_group, pool_n);
      const int p = counter++;
      if (p >= w.pool_total) continue;
      int tm, tn;
      scan_walk_pool(w, p, tm, tn);
      if (tm < 0 || tm >= tiles_m || tn < 0 || tn >= tiles_n) {
        msa_set_error("msa_diag_scan_walk: pool position %d -> (%d, %d)", p, tm, tn);
        return MSA_ESTATE;
      }
      ++visits[(int64_t)tm * tiles_n + tn];
      still.push_back(b);
    }
    draws.swap(still);
  }
  return MSA_OK;
}

// How route_scores_to_keys lays the rows of a call's queries (a test aid).
extern "C" int msa_diag_row_packing(int32_t B, int32_t S, int64_t C, int32_t gathers, int32_t* unit, int32_t* by_units) {
  MSA_REQUIRE(unit != nullptr && by_units != nullptr && B > 0 && S > 0 && C > 0, "msa_diag_row_packing: null output, or no rows");
  const RowPacking p = row_packing(B, S, C, gathers != 0);
  *unit = p.unit;
  *by_units = p.by_units;
  return MSA_OK;
}

// The tile pool of the large-tile scan can be switched off (every tile then belongs to a fixed workgroup).
extern "C" int msa_diag_asm_kernel_resources(int32_t which, int32_t* num_regs, int32_t* scratch_bytes) {
  MSA_REQUIRE(num_regs && scratch_bytes, "msa_diag_asm_kernel_resources: null pointer");
  std::atomic<int> unused{0};
  int regs = 0, scratch = 0, rc;
  if (which == 0)
    rc = check_asm_kernel_resources(unused, reinterpret_cast<const void*>(score_scan4_kernel<true>), "score_scan4_kernel", &regs,
                                    &scratch);
  else if (which == 1)
    rc = flash_wide_kernel_resources(&regs, &scratch);
  else {
    msa_set_error("msa_diag_asm_kernel_resources: which = 0 (routing scan) or 1 (wide flash attention)");
    return MSA_EINVAL;
  }
  *num_regs = regs;
  *scratch_bytes = scratch;
  return rc;
}

extern "C" int msa_route_set_tile_pool(int32_t enabled) {
  g_tile_pool_enabled.store(enabled ? 1 : 0, std::memory_order_relaxed);
  return MSA_OK;
}

extern "C" int msa_profile_enable(int32_t max_records) {
  std::lock_guard<std::mutex> lock(g_timer.mu);
  g_timer.on.store(0, std::memory_order_release);
  for (int i = 0; i < g_timer.cap; ++i) {
    (void)hipEventDestroy(g_timer.start[i]);
    (void)hipEventDestroy(g_timer.stop[i]);
  }
  delete[] g_timer.start;
  delete[] g_timer.stop;
  g_timer.start = g_timer.stop = nullptr;
  g_timer.cap = g_timer.n = 0;
  MSA_REQUIRE(max_records >= 0 && max_records <= 1 << 20, "msa_profile_enable: max_records=%d", max_records);
  if (max_records == 0) return MSA_OK;
  g_timer.start = new hipEvent_t[max_records];
  g_timer.stop = new hipEvent_t[max_records];
  for (int i = 0; i < max_records; ++i) {
    MSA_HIP(hipEventCreate(&g_timer.start[i]));
    MSA_HIP(hipEventCreate(&g_timer.stop[i]));
    g_timer.cap = i + 1;
  }
  g_timer.on.store(1, std::memory_order_release);
  return MSA_OK;
}

extern "C" int msa_profile_collect(float* ms_host, int32_t cap, int32_t* n_out) {
  MSA_REQUIRE(ms_host && n_out, "msa_profile_collect: null pointer");
  std::lock_guard<std::mutex> lock(g_timer.mu);
  const int n = std::min(g_timer.n, cap);
  for (int i = 0; i < n; ++i) {
    MSA_HIP(hipEventSynchronize(g_timer.stop[i]));
    MSA_HIP(hipEventElapsedTime(&ms_host[i], g_timer.start[i], g_timer.stop[i]));
  }
  *n_out = n;
  g_timer.n = 0;
  return MSA_OK;
}

extern "C" size_t msa_route_workspace_bytes(int32_t B, int32_t S, int32_t Hq, int32_t Hkv, int32_t D, int64_t C,
                                            int64_t n_docs, int32_t topk) {
  (void)Hq; (void)topk;
  if (B <= 0 || S <= 0 || Hkv <= 0 || D <= 0 || C <= 0 || n_docs <= 0) return 0;
  // sized for fp32 queries so one workspace serves both dtypes, and for the per-chunk plane of msa_chunk_scores
  return route_workspace_layout(B, S, Hkv, D, C + n_docs, n_docs, MSA_F32, may_take_parts(B, S, Hkv, D)).bytes;
}

extern "C" size_t msa_route_topk_workspace_bytes(int32_t B, int32_t S, int32_t Hq, int32_t Hkv, int32_t D,
                                                 int64_t n_docs, int32_t topk) {
  (void)Hq; (void)topk;
  if (B <= 0 || S <= 0 || Hkv <= 0 || D <= 0 || n_docs <= 0) return 0;
  return route_workspace_layout(B, S, Hkv, D, n_docs, n_docs, MSA_F32, may_take_parts(B, S, Hkv, D)).bytes;
}

int route_scores_to_keys(const msa_bank* bank, int32_t layer, const void* q, const uint8_t* qmask_u8, int32_t B,
                         int32_t S, int32_t Hq, int32_t mode, float scale, bool doc_max, void* workspace,
                         size_t workspace_bytes, hipStream_t st, RouteWorkspace* layout_out, float* mul_out,
                         const char* who, const GatherJob* job, bool* job_taken, int32_t query_reduce,
                         int64_t extra_plane_cols) {
  if (job_taken) *job_taken = false;
  MSA_REQUIRE(query_reduce == kQueryMax || query_reduce == kQueryMean || query_reduce == kQueryLast,
              "%s: bad query reduction %d", who, query_reduce);
  MSA_REQUIRE(bank != nullptr, "%s: null bank", who);
  MSA_REQUIRE(layer >= 0 && layer < bank->n_layers, "%s: layer %d out of range", who, layer);
  if (bank->kr_dev[layer] == nullptr) {
    msa_set_error("%s: layer %d has no K_r set", who, layer);
    return MSA_ESTATE;
  }
  MSA_REQUIRE(q != nullptr && workspace != nullptr, "%s: null pointer", who);
  MSA_REQUIRE(B > 0 && B <= 4096 && S > 0 && S <= 65536, "%s: B=%d S=%d out of range", who, B, S);
  MSA_REQUIRE(Hq > 0 && Hq % bank->Hkv == 0, "%s: Hq=%d not a multiple of Hkv=%d", who, Hq, bank->Hkv);
  MSA_REQUIRE(bank->Hkv <= 16, "%s: Hkv=%d unsupported (max 16)", who, bank->Hkv);
  MSA_REQUIRE(mode == MSA_MODE_COSINE || mode == MSA_MODE_SCALED_DOT, "%s: bad mode %d", who, mode);
  MSA_REQUIRE(((uintptr_t)q & 15) == 0 && ((uintptr_t)workspace & 255) == 0, "%s: q / workspace misaligned", who);
  const float sc = mode == MSA_MODE_COSINE ? 1.0f : scale;
  MSA_REQUIRE(sc > 0.f && sc < INFINITY, "%s: scale must be positive and finite", who);
  MSA_REQUIRE((int64_t)B * ((S + 31) / 32 * 32) < (int64_t)1 << 24, "%s: too many query rows", who);

  const int64_t plane_cols = doc_max ? bank->n_docs : bank->C;
  // a collapsed query (mean / last over its tokens) is one row: one row block per query
  const int32_t S_scan = query_reduce == kQueryMax ? S : 1;
  RouteWorkspace w = route_workspace_layout(B, S_scan, bank->Hkv, bank->D, plane_cols + extra_plane_cols, bank->n_docs, bank->dtype, true);
  const bool parts = takes_parts(bank->dtype, bank->C, bank->Hkv * bank->D, w.M_rows, query_reduce) && w.bytes <= workspace_bytes;
  if (!parts) w = route_workspace_layout(B, S_scan, bank->Hkv, bank->D, plane_cols + extra_plane_cols, bank->n_docs, bank->dtype, false);
  if (w.bytes > workspace_bytes) {
    msa_set_error("%s: workspace of %zu bytes, need %zu", who, workspace_bytes, w.bytes);
    return MSA_ESIZE;
  }
  RowPacking packing{32, false};
  if (bank->dtype == MSA_BF16 && doc_max && query_reduce == kQueryMax) packing = row_packing(B, S, bank->C, job != nullptr && job->active);
  if (packing.unit != 32)      // (no more rows than whole blocks have: it fits where they do)
    w = route_workspace_layout(B, S, bank->Hkv, bank->D, plane_cols + extra_plane_cols, bank->n_docs, bank->dtype, false, packing.unit);
  char* ws = static_cast<char*>(workspace);
  void* qs = ws + w.off_qs;
  uint32_t* row_bits = reinterpret_cast<uint32_t*>(ws + w.off_row_bits);
  uint32_t* key = reinterpret_cast<uint32_t*>(ws + w.off_key);
  uint32_t* sched = reinterpret_cast<uint32_t*>(ws + w.off_sched);

  const int normalize = mode == MSA_MODE_COSINE ? 1 : 0;
  const int pthreads = bank->Hkv * 16;
  const int64_t clear_words = (int64_t)B * plane_cols;
  if (query_reduce != kQueryMax) {
    float* rows = reinterpret_cast<float*>(ws + w.off_collapsed);
    int32_t* counts = reinterpret_cast<int32_t*>(rows + (size_t)B * bank->Hkv * bank->D);
    const dim3 cgrid((unsigned)B, (unsigned)bank->Hkv);
    if (bank->dtype == MSA_BF16) {
      collapse_queries_kernel<bf16_t><<<cgrid, 256, 0, st>>>(static_cast<const bf16_t*>(q), qmask_u8, S, Hq, bank->Hkv,
                                                             normalize, query_reduce, rows, counts);
      MSA_LAUNCH_CHECK();
      broadcast_rows_kernel<bf16_t><<<w.M_rows, 256, 0, st>>>(rows, counts, bank->Hkv, static_cast<bf16_t*>(qs), row_bits,
                                                              w.mask_words, key, clear_words, sched);
    } else {
      collapse_queries_kernel<float><<<cgrid, 256, 0, st>>>(static_cast<const float*>(q), qmask_u8, S, Hq, bank->Hkv,
                                                            normalize, query_reduce, rows, counts);
      MSA_LAUNCH_CHECK();
      broadcast_rows_kernel<float><<<w.M_rows, 256, 0, st>>>(rows, counts, bank->Hkv, static_cast<float*>(qs), row_bits,
                                                             w.mask_words, key, clear_words, sched);
    }
  } else if (bank->dtype == MSA_BF16) {
    presum_queries_kernel<bf16_t, bf16_t><<<w.M_rows, pthreads, 0, st>>>(
        static_cast<const bf16_t*>(q), qmask_u8, B, S, w.S_pad, Hq, bank->Hkv, normalize, static_cast<bf16_t*>(qs),
        row_bits, w.mask_words, key, clear_words, sched, packing.unit != 32, packing.by_units);
  } else if (parts) {
    presum_queries_kernel<float, float, true><<<w.M_rows, pthreads, 0, st>>>(
        static_cast<const float*>(q), qmask_u8, B, S, w.S_pad, Hq, bank->Hkv, normalize, static_cast<float*>(qs),
        row_bits, w.mask_words, key, clear_words, sched, 0, 0);
  } else {
    presum_queries_kernel<float, float><<<w.M_rows, pthreads, 0, st>>>(
        static_cast<const float*>(q), qmask_u8, B, S, w.S_pad, Hq, bank->Hkv, normalize, static_cast<float*>(qs),
        row_bits, w.mask_words, key, clear_words, sched, 0, 0);
  }
  MSA_LAUNCH_CHECK();

  const int32_t K = bank->Hkv * bank->D;
  const int32_t bpq = w.S_pad / packing.unit;      // row blocks (units) of a query
  const auto by_parts = doc_max ? launch_parts<true> : launch_parts<false>;
  const int rc = parts ? by_parts(qs, bank->kr_dev[layer], row_bits, key, doc_max ? bank->chunk_doc_dev : nullptr, w.M_rows, (int32_t)bank->C, bpq,
                                  (int32_t)bank->n_docs, st)
                 : doc_max ? launch_gemm_for<true>(bank->dtype, qs, bank->kr_dev[layer], row_bits, key, bank->chunk_doc_dev,
                                                 w.M_rows, (int32_t)bank->C, K, bpq, (int32_t)bank->n_docs, st, job,
                                                 job_taken, sched, packing.unit, packing.by_units)
                         : launch_gemm_for<false>(bank->dtype, qs, bank->kr_dev[layer], row_bits, key, nullptr, w.M_rows,
                                                  (int32_t)bank->C, K, bpq, (int32_t)bank->n_docs, st, job, job_taken, sched, 32, false);
  if (rc != MSA_OK) return rc;
  *layout_out = w;
  *mul_out = sc / (float)Hq;
  return MSA_OK;
}

extern "C" int msa_chunk_scores(const msa_bank* bank, int32_t layer, const void* q, const uint8_t* qmask_u8, int32_t B,
                                int32_t S, int32_t Hq, int32_t mode, float scale, float* chunk_scores,
                                void* workspace, size_t workspace_bytes, void* stream) {
  MSA_REQUIRE(chunk_scores != nullptr, "msa_chunk_scores: null output");
  RouteWorkspace w;
  float mul;
  hipStream_t st = as_stream(stream);
  int rc = route_scores_to_keys(bank, layer, q, qmask_u8, B, S, Hq, mode, scale, false, workspace, workspace_bytes, st,
                                &w, &mul, "msa_chunk_scores");
  if (rc != MSA_OK) return rc;
  const int64_t n = (int64_t)B * bank->C;
  const uint32_t* key = reinterpret_cast<const uint32_t*>(static_cast<char*>(workspace) + w.off_key);
  decode_scores_kernel<<<(int)std::min<int64_t>((n + 255) / 256, 8192), 256, 0, st>>>(key, n, mul, chunk_scores);
  MSA_LAUNCH_CHECK();
  return MSA_OK;
}
