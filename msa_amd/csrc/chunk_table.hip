// Segments and chunk table of a packed block: tiny kernels, no host synchronisation.
#include "common.h"

namespace {

constexpr int kScanThreads = 1024;

// One workgroup: exclusive scan of ceil(len_d / P) over all documents.
__global__ __launch_bounds__(kScanThreads) void doc_chunk_scan_kernel(const int32_t* __restrict__ doc_start,
                                                                      int32_t n_docs, int32_t P,
                                                                      int32_t* __restrict__ doc_chunk_off,
                                                                      int64_t* __restrict__ n_chunks_out) {
  __shared__ int32_t part[kScanThreads];
  const int tid = threadIdx.x;
  const int per = (n_docs + kScanThreads - 1) / kScanThreads;
  const int lo = min(tid * per, n_docs), hi = min(lo + per, n_docs);
  int32_t sum = 0;
  for (int d = lo; d < hi; ++d) sum += (doc_start[d + 1] - doc_start[d] + P - 1) / P;
  part[tid] = sum;
  __syncthreads();
  for (int off = 1; off < kScanThreads; off <<= 1) {   // Hillis-Steele inclusive scan
    int32_t add = tid >= off ? part[tid - off] : 0;
    __syncthreads();
    part[tid] += add;
    __syncthreads();
  }
  int32_t run = part[tid] - sum;
  for (int d = lo; d < hi; ++d) {
    doc_chunk_off[d] = run;
    run += (doc_start[d + 1] - doc_start[d] + P - 1) / P;
  }
  if (tid == kScanThreads - 1) {
    doc_chunk_off[n_docs] = part[tid];
    n_chunks_out[0] = part[tid];
  }
}

// One thread per document writes that document's chunk rows.
__global__ void chunk_fill_kernel(const int32_t* __restrict__ doc_start, const int32_t* __restrict__ doc_chunk_off,
                                  int32_t n_docs, int32_t P, int64_t chunk_cap, int32_t* __restrict__ chunk_start,
                                  int32_t* __restrict__ chunk_len, int32_t* __restrict__ chunk_doc) {
  const int d = blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= n_docs) return;
  const int32_t s = doc_start[d], n = doc_start[d + 1] - s;
  const int32_t base = doc_chunk_off[d], nch = (n + P - 1) / P;
  for (int32_t j = 0; j < nch; ++j) {
    const int64_t c = (int64_t)base + j;
    if (c >= chunk_cap) return;
    chunk_start[c] = s + j * P;
    chunk_len[c] = min(P, n - j * P);
    chunk_doc[c] = d;
  }
}

// Runs of equal ids behind the template (the ids that are -2, in front): what the host reads of them (`head`), and where every segment begins
// for the kernels that follow.  Every layer counted, compared and copied on its own before, and the host waited for the layer in front each
// time (encoding 2048 tokens through two layers 1610 us, 1050 so; 32,768 11,840 and 11,140).  Both together 13 us for 32,771 tokens.  scan_ids_kernel, a workgroup per 1024 tokens: a bit a token that
// opens a run, the counts and largest values (by one workgroup the ids of 32,771 tokens took 47 us, a compute unit's share of the memory);
// block_segments_kernel, one workgroup, 64 words of bits a wavefront.
constexpr int kScanTokens = 1024;
struct IdSums {
  int32_t n_template, last_wrong, last_pos, unused;      // ids that are -2, the last that is not positive, the largest position
  int64_t mask_sum;
};
static_assert(sizeof(IdSums) == 3 * sizeof(int64_t), "three words a workgroup");
__host__ __device__ inline int64_t id_words(int64_t T) { return (T + 63) / 64; }
__host__ __device__ inline int64_t id_parts(int64_t T) { return (T + kScanTokens - 1) / kScanTokens; }

__global__ __launch_bounds__(256) void scan_ids_kernel(const int64_t* __restrict__ ids, const int64_t* __restrict__ mask, const int64_t* __restrict__ pos,
                                                       int32_t T, uint64_t* __restrict__ words, IdSums* __restrict__ sums) {
  __shared__ IdSums parts[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  IdSums own{0, -1, INT32_MIN, 0, 0};
#pragma unroll
  for (int k = 0; k < kScanTokens / 256; ++k) {
    const int i = blockIdx.x * kScanTokens + k * 256 + threadIdx.x, at = min(i, T - 1);
    const int64_t id = ids[at], before = ids[max(at - 1, 0)], m = mask != nullptr ? mask[at] : 0, p = pos != nullptr ? pos[at] : INT32_MIN;
    const uint64_t bits = __ballot(i < T && i > 0 && id != before);
    if (lane == 0 && i < T) words[i >> 6] = bits;
    if (i < T) {
      own.n_template += id == -2;
      own.last_wrong = id <= 0 ? i : own.last_wrong;
      own.last_pos = max(own.last_pos, (int32_t)min(max(p, (int64_t)INT32_MIN), (int64_t)INT32_MAX));
      own.mask_sum += m;
    }
  }
#pragma unroll
  for (int x = 32; x > 0; x >>= 1) {
    own.n_template += __shfl_xor(own.n_template, x);
    own.last_wrong = max(own.last_wrong, __shfl_xor(own.last_wrong, x));
    own.last_pos = max(own.last_pos, __shfl_xor(own.last_pos, x));
    own.mask_sum += __shfl_xor(own.mask_sum, x);
  }
  if (lane == 0) parts[wave] = own;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      own.n_template += parts[w].n_template;
      own.last_wrong = max(own.last_wrong, parts[w].last_wrong);
      own.last_pos = max(own.last_pos, parts[w].last_pos);
      own.mask_sum += parts[w].mask_sum;
    }
    sums[blockIdx.x] = own;
  }
}

// words and sums lie where `start` will: it is written once they have been read.
__global__ __launch_bounds__(kScanThreads) void block_segments_kernel(int32_t T, int32_t* __restrict__ head, int32_t* __restrict__ cu, int64_t* start,
                                                                      int32_t* __restrict__ len) {
  __shared__ unsigned long long mask_sum;
  __shared__ int32_t n_template, last_wrong, last_pos, part[kScanThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n_words = (int)id_words(T);
  const uint64_t* words = reinterpret_cast<const uint64_t*>(start);
  const IdSums* sums = reinterpret_cast<const IdSums*>(words + n_words);
  if (tid == 0) {
    mask_sum = 0;
    n_template = 0;
    last_wrong = -1;
    last_pos = INT32_MIN;
  }
  __syncthreads();
  for (int i = tid; i < (int)id_parts(T); i += kScanThreads) {
    const IdSums own = sums[i];
    atomicAdd(&n_template, own.n_template);
    atomicMax(&last_wrong, own.last_wrong);
    atomicMax(&last_pos, own.last_pos);
    atomicAdd(&mask_sum, (unsigned long long)own.mask_sum);
  }
  __syncthreads();
  const int first = n_template;
  int n = first > 0 ? 1 : 0;                             // segments so far
  for (int base = 0; base < n_words; base += kScanThreads) {
    // a word a thread: the runs behind the template, whose first token opens one as well
    const int w = base + tid;
    uint64_t mine = w < n_words ? words[w] : 0;
    if (first >> 6 == w && first < T) mine |= 1ull << (first & 63);
    if (64 * w < first) mine = 64 * w + 64 <= first ? 0 : mine & ~0ull << (first & 63);
    const int runs = __popcll(mine);
    int sum = runs;
#pragma unroll
    for (int x = 1; x < 64; x <<= 1) {
      const int below = __shfl_up(sum, x);
      sum += lane >= x ? below : 0;
    }
    if (lane == 63) part[wave] = sum;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int v = 0; v < kScanThreads / 64; ++v) {
      before += v < wave ? part[v] : 0;
      all += part[v];
    }
    for (int at = n + before + sum - runs; mine != 0; mine &= mine - 1) cu[at++] = 64 * w + __builtin_ctzll(mine);
    n += all;
    __syncthreads();
  }
  if (tid == 0) {
    if (first > 0) cu[0] = 0;
    cu[n] = T;
    head[0] = first;
    head[1] = n - (first > 0 ? 1 : 0);
    head[2] = last_wrong >= first;
    head[3] = last_pos;
    head[4] = (int32_t)(uint32_t)mask_sum;
    head[5] = (int32_t)(uint32_t)(mask_sum >> 32);
  }
  __syncthreads();
  for (int s = tid; s < n; s += kScanThreads) {
    start[s] = cu[s];
    len[s] = cu[s + 1] - cu[s];
  }
}

}  // namespace

extern "C" int msa_block_segments(const int64_t* ids, const int64_t* mask, const int64_t* pos, int64_t T, int32_t* head, int32_t* cu,
                                  int64_t* start, int32_t* len, void* stream) {
  MSA_REQUIRE(ids && head && cu && start && len, "msa_block_segments: null pointer");
  MSA_REQUIRE(T > 0 && T < ((int64_t)1 << 30), "msa_block_segments: T=%lld", (long long)T);
  hipStream_t st = as_stream(stream);
  uint64_t* words = reinterpret_cast<uint64_t*>(start);
  scan_ids_kernel<<<(int)id_parts(T), 256, 0, st>>>(ids, mask, pos, (int32_t)T, words, reinterpret_cast<IdSums*>(words + id_words(T)));
  MSA_LAUNCH_CHECK();
  block_segments_kernel<<<1, kScanThreads, 0, st>>>((int32_t)T, head, cu, start, len);
  MSA_LAUNCH_CHECK();
  return MSA_OK;
}

extern "C" int msa_chunk_table(const int32_t* doc_start, int32_t n_docs, int32_t P, int64_t chunk_cap,
                               int32_t* doc_chunk_off, int32_t* chunk_start, int32_t* chunk_len,
                               int32_t* chunk_doc, int64_t* n_chunks_out, void* stream) {
  MSA_REQUIRE(doc_start && doc_chunk_off && chunk_start && chunk_len && chunk_doc && n_chunks_out,
              "msa_chunk_table: null pointer");
  MSA_REQUIRE(n_docs > 0, "msa_chunk_table: n_docs=%d", n_docs);
  MSA_REQUIRE(P > 0, "msa_chunk_table: P=%d", P);
  MSA_REQUIRE(chunk_cap > 0, "msa_chunk_table: chunk_cap=%lld", (long long)chunk_cap);
  hipStream_t st = as_stream(stream);
  doc_chunk_scan_kernel<<<1, kScanThreads, 0, st>>>(doc_start, n_docs, P, doc_chunk_off, n_chunks_out);
  MSA_LAUNCH_CHECK();
  chunk_fill_kernel<<<(n_docs + 255) / 256, 256, 0, st>>>(doc_start, doc_chunk_off, n_docs, P, chunk_cap,
                                                          chunk_start, chunk_len, chunk_doc);
  MSA_LAUNCH_CHECK();
  return MSA_OK;
}
