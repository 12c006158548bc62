// Shared between attn.hip (single rows, combine) and flash_attn.hip (MFMA kernels).
#pragma once
#include <algorithm>

#include "common.h"

constexpr int kMinSplitKeys = 256;   // fewest keys worth a workgroup of its own

// Splits of the key range: enough workgroups to fill the chip (about 1024) when there are few
// (query row, KV head) pairs, a single pass over the keys when there are many.  split_keys is a
// multiple of 64.
struct SplitPlan {
  int n_split;
  int split_keys;
};
static inline SplitPlan plan_splits_for(int64_t total_q, int32_t Hkv, int32_t max_kv, int target) {
  const int64_t pairs = std::max<int64_t>(1, total_q * Hkv);
  const int by_fill = (int)std::max<int64_t>(1, (target + pairs - 1) / pairs);
  const int by_size = std::max(1, (max_kv + kMinSplitKeys - 1) / kMinSplitKeys);
  const int n = std::min(by_fill, by_size);
  const int keys = ((max_kv + n - 1) / n + 63) / 64 * 64;
  return {(max_kv + keys - 1) / keys, keys};
}
// MFMA split kernel: about 1024 workgroups.
static inline SplitPlan plan_splits(int64_t total_q, int32_t Hkv, int32_t max_kv) {
  return plan_splits_for(total_q, Hkv, max_kv, 1024);
}
// The same for blocks of query rows, by what the kernel makes workgroups of: tiles of 128 (token, head) columns, at least one a sample, and
// two workgroups a compute unit.  By rows, as above, 128 rows of 8 KV heads were 1024 pairs and never split.  us, by rows and by tiles, 8 KV heads, groups of
// four: one sample of 64 rows and 4096 keys 44.1 and 27.8, of 128 77.0 and 31.3, of 256 80.7 and 39.6, of 512 88.9 and 54.2, 4 of 64 79.0 and 43.3,
// 8 of 64 83.9 and 59.0, 16 of 64 111 and 101; 2048 keys, one of 128 45.7 and 28.3.
static inline SplitPlan plan_splits_tiles(int64_t total_q, int64_t samples, int G, int32_t Hkv, int32_t max_kv) {
  const int64_t tiles = std::max(samples, (total_q * G + 127) / 128) * Hkv;
  const int by_fill = (int)std::min<int64_t>(16, std::max<int64_t>(1, 512 / tiles)), by_size = std::max(1, (max_kv + kMinSplitKeys - 1) / kMinSplitKeys);
  const int n = std::min(by_fill, by_size), keys = ((max_kv + n - 1) / n + 63) / 64 * 64;
  return {(max_kv + keys - 1) / keys, keys};
}
// Single rows (decode): one workgroup per compute unit (fewer, longer key streams); the kernels divide each sample's own length
// evenly over n_split.  The bf16 ring, of which two fit, is cut finer where that does not come out even and leaves 256 keys a split
// or more (groups of four, us: 24 samples of 2200 to 4400 keys with 2 KV heads in 288 workgroups 28.2, in 528 23.6; but 16 of 256 to
// 512 with 8, even in 256, 13.4 against 15.1 in 384).
static inline SplitPlan plan_splits_rows(int64_t total_q, int32_t Hkv, int32_t max_kv, bool ring) {
  constexpr int kUnits = 256;
  const int64_t pairs = std::max<int64_t>(1, total_q * Hkv), finer = (2 * kUnits + pairs - 1) / pairs;
  const bool even = (kUnits + pairs - 1) / pairs * pairs == kUnits;
  return plan_splits_for(total_q, Hkv, max_kv, ring && !even && max_kv >= kMinSplitKeys * finer ? 2 * kUnits : kUnits);
}
// The line between the two forms for bf16 rows with G query heads a KV head.  With four and eight the vector units do not keep up
// with memory; with one they do, and with two nearly: there the ring's own start and end count.  It is ahead with two heads, unless
// short rows fill the chip several times over, and with one where a wavefront has one step of 32 keys.  On the vector units and in the
// ring, us, 8 KV heads: two heads, one sample of 4388 keys 16.7 / 11.8, 8 of 500 to 1000 13.1 / 11.2, 16 of 2194 to 4388 53.6 / 47.1;
// one head, 16 of 32 to 64 keys 6.0 / 4.8, but of 128 to 256 7.8 / 8.6 and of 2194 to 4388 46.3 / 48.4.  64 samples of 64 to 128 keys
// with 32 KV heads: two heads 24.9 / 29.9, one 22.2 / 29.5 (of 256 to 512 with two 76.9 / 84.4).
static inline bool takes_ring(int64_t total_q, int32_t Hkv, int32_t max_kv, int G) {
  const int64_t pairs = total_q * Hkv;
  return G > 2 || (G == 2 ? pairs <= 512 || max_kv > 1024 : pairs <= 512 && max_kv <= 128);
}

// flash_attn.hip: bf16 partial pass over split `blockIdx.z` of the keys; writes un-normalised
// accumulators and (reference max, sum) pairs in the layout attn_combine_kernel reads.
int flash_attn_split_launch(const void* q, const int32_t* cu_q, const void* k, const void* v, const int64_t* kv_off,
                            const int32_t* kv_len, int32_t B, int32_t total_q, int32_t Hq, int32_t Hkv, float scale,
                            int32_t causal, SplitPlan plan, float* part_ml, float* part_acc, hipStream_t st);
