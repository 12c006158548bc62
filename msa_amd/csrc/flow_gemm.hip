// y[T, N] = x[T, K] . w[N, K]^T in bf16 with fp32 sums where one round of mid-sized tiles, or of pieces of K of them, fills the chip:
// prompts of some hundred tokens, whose products have fewer than a round of gemm.hip's tiles and take several of block_gemm.hip's.
//
// A workgroup of four wavefronts, one per SIMD, makes a tile of kN weight rows and kT tokens, a quarter each.  What bounds a K tile
// (64 elements; 128 x 128 outputs, us, each part alone): the operands' way into the compute unit 0.40, LDS reads and writes 0.30, the
// matrix cores 0.35 at the clock that the power allows.  So all of it has to run at once, and in one wavefront that takes an order of
// issue: operands go straight into a ring of kStages K tiles in LDS, each half of a K tile is read into registers during the products of
// the half before, and reads and requests stand between the products, one behind every few.  One barrier a K tile: behind it the next K
// tile has arrived and the one whose second half has just been read is requested again, kStages tiles ahead.  us a K tile: 0.53; with
// operands through registers in the same order 0.65, read and written in front of the products 0.85, by block_gemm.hip's eight
// wavefronts, which overlap by being two per SIMD, 0.59.
//
// Whole products, weights from memory, us (the faster of the vendor's and the other forms, and here): 450 x 4096 x 2560 22.7 and 18.9, 100 x
// 9728 x 2560 31.1 and 21.2, 300 x 9728 x 2560 40.6 and 30.7, 300 x 2560 x 12288 38.1 and 32.2, 700 x 2560 x 8480 43.8 and 38.2, 1000 x 1024 x
// 6144 19.1 and 17.6, 1500 x 1024 x 6144 28.5 and 23.3.
//
// The products are asm statements on accumulators that stay in place (the compiler moves them to other registers in every round), so it
// does not know their latency: nops stand in front of the first and behind the last.
#include <algorithm>

#include "common.h"
#include "seq_common.h"
#include "seq_mfma.h"

namespace {

constexpr int kK = 64, kRowBytes = 2 * kK, kThreads = 256, kXcds = 8;
constexpr int kMaxPieces = 6, kMinSteps = 6;              // of K, and K tiles of one at least

struct FlowArgs {
  const bf16_t* x;          // [T, K], rows ldx apart
  const bf16_t* w;          // [N, K]
  bf16_t* out;              // [T, N] (or [T, N / 2]), rows ldo apart
  float* part;              // [pieces][T][N] sums, where there are several
  int64_t ldx, ldo;
  int32_t T, K, N;
  int32_t tiles_t, tiles_n, strip, pieces;
  msa_tile_end end;
};

// LDS row -> weight row: row block i, lane group g, register r of a fragment's 32 rows is row 8 g + 4 i + r, so that a lane holds eight
// neighbouring outputs of a token.
__device__ __forceinline__ int weight_row(int lds_row) {
  return (lds_row & ~31) + 8 * ((lds_row >> 2) & 3) + 4 * ((lds_row >> 4) & 1) + (lds_row & 3);
}
// 16-byte units of a row lie in an order that spreads a fragment's sixteen rows over all banks.
__device__ __forceinline__ int unit_at(int row, int unit) { return row * kRowBytes + ((unit ^ ((row >> 1) & 7)) << 4); }
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const bf16_t* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p), 0, bytes, 0x00020000);
}

// Eight neighbouring outputs of a token, from column n on.
__device__ __forceinline__ void finish8(const FlowArgs& a, int token, int n, const float (&v)[8]) {
  uint32_t p[4];                                         // the product, rounded as it would be on its way through memory
#pragma unroll
  for (int e = 0; e < 4; ++e) p[e] = pack_bf16x2(v[2 * e], v[2 * e + 1]);
  bf16_t* out = a.out + (int64_t)token * a.ldo;
  if (a.end.mode == MSA_TILE_GLU) {
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = clamped_glu_f(bf16lo(p[e]), bf16hi(p[e]), a.end.limit, a.end.alpha, a.end.shift);
    *reinterpret_cast<uint2*>(out + n / 2) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
    return;
  }
  if (a.end.mode == MSA_TILE_GELU && n < a.end.gelu_n)
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] = pack_bf16x2(gelu_tanh_f(bf16lo(p[e])), gelu_tanh_f(bf16hi(p[e])));
  *reinterpret_cast<uint4*>(out + n) = make_uint4(p[0], p[1], p[2], p[3]);
}

template <int kN, int kT, int kStages>
__global__ __launch_bounds__(kThreads, kStages * (kN + kT) * kRowBytes <= 80 * 1024 ? 2 : 1) void flow_gemm_kernel(FlowArgs a) {
  constexpr int kLoadsN = kN / 32, kLoads = kLoadsN + kT / 32;      // direct-to-LDS loads of a wavefront and K tile, 1 KB (8 rows) each
  constexpr int kBN = kN / 32, kBT = kT / 32, kM = kBN * kBT;       // 16 x 16 blocks of a wavefront
  constexpr int kReads = kBN + kBT, kBuffer = (kN + kT) * kRowBytes;
  static_assert(kN % 64 == 0 && kT % 32 == 0 && kStages >= 3 && kStages * kBuffer <= 160 * 1024);
  extern __shared__ __align__(16) char lds[];
  // an XCD's workgroups (dealt round-robin) take neighbouring tiles, in strips of `strip` tiles of weights so that what they read together is least
  const int per_xcd = gridDim.x / kXcds, id = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds, tiles = a.tiles_t * a.tiles_n;
  if (id >= tiles * a.pieces) return;
  const int piece = id / tiles, tile = id - piece * tiles;
  const int strip = tile / (a.strip * a.tiles_t), in_strip = tile - strip * a.strip * a.tiles_t, wide = min(a.strip, a.tiles_n - strip * a.strip);
  const int tile_t = in_strip / wide, t0 = tile_t * kT, n0 = (strip * a.strip + in_strip - tile_t * wide) * kN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l15 = lane & 15, g = lane >> 4;
  const int wave_n = (wave >> 1) * (kN / 2), wave_t = (wave & 1) * (kT / 2);
  const bf16_t* w = a.w + (int64_t)n0 * a.K;
  const bf16_t* x = a.x + (int64_t)t0 * a.ldx;
  const int bytes_w = min(kN, a.N - n0) * a.K * 2, bytes_x = ((min(kT, a.T - t0) - 1) * (int)a.ldx + a.K) * 2;
  // rows behind the last read as zero (the K displacement is scalar and stays inside a row), and so do K tiles behind the last
  int from[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int row = 8 * (wave + 4 * (i < kLoadsN ? i : i - kLoadsN)) + (lane >> 3), unit = (lane & 7) ^ ((row >> 1) & 7);
    from[i] = (i < kLoadsN ? weight_row(row) * a.K : row * (int)a.ldx) * 2 + unit * 16;
  }
  const int all = a.K / kK, first = all * piece / a.pieces, last = all * (piece + 1) / a.pieces;
  auto load = [&](char* stage, int step, int i) {
    const bool in = step < last;
    const __amdgpu_buffer_rsrc_t rs = i < kLoadsN ? rows_rsrc(w, in ? bytes_w : 0) : rows_rsrc(x, in ? bytes_x : 0);
    MSA_LOAD_TO_LDS(rs, stage + wave * 1024 + (i < kLoadsN ? i * 4096 : kN * kRowBytes + (i - kLoadsN) * 4096), from[i], in ? step * kRowBytes : 0, 0);
  };
#pragma unroll
  for (int s = 0; s < kStages; ++s)
#pragma unroll
    for (int i = 0; i < kLoads; ++i) load(lds + s * kBuffer, first + s, i);
  int at_n[2], at_t[2];                                  // a lane's 16 bytes of row block 0 in the two halves of a K tile
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    at_n[h] = unit_at(wave_n + l15, 4 * h + g);
    at_t[h] = kN * kRowBytes + unit_at(wave_t + l15, 4 * h + g);
  }
  floatx4_t acc[kBN][kBT];
#pragma unroll
  for (int i = 0; i < kBN; ++i)
#pragma unroll
    for (int j = 0; j < kBT; ++j) {
      acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(acc[i][j]));
    }
  struct Half { bf16x8_t w[kBN], x[kBT]; } f0, f1;
  auto read = [&](Half& f, const char* buffer, int h, int i) {
    if (i < kBT) f.x[i] = *reinterpret_cast<const bf16x8_t*>(buffer + at_t[h] + i * 16 * kRowBytes);
    else f.w[i - kBT] = *reinterpret_cast<const bf16x8_t*>(buffer + at_n[h] + (i - kBT) * 16 * kRowBytes);
  };
  // the products of a half, `part` o of `count` in front of product o kM / count
  auto products = [&](const Half& f, auto count, auto part) {
#pragma unroll
    for (int m = 0; m < kM; ++m) {
#pragma unroll
      for (int o = 0; o < count(); ++o)
        if (o * kM / count() == m) part(o);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[m / kBT][m % kBT]) : "v"(f.w[m / kBT]), "v"(f.x[m % kBT]));
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier\n\ts_nop 7" ::"n"((kStages - 1) * kLoads) : "memory");
#pragma unroll
  for (int i = 0; i < kReads; ++i) read(f0, lds, 0, i);
  int now = 0;
  for (int step = first; step < last; ++step) {
    const int next = now + kBuffer == kStages * kBuffer ? 0 : now + kBuffer;
    products(f0, [] { return kReads; }, [&](int o) { read(f1, lds + now, 1, o); });
    // the next K tile is here; this one has been read by all
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((kStages - 2) * kLoads) : "memory");
    products(f1, [] { return kReads + kLoads; }, [&](int o) {
      if (o < kReads) read(f0, lds + next, 0, o);
      else load(lds + now, step + kStages, o - kReads);
    });
    now = next;
  }
  asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");      // (nothing may still be writing LDS when the workgroup ends)
#pragma unroll
  for (int i = 0; i < kBN; ++i)
#pragma unroll
    for (int j = 0; j < kBT; ++j) asm volatile("" : "+a"(acc[i][j]));
  // a lane's token of column block j, outputs 8 g + 0..7 of each 32
#pragma unroll
  for (int j = 0; j < kBT; ++j) {
    const int token = t0 + wave_t + 16 * j + l15;
    if (token >= a.T) continue;
#pragma unroll
    for (int m = 0; m < kBN / 2; ++m) {
      const int n = n0 + wave_n + 32 * m + 8 * g;
      if (n >= a.N) continue;
      if (a.pieces > 1) {
        floatx4_t* o = reinterpret_cast<floatx4_t*>(a.part + ((int64_t)piece * a.T + token) * a.N + n);
        o[0] = acc[2 * m][j];
        o[1] = acc[2 * m + 1][j];
      } else {
        const floatx4_t u = acc[2 * m][j], v = acc[2 * m + 1][j];
        finish8(a, token, n, {u[0], u[1], u[2], u[3], v[0], v[1], v[2], v[3]});
      }
    }
  }
}

// The pieces' sums, in their order: eight outputs a thread.
__global__ __launch_bounds__(256) void flow_finish_kernel(FlowArgs a) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8, all = (int64_t)a.T * a.N;
  if (i >= all) return;
  float4 p[kMaxPieces][2];
#pragma unroll
  for (int s = 0; s < kMaxPieces; ++s)
    if (s < a.pieces) {
      p[s][0] = *reinterpret_cast<const float4*>(a.part + s * all + i);
      p[s][1] = *reinterpret_cast<const float4*>(a.part + s * all + i + 4);
    }
  float v[8] = {};
#pragma unroll
  for (int s = 0; s < kMaxPieces; ++s)
    if (s < a.pieces) {
      v[0] += p[s][0].x; v[1] += p[s][0].y; v[2] += p[s][0].z; v[3] += p[s][0].w;
      v[4] += p[s][1].x; v[5] += p[s][1].y; v[6] += p[s][1].z; v[7] += p[s][1].w;
    }
  const int token = (int)(i / a.N);
  finish8(a, token, (int)(i - (int64_t)token * a.N), v);
}

template <int kN, int kT, int kStages>
int launch(FlowArgs a, hipStream_t st) {
  constexpr int lds = kStages * (kN + kT) * kRowBytes;
  static std::atomic<int> lds_limit_raised{0};
  MSA_HIP(raise_dynamic_lds_limit(lds_limit_raised, reinterpret_cast<const void*>(flow_gemm_kernel<kN, kT, kStages>), lds));
  a.tiles_t = (a.T + kT - 1) / kT;
  a.tiles_n = (a.N + kN - 1) / kN;
  const int wgs = a.tiles_t * a.tiles_n * a.pieces, share = std::max(1, wgs / kXcds);
  int64_t least = INT64_MAX;
  for (int s = 1; s <= a.tiles_n; ++s) {                 // rows that an XCD's tiles read together
    const int64_t rows = (int64_t)s * kN + (int64_t)std::min((share + s - 1) / s, a.tiles_t) * kT;
    if (rows < least) { least = rows; a.strip = s; }
  }
  flow_gemm_kernel<kN, kT, kStages><<<(wgs + kXcds - 1) / kXcds * kXcds, kThreads, lds, st>>>(a);
  MSA_LAUNCH_CHECK();
  if (a.pieces > 1) {
    flow_finish_kernel<<<(unsigned)(((int64_t)a.T * a.N / 8 + 255) / 256), 256, 0, st>>>(a);
    MSA_LAUNCH_CHECK();
  }
  return MSA_OK;
}

// The tiles, and what a K tile of them and storing them cost, us.  A launch costs 2.8 more; the operands come at 6.7 TB/s, at a share of
// that where compute units are left without a tile; pieces cost another launch of 3.5 and their sums' way at 5.6 TB/s, to and fro.  Fitted to
// the times of 14 matrices of the models by 10 numbers of tokens from 20 to 2200 (9 % off them, the best tile's time 2 % below the chosen one's).
// `behind`: with whole K behind the vendor's product.  That has tiles of its own for every size, whose times follow no measure of ours, so it is told
// tile by tile (288 products of 22 matrices and 41 numbers of tokens of 17 to 2304, weights from memory, their time over the vendor's: in pieces of K
// 0.43 to 0.98, 64 x 96 0.81 to 0.98, 128 x 160 0.81 to 0.99, 192 x 192 0.75 to 0.97, 128 x 128 0.84 to 1.03; half of them under 0.92, 0.96 and 0.97:
// 192 x 160 0.86 to 1.11, 128 x 96 0.82 to 1.10, 192 x 128 0.92 to 1.04; but 64 x 128 0.97 to 1.07, 256 x 128 1.02 to 1.09).
struct Tile { int n, t; float step, end; bool behind; };
constexpr Tile kTile[] = {{64, 32, .175f, .06f, false},   {64, 64, .208f, .83f, false},   {64, 96, .247f, .78f, false},   {64, 128, .331f, .72f, true},
                          {128, 96, .405f, 2.03f, false}, {128, 128, .485f, 2.25f, false}, {128, 160, .534f, 3.23f, false}, {192, 128, .651f, 3.27f, false},
                          {192, 160, .71f, 3.91f, false}, {192, 192, .886f, 3.99f, false}, {256, 128, .848f, 3.77f, true}};

struct Plan { int tile, pieces; float us; };
// The cheapest tile and pieces of one round; none (us = 0) where there is none.  A gated unit or gelu costs kEnd for every output of a lane, of
// which nothing is hidden where a compute unit has one tile (2000 x 1024 x 4096 in tiles of 256 x 128 21.5 us, with gelu 27.3).
constexpr float kEnd = 0.04f;
Plan plan_of(int64_t T, int32_t K, int64_t N, bool end, bool whole) {
  const int units = device_compute_units(), steps = K / kK;
  Plan best{0, 1, 0.f};
  for (int v = 0; v < (int)(sizeof(kTile) / sizeof(kTile[0])); ++v)
    for (int p = 1; p <= (whole ? 1 : kMaxPieces) && (p == 1 || p * kMinSteps <= steps); ++p) {
      const int64_t wgs = ((T + kTile[v].t - 1) / kTile[v].t) * ((N + kTile[v].n - 1) / kTile[v].n) * p;
      if (wgs > units) break;
      const float bytes = ((float)(N + T) * (float)K + (float)T * (float)N) * 2.f;
      const float ends = end && p == 1 ? kEnd * (float)(kTile[v].n * kTile[v].t / kThreads) : 0.f;
      float us = 2.8f + ends + std::max((float)((steps + p - 1) / p) * kTile[v].step + kTile[v].end, bytes / 6.7e6f * (float)units / (float)wgs);
      if (p > 1) us += 3.5f + (float)p * (float)T * (float)N * 8.f / 5.6e6f;
      if (best.us == 0.f || us < best.us) best = {v, p, us};
    }
  return best;
}

// Where this form is taken: one round.  Up to the length that block_gemm.hip's is asked for it has to be faster than that by its own measure,
// plain products by a little more (177 of them, their time over block_gemm.hip's: of the eleven whose measures are within 1 to 4 % 0.88 to 1.11).
// Behind it the vendor's product is the other choice, of plain products in tiles that are not behind it (us, weights from memory, here and the vendor's:
// 573 x 2560 x 12384 47.8 and 44.7, 640 x 4096 x 2560 29.1 and 27.1); an end saves the launch that it needs besides.  With fewer tokens the weights' way
// is all there is, which more workgroups of smaller tiles do better, except for long rows, which are cut (us, the faster other form and here: 100 x 2560 x 12288
// 22.9 and 24.4, 48 x 2560 x 8480 16.2 and 18.3, but 48 x 9728 x 2560 20.4 and 17.1, 20 x 5120 x 2560 15.1 and 12.1).  More tokens and shorter rows
// were not measured.  (Behind 2304 tokens full rounds are level with the vendor's, 4096 x 3072 x 1024 29.6 and 29.2, 8192 47.0 and 50.6; tiles of
// 256 x 160 to 256 x 256 are behind it, 850 x 2560 x 12368 53.9 and 65.3.)
constexpr float kBlockUs = 23.f, kSure = 0.96f, kSooner = 0.99f;
constexpr int64_t kLeastTokens = 17, kTokens = 160, kMostTokens = 2304;
constexpr int32_t kLong = 3072, kShort = 1024;

}  // namespace

extern "C" float msa_flow_linear_us(int64_t T, int32_t K, int32_t N, int32_t mode) {
  if (T < kLeastTokens || T > kMostTokens || K < kShort || K > 32768 || K % kK != 0 || N < 16 || N >= (1 << 20) || (T < kTokens && K < kLong)) return 0.f;
  const bool end = mode != MSA_TILE_STORE;
  const Plan plan = plan_of(T, K, N, end, false);
  const float block = msa_block_linear_us(T, K, N);
  const bool taken = block <= kBlockUs ? plan.us < (end ? kSooner : kSure) * block : end || plan.pieces > 1 || !kTile[plan.tile].behind;
  return taken ? plan.us : 0.f;
}

extern "C" size_t msa_flow_workspace_bytes(int64_t T, int32_t K, int32_t N, int32_t mode) {
  if (T <= 0 || K < kK || N <= 0) return 0;
  const Plan plan = plan_of(T, K, N, mode != MSA_TILE_STORE, false);
  return plan.us > 0.f && plan.pieces > 1 ? (size_t)plan.pieces * (size_t)T * (size_t)N * sizeof(float) : 0;
}

extern "C" int msa_flow_linear(const void* x, int64_t ldx, int64_t T, int32_t K, const void* w, int32_t N, const msa_tile_end* end, void* out, int64_t ldo,
                               void* workspace, size_t workspace_bytes, void* stream) {
  MSA_REQUIRE(x && w && out && end, "msa_flow_linear: null pointer");
  const int mode = end->mode;
  MSA_REQUIRE(mode == MSA_TILE_STORE || mode == MSA_TILE_GLU || mode == MSA_TILE_GELU, "msa_flow_linear: mode %d", mode);
  MSA_REQUIRE(T > 0 && T < ((int64_t)1 << 22) && K >= kK && K % kK == 0 && K <= 32768 && N > 0 && N < (1 << 20) && N % (mode == MSA_TILE_GLU ? 16 : 8) == 0,
              "msa_flow_linear: T=%lld K=%d (a multiple of 64 up to 32768) N=%d", (long long)T, K, N);
  MSA_REQUIRE(ldx >= K && ldx % 8 == 0 && ldx < ((int64_t)1 << 21) && ldo >= (mode == MSA_TILE_GLU ? N / 2 : N) && ldo % 8 == 0,
              "msa_flow_linear: row strides %lld and %lld", (long long)ldx, (long long)ldo);
  MSA_REQUIRE(mode != MSA_TILE_GELU || (end->gelu_n >= 0 && end->gelu_n <= N && end->gelu_n % 8 == 0), "msa_flow_linear: gelu_n=%d", end->gelu_n);
  MSA_REQUIRE((((uintptr_t)x | (uintptr_t)w | (uintptr_t)out | (uintptr_t)workspace) & 15) == 0, "msa_flow_linear: operands must be 16-byte aligned");
  const bool with_end = mode != MSA_TILE_STORE;
  Plan plan = plan_of(T, K, N, with_end, false);
  if (plan.pieces > 1 && (workspace == nullptr || workspace_bytes < msa_flow_workspace_bytes(T, K, N, mode))) plan = plan_of(T, K, N, with_end, true);
  if (plan.us == 0.f) return msa_block_linear(x, ldx, T, K, w, N, end, out, ldo, stream);      // (more than a round)
  const FlowArgs a{static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), static_cast<bf16_t*>(out), static_cast<float*>(workspace), ldx, ldo,
                   (int32_t)T, K, N, 0, 0, 1, plan.pieces, *end};
  hipStream_t st = as_stream(stream);
  switch (kTile[plan.tile].n * 1000 + kTile[plan.tile].t) {
    case 64032: return launch<64, 32, 5>(a, st);
    case 64064: return launch<64, 64, 5>(a, st);
    case 64096: return launch<64, 96, 4>(a, st);
    case 64128: return launch<64, 128, 3>(a, st);
    case 128096: return launch<128, 96, 5>(a, st);
    case 128128: return launch<128, 128, 4>(a, st);
    case 128160: return launch<128, 160, 4>(a, st);
    case 192128: return launch<192, 128, 4>(a, st);
    case 192160: return launch<192, 160, 3>(a, st);
    case 192192: return launch<192, 192, 3>(a, st);
    case 256128: return launch<256, 128, 3>(a, st);
  }
  msa_set_error("msa_flow_linear: no kernel of tile %d", plan.tile);
  return MSA_EINVAL;
}
