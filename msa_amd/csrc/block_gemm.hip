// y[T, N] = x[T, K] . w[N, K]^T in bf16 with fp32 sums for blocks of tokens that leave the 256 x 256 tiles of gemm.hip without work for the
// chip: the products of short prompts (the projections around the sequence layers of the mixed-layer decoders), a few microseconds each.
//
// A workgroup makes a tile of kN weight rows and kT tokens.  What bounds it is the chain of a K tile (wait, LDS write, barrier, LDS read,
// matrix cores), so kAhead K tiles are on their way in registers, LDS has two buffers with one barrier a K tile, and the tile is the one
// whose rounds over the compute units cost least (block_us).  us a K tile of 64, one workgroup per compute unit: 64 x 32 with four
// wavefronts 0.18, 64 x 64 with eight 0.21 (with four 0.26), 128 x 64 with eight 0.32, 128 x 128 with eight 0.50 (with four 0.68).  Twice
// the K tile a barrier (64 x 64: 6.6 us for 64 x 1024 x 1024 against 6.4) and eight K tiles ahead (5.3 against 5.0) gain nothing;
// wavefronts that share a tile by K and load their fragments without LDS take 6.3 there and 20 for 1000 rows, against 7: a fragment's
// load touches sixteen lines, a row-wise one eight.
// Whole calls, us, the vendor's and here: 64 x 1024 x 1024 6.6 and 5.0, 300 x 1024 x 6176 11.7 and 9.2, 573 x 1024 x 4096 13.4 and 11.8, 1000 x
// 3072 x 1024 15.1 and 14.4, 2048 x 1024 x 4096 20.6 and 22.1.
//
// The weights are the MFMA's A operand, the tokens its B operand: a lane holds outputs of one token, and with the weight rows of a tile
// in the order of `weight_row` eight neighbouring ones of two row blocks, which leave in one store.
#include <algorithm>

#include "common.h"
#include "seq_common.h"
#include "seq_mfma.h"

namespace {

enum { kStore = MSA_TILE_STORE, kGlu = MSA_TILE_GLU, kGelu = MSA_TILE_GELU };
constexpr int kK = 64, kRowBytes = 2 * kK, kUnits = kRowBytes / 16;      // K elements of a K tile, bytes and 16-byte units of a row of it
constexpr int kXcds = 8;

struct BlockArgs {
  const bf16_t* x;          // [T, K], rows ldx apart
  const bf16_t* w;          // [N, K]
  bf16_t* out;              // [T, N] (or [T, N / 2]), rows ldo apart
  int64_t ldx, ldo;
  int32_t T, K, N;
  int32_t tiles_t, tiles;   // of tokens, of both
  msa_tile_end end;
};

// LDS row -> weight row: row block i, lane group g, register r of a fragment's 32 rows is row 8 g + 4 i + r.
__device__ __forceinline__ int weight_row(int lds_row) {
  return (lds_row & ~31) + 8 * ((lds_row >> 2) & 3) + 4 * ((lds_row >> 4) & 1) + (lds_row & 3);
}
// 16-byte units of a row lie in an order that spreads a fragment's sixteen rows over all banks.
__device__ __forceinline__ int unit_at(int row, int unit) { return row * kRowBytes + ((unit ^ ((row >> 1) & 7)) << 4); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const bf16_t* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p), 0, bytes, 0x00020000);
}

template <int kN, int kT, int kWN, int kWT, int kAhead, int kMode>
__global__ __launch_bounds__(kWN * kWT * 64) void block_gemm_kernel(BlockArgs a) {
  constexpr int kThreads = kWN * kWT * 64;
  constexpr int kLoadsN = kN * kUnits / kThreads, kLoadsT = kT * kUnits / kThreads;
  constexpr int kBlocksN = kN / kWN / 16, kBlocksT = kT / kWT / 16;         // 16 x 16 blocks of a wavefront
  constexpr int kBuffer = (kN + kT) * kRowBytes;
  __shared__ __align__(16) char lds[2 * kBuffer];
  // an XCD's workgroups (dealt round-robin) take neighbouring tiles, the tokens' innermost: a weight tile is read into one L2 only
  const int per_xcd = gridDim.x / kXcds, id = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
  if (id >= a.tiles) return;
  const int tile_n = id / a.tiles_t, t0 = (id - tile_n * a.tiles_t) * kT, n0 = tile_n * kN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l15 = lane & 15, g = lane >> 4;
  const int wave_n = wave / kWT * (kN / kWN), wave_t = wave % kWT * (kT / kWT);
  const bf16_t* w = a.w + (int64_t)n0 * a.K;
  const bf16_t* x = a.x + (int64_t)t0 * a.ldx;
  const int bytes_w = min(kN, a.N - n0) * a.K * 2, bytes_x = ((min(kT, a.T - t0) - 1) * (int)a.ldx + a.K) * 2;
  // rows behind the last read as zero (the K displacement is scalar and stays inside a row), and so do K tiles behind the last
  int from[kLoadsN + kLoadsT], to[kLoadsN + kLoadsT];
#pragma unroll
  for (int i = 0; i < kLoadsN + kLoadsT; ++i) {
    const int at = tid + kThreads * (i < kLoadsN ? i : i - kLoadsN), row = at / kUnits, unit = at % kUnits;
    from[i] = (i < kLoadsN ? weight_row(row) * a.K : row * (int)a.ldx) * 2 + unit * 16;
    to[i] = (i < kLoadsN ? 0 : kN * kRowBytes) + unit_at(row, unit);
  }
  const int steps = a.K / kK;
  u32x4_t ahead[kAhead][kLoadsN + kLoadsT];
  auto request = [&](u32x4_t (&r)[kLoadsN + kLoadsT], int step) {
    const bool in = step < steps;
    const __amdgpu_buffer_rsrc_t rw = rows_rsrc(w, in ? bytes_w : 0), rx = rows_rsrc(x, in ? bytes_x : 0);
    const int k = in ? step * kRowBytes : 0;
#pragma unroll
    for (int i = 0; i < kLoadsN + kLoadsT; ++i) r[i] = __builtin_amdgcn_raw_buffer_load_b128(i < kLoadsN ? rw : rx, from[i], k, 0);
    __builtin_amdgcn_sched_barrier(0);             // (in this order: a K tile's wait counts what was requested behind it)
  };
#pragma unroll
  for (int i = 0; i < kAhead; ++i) request(ahead[i], i);
  int at_n[2], at_t[2];                                  // a lane's 16 bytes of row block 0 in the two halves of a K tile
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    at_n[h] = unit_at(wave_n + l15, 4 * h + g);
    at_t[h] = kN * kRowBytes + unit_at(wave_t + l15, 4 * h + g);
  }
  floatx4_t acc[kBlocksN][kBlocksT];
#pragma unroll
  for (int i = 0; i < kBlocksN; ++i)
#pragma unroll
    for (int j = 0; j < kBlocksT; ++j) acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};

  for (int step = 0; step < steps; step += kAhead) {
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      char* buffer = lds + (u & 1) * kBuffer;
#pragma unroll
      for (int i = 0; i < kLoadsN + kLoadsT; ++i) *reinterpret_cast<u32x4_t*>(buffer + to[i]) = ahead[u][i];
      request(ahead[u], step + u + kAhead);
      __syncthreads();
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        bf16x8_t wf[kBlocksN], xf[kBlocksT];
#pragma unroll
        for (int i = 0; i < kBlocksN; ++i) wf[i] = *reinterpret_cast<const bf16x8_t*>(buffer + at_n[h] + i * 16 * kRowBytes);
#pragma unroll
        for (int j = 0; j < kBlocksT; ++j) xf[j] = *reinterpret_cast<const bf16x8_t*>(buffer + at_t[h] + j * 16 * kRowBytes);
#pragma unroll
        for (int i = 0; i < kBlocksN; ++i)
#pragma unroll
          for (int j = 0; j < kBlocksT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i], xf[j], acc[i][j], 0, 0, 0);
      }
    }
  }
  // a lane's token of column block j, outputs 8 g + 0..7 of each 32
#pragma unroll
  for (int j = 0; j < kBlocksT; ++j) {
    const int token = t0 + wave_t + 16 * j + l15;
    if (token >= a.T) continue;
#pragma unroll
    for (int m = 0; m < kBlocksN / 2; ++m) {
      const int n = n0 + wave_n + 32 * m + 8 * g;
      if (n >= a.N) continue;
      uint32_t p[4];                                     // the product, rounded as it would be on its way through memory
#pragma unroll
      for (int e = 0; e < 4; ++e) p[e] = pack_bf16x2(acc[2 * m + (e >> 1)][j][2 * (e & 1)], acc[2 * m + (e >> 1)][j][2 * (e & 1) + 1]);
      bf16_t* out = a.out + (int64_t)token * a.ldo;
      if constexpr (kMode == kGlu) {
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = clamped_glu_f(bf16lo(p[e]), bf16hi(p[e]), a.end.limit, a.end.alpha, a.end.shift);
        *reinterpret_cast<uint2*>(out + n / 2) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
      } else {
        if (kMode == kGelu && n < a.end.gelu_n)
#pragma unroll
          for (int e = 0; e < 4; ++e) p[e] = pack_bf16x2(gelu_tanh_f(bf16lo(p[e])), gelu_tanh_f(bf16hi(p[e])));
        *reinterpret_cast<uint4*>(out + n) = make_uint4(p[0], p[1], p[2], p[3]);
      }
    }
  }
}

template <int kN, int kT, int kWN, int kWT, int kAhead>
int launch(BlockArgs a, hipStream_t st) {
  static_assert(kAhead % 2 == 0, "a K tile's buffer is its number in the unrolled loop");
  constexpr int kThreads = kWN * kWT * 64;
  a.tiles_t = (a.T + kT - 1) / kT;
  a.tiles = a.tiles_t * ((a.N + kN - 1) / kN);
  const int grid = (a.tiles + kXcds - 1) / kXcds * kXcds;
  if (a.end.mode == kGlu) block_gemm_kernel<kN, kT, kWN, kWT, kAhead, kGlu><<<grid, kThreads, 0, st>>>(a);
  else if (a.end.mode == kGelu) block_gemm_kernel<kN, kT, kWN, kWT, kAhead, kGelu><<<grid, kThreads, 0, st>>>(a);
  else block_gemm_kernel<kN, kT, kWN, kWT, kAhead, kStore><<<grid, kThreads, 0, st>>>(a);
  MSA_LAUNCH_CHECK();
  return MSA_OK;
}

// The tiles, and what a K tile of them and storing them costs, us (half way between one workgroup on a compute unit and several).
enum { k64x32, k64x64, k128x64, k128x128, kTiles };
struct Tile { int n, t; float step, end; };
constexpr Tile kTile[kTiles] = {{64, 32, 0.18f, 0.2f}, {64, 64, 0.225f, 0.4f}, {128, 64, 0.325f, 0.9f}, {128, 128, 0.52f, 1.8f}};

// The best tile for a product and what it takes about: a launch's 2.3 us, and its rounds or the operands' and results' way.
float block_us(int64_t T, int32_t K, int64_t N, int& best) {
  const int units = std::max(1, device_compute_units());
  float least = 0.f;
  for (int v = 0; v < kTiles; ++v) {
    const int64_t tiles = ((T + kTile[v].t - 1) / kTile[v].t) * ((N + kTile[v].n - 1) / kTile[v].n);
    const float us = (kTile[v].step * (float)(K / kK) + kTile[v].end) * (float)((tiles + units - 1) / units);
    if (v == 0 || us < least) { least = us; best = v; }
  }
  return 2.3f + std::max(least, ((float)(N + T) * (float)K + (float)T * (float)N) * 2.f / 3.5e6f);
}

}  // namespace

extern "C" float msa_block_linear_us(int64_t T, int32_t K, int32_t N) {
  int best;
  return T > 0 && K >= kK && N > 0 ? block_us(T, K, N, best) : 0.f;
}

extern "C" int msa_block_linear(const void* x, int64_t ldx, int64_t T, int32_t K, const void* w, int32_t N, const msa_tile_end* end, void* out,
                                int64_t ldo, void* stream) {
  MSA_REQUIRE(x && w && out && end, "msa_block_linear: null pointer");
  const int mode = end->mode;
  MSA_REQUIRE(mode == kStore || mode == kGlu || mode == kGelu, "msa_block_linear: mode %d", mode);
  MSA_REQUIRE(T > 0 && T < ((int64_t)1 << 22) && K >= kK && K % kK == 0 && K <= 32768 && N > 0 && N < (1 << 20) && N % (mode == kGlu ? 16 : 8) == 0,
              "msa_block_linear: T=%lld K=%d (a multiple of 64 up to 32768) N=%d", (long long)T, K, N);
  MSA_REQUIRE(ldx >= K && ldx % 8 == 0 && ldx < ((int64_t)1 << 21) && ldo >= (mode == kGlu ? N / 2 : N) && ldo % 8 == 0,
              "msa_block_linear: row strides %lld and %lld", (long long)ldx, (long long)ldo);
  MSA_REQUIRE(mode != kGelu || (end->gelu_n >= 0 && end->gelu_n <= N && end->gelu_n % 8 == 0), "msa_block_linear: gelu_n=%d", end->gelu_n);
  MSA_REQUIRE((((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) == 0, "msa_block_linear: x, w and out must be 16-byte aligned");
  const BlockArgs a{static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), static_cast<bf16_t*>(out), ldx, ldo, (int32_t)T, K, N, 0, 0, *end};
  int best;
  block_us(T, K, N, best);
  switch (best) {
    case k64x32: return launch<64, 32, 2, 2, 4>(a, as_stream(stream));
    case k64x64: return launch<64, 64, 2, 4, 4>(a, as_stream(stream));
    case k128x64: return launch<128, 64, 4, 2, 4>(a, as_stream(stream));
    default: return launch<128, 128, 4, 2, 2>(a, as_stream(stream));
  }
}
