// Products of a block of tokens with a weight matrix, y[T, N] = x[T, K] . w[N, K]^T in bf16 with fp32 sums, finished in registers:
// stored, added to a residual stream, gated (silu(gate) up), or taken apart into heads with their RMSNorm and rotary (the projections
// of src/msa/memory_sparse_attention.py:125-133, 178, 263 and the MLP around them).
//
// What bounds a large product here is power: the clock falls until the chip is inside its budget, so what counts is energy per product
// (32771 x 2560 x 19456 with silu-mul: matrix cores busy 0.76 of the cycles at 1.79 GHz, of 2.4; the smaller ones below 0.7 of 2.1).
// Hence the K step of the routing scan (gen_scan_asm.py): a 256 x 256 tile by four wavefronts of 128 x 128 (a third fewer LDS operand
// reads than eight of 64 x 128), v_mfma_f32_16x16x32_bf16, operand tiles straight into LDS two steps ahead, one barrier a step, a
// workgroup per compute unit walking over its tiles as one sequence of steps.
//
// The weights are the MFMA's A operand, the tokens its B operand: a lane holds values of ONE token (column l % 16 of a column block).
// The weight rows of a tile are put into LDS in an order that gives a lane eight neighbouring outputs of two row blocks (or the gates
// and ups of eight outputs of four), so that a token's outputs leave in 16-byte stores, 64 contiguous bytes a token and instruction,
// the rotary partners d and d + 64 are registers of one lane, and nothing passes LDS on its way out.
#include <algorithm>

#include "common.h"
#include "seq_common.h"

namespace {

#include "gemm_asm.inc"

constexpr int kRowBytes = 128;                 // one K tile of a row: 64 bf16
constexpr int kTile = 256, kThreads = 256;
constexpr int kLdsBytes = 5 * kTile * kRowBytes;         // two stages of the weight tile, three of the token tile (the statements' addresses)
constexpr int kCompilerVgprs = 128;            // the compiler's share of the vector registers
constexpr int kXcds = 8;
constexpr int kPieceBytes = kTile * kTile * 4;

enum { kStore = MSA_TILE_STORE, kAdd = MSA_TILE_ADD, kSiluMul = MSA_TILE_SILU_MUL, kHeads = 3, kGlu = MSA_TILE_GLU, kGelu = MSA_TILE_GELU };
constexpr bool is_pair(int mode) { return mode == kSiluMul || mode == kGlu; }      // two weight rows an output

struct TileArgs {
  const bf16_t* x;          // [T, K], rows ldx apart
  const bf16_t* w;          // [N, K]
  bf16_t* out;              // [T, N] (or [T, N / 2]), rows ldo apart
  float* pieces;            // partial tiles
  int64_t ldx, ldo;
  int32_t T, K, N;
  int32_t tiles_t, tiles_n, group;
  int32_t split;            // K pieces of a tile of the last, incomplete round
  int32_t max_rem;          // tiles of that round in the XCD that has most of them
  int32_t stream;           // the output is larger than what the caches would keep for its reader: stored non-temporal
  msa_tile_end end;
  float rate;               // -log2(e) alpha
  // kHeads: w's heads are front plain heads | q | k | v | back plain heads
  const int64_t* pos;       // [T]
  const bf16_t* q_norm_w;   // [128]
  const bf16_t* k_norm_w;   // [128]
  const float* rope_cos;    // [rope_rows, 64]
  const float* rope_sin;
  bf16_t* q_out;            // [T, Hq, 128]
  bf16_t* k_out;            // [T, Hkv, 128]
  bf16_t* v_out;            // [T, Hkv, 128]
  bf16_t* r_out;            // [T, Hr_front + Hr_back, 128]
  int32_t Hq, Hkv, Hr_front, Hr_back;
  int32_t rope_rows;
  float eps;
};

// The walk.  Tiles in linear order: groups of `group` token tiles, inside a group all weight tiles, the group's token tiles innermost,
// so that the 32 workgroups of an XCD (dealt round-robin) share a few token and weight tiles in their L2.  An XCD takes an eighth of that
// order, its workgroups a tile each per round.  The tiles of the last, incomplete round are cut into `split` pieces of K each, so that
// all workgroups have a share of them; the pieces meet in tile_finish_kernel.
struct Share {
  int first, rounds, rem;   // the XCD's first tile, complete rounds, tiles of the incomplete one
};

__host__ __device__ inline Share tile_share(int tiles, int per_xcd, int xcd) {
  const int lo = (int)((int64_t)tiles * xcd / kXcds), hi = (int)((int64_t)tiles * (xcd + 1) / kXcds);
  return {lo, (hi - lo) / per_xcd, (hi - lo) % per_xcd};
}

// what a workgroup multiplies: K tiles k0 .. k0 + nk of a tile; piece < 0: all of it
struct Item {
  int tile_t, tile_n, k0, nk, piece;
};

__device__ inline void tile_at(const TileArgs& a, int linear, int& tile_t, int& tile_n) {
  const int per_group = a.tiles_n * a.group;
  const int g = linear / per_group, rem = linear - g * per_group;
  const int width = min(a.group, a.tiles_t - g * a.group);
  tile_n = rem / width;
  tile_t = g * a.group + rem - tile_n * width;
}

// Item `n` of workgroup (xcd, slot); false: there is none.  (nothing here depends on the lane)
__device__ inline bool item_at(const TileArgs& a, const Share& share, int xcd, int slot, int per_xcd, int k_tiles, int n, Item& it) {
  if (n < share.rounds) {
    tile_at(a, share.first + n * per_xcd + slot, it.tile_t, it.tile_n);
    it.k0 = 0; it.nk = k_tiles; it.piece = -1;
    return true;
  }
  const int at = (n - share.rounds) * per_xcd + slot;
  if (at >= share.rem * a.split) return false;
  const int p = at / share.rem;
  const int u = at - p * share.rem;
  tile_at(a, share.first + share.rounds * per_xcd + u, it.tile_t, it.tile_n);
  it.k0 = (int)((int64_t)k_tiles * p / a.split);
  it.nk = (int)((int64_t)k_tiles * (p + 1) / a.split) - it.k0;
  it.piece = a.split == 1 ? -1 : (xcd * a.max_rem + u) * a.split + p;
  return true;
}

// Output of a lane's value: row block i (of eight), register r, lane group g.
//  kStore, kAdd, kGelu, kHeads: weight row 32 (i / 2) + 8 g + 4 (i % 2) + r of the wavefront's 128
//  kSiluMul, kGlu: output 32 (i / 4) + 8 g + 4 (i % 2) + r of its 64, gate in blocks with i / 2 even, up in the others; the weight's
//                  rows are 8 gates, 8 ups, 8 gates, ... (kSiluMul) or gate, up, gate, ... (kGlu)
template <int kMode>
__host__ __device__ inline int weight_row(int lds_row) {
  const int wave_rows = lds_row & ~127, i = (lds_row >> 4) & 7, g = (lds_row >> 2) & 3, r = lds_row & 3;
  if (is_pair(kMode)) {
    const int o = 32 * (i >> 2) + 8 * g + 4 * (i & 1) + r, up = (i >> 1) & 1;
    return wave_rows + (kMode == kGlu ? 2 * o + up : 16 * (o >> 3) + (o & 7) + 8 * up);
  }
  return wave_rows + 32 * (i >> 1) + 8 * g + 4 * (i & 1) + r;
}

__device__ __forceinline__ uint4 pack8(const float* v) {
  return make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
}

__device__ __forceinline__ void unpack8(const uint4& w, float* v) {
  v[0] = bf16lo(w.x); v[1] = bf16hi(w.x); v[2] = bf16lo(w.y); v[3] = bf16hi(w.y);
  v[4] = bf16lo(w.z); v[5] = bf16hi(w.z); v[6] = bf16lo(w.w); v[7] = bf16hi(w.w);
}

// Two 16-byte groups of every token, 32 columns apart, of which a lane has the parts behind column 8 g: token t's lanes and those of
// token t + 8 change halves first, so that a store writes whole cache lines of eight tokens (halves of sixteen cost a product of
// 32771 x 2560 x 19456 2217 us, whole lines 2170).  `to` is the lane's token's first group.
__device__ __forceinline__ uint32_t other_half(uint32_t v) { return __builtin_amdgcn_mov_dpp(v, 0x128, 0xf, 0xf, false); }     // row_ror:8
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void store16(bf16_t* to, const uint4& v, bool stream) {
  if (stream) __builtin_nontemporal_store(u32x4_t{v.x, v.y, v.z, v.w}, reinterpret_cast<u32x4_t*>(to));
  else *reinterpret_cast<uint4*>(to) = v;
}
__device__ __forceinline__ void store_lines(bf16_t* to, int64_t ld, int token, int T, int columns, uint4 p0, uint4 p1, bool stream) {
  const bool low = (threadIdx.x & 8) == 0;
  const uint4 x = make_uint4(other_half(low ? p1.x : p0.x), other_half(low ? p1.y : p0.y), other_half(low ? p1.z : p0.z), other_half(low ? p1.w : p0.w));
  p0 = make_uint4(low ? p0.x : x.x, low ? p0.y : x.y, low ? p0.z : x.z, low ? p0.w : x.w);
  p1 = make_uint4(low ? x.x : p1.x, low ? x.y : p1.y, low ? x.z : p1.z, low ? x.w : p1.w);
  const int first = low ? token : token - 8;
  bf16_t* row = to + (low ? (int64_t)0 : 32 - 8 * ld);
  if ((low ? 0 : 32) < columns) {
    if (first < T) store16(row, p0, stream);
    if (first + 8 < T) store16(row + 8 * ld, p1, stream);
  }
}

// Sum over the four lanes that hold a column.
__device__ __forceinline__ float column_sum(float v) {
  v += __shfl_xor(v, 16);
  return v + __shfl_xor(v, 32);
}

// Epilogue of a wavefront's 128 weight rows x 16 tokens (a column block): a lane has token `token` and the values v[4 i + r].
// kRounded: the gated ends and gelu take the sums rounded to bf16, as tile_flow_kernel does of the call's whole tiles: a token's result
// does not depend on which tiles are cut into pieces.
template <int kMode, bool kRounded = false>
struct Finish {
  static __device__ __forceinline__ float taken(float sum) { return kRounded ? bf16_to_f32(f32_to_bf16(sum)) : sum; }
  const TileArgs& a;
  int n0, g;                // first weight row of the wavefront, lane group
  // kHeads
  bf16_t* dst = nullptr;
  const bf16_t* norm_w = nullptr;
  int heads = 0, head_at = 0;
  uint4 nw[4];

  __device__ Finish(const TileArgs& a, int n0, int lane) : a(a), n0(n0), g(lane >> 4) {
    if constexpr (kMode == kHeads) {
      const int head = n0 / kHeadDim;
      const int h_q0 = a.Hr_front, h_k0 = h_q0 + a.Hq, h_v0 = h_k0 + a.Hkv, h_b0 = h_v0 + a.Hkv, h_end = h_b0 + a.Hr_back;
      if (head >= h_end) return;                   // half of the last tile may lie behind the last head
      if (head < h_q0) { dst = a.r_out; heads = a.Hr_front + a.Hr_back; head_at = head; }
      else if (head < h_k0) { dst = a.q_out; heads = a.Hq; head_at = head - h_q0; norm_w = a.q_norm_w; }
      else if (head < h_v0) { dst = a.k_out; heads = a.Hkv; head_at = head - h_k0; norm_w = a.k_norm_w; }
      else if (head < h_b0) { dst = a.v_out; heads = a.Hkv; head_at = head - h_v0; }
      else { dst = a.r_out; heads = a.Hr_front + a.Hr_back; head_at = a.Hr_front + head - h_b0; }
      if (norm_w != nullptr)
#pragma unroll
        for (int m = 0; m < 4; ++m) nw[m] = *reinterpret_cast<const uint4*>(norm_w + 32 * m + 8 * g);
    }
  }

  // the token's row of the rotary tables, inside them whatever its position: a block's first layer runs before the host has heard that one
  // is refused
  __device__ int table_row(int token) const {
    return token < a.T ? (int)min(max((int64_t)0, a.pos[token]), (int64_t)a.rope_rows - 1) : 0;
  }

  // What a token's outputs need from memory, in parts.  A part of the next token's is requested when this one's has been used: what
  // follows covers the latency, and one set of registers does.
  struct Ahead {
    float4 cs[2][2], sn[2][2];
    uint4 res[4];
  };
  __device__ void request(int m, int token, int row, Ahead& h) const {
    if constexpr (kMode == kHeads) {
      if (norm_w == nullptr || m >= 2) return;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        h.cs[m][u] = *reinterpret_cast<const float4*>(a.rope_cos + (int64_t)row * 64 + 32 * m + 8 * g + 4 * u);
        h.sn[m][u] = *reinterpret_cast<const float4*>(a.rope_sin + (int64_t)row * 64 + 32 * m + 8 * g + 4 * u);
      }
    } else if constexpr (kMode == kAdd) {
      const int n = n0 + 32 * m + 8 * g;
      h.res[m] = token < a.T && n < a.N ? *reinterpret_cast<const uint4*>(a.out + (int64_t)token * a.ldo + n) : make_uint4(0, 0, 0, 0);
    }
  }
  // next: the token whose parts are requested (its table row), behind T there is none
  __device__ void finish(int token, float (&v)[32], Ahead& h, bool more, int next, int next_row) {
    if constexpr (kMode == kStore || kMode == kAdd || kMode == kGelu) {
      bf16_t* row = a.out + (int64_t)token * a.ldo + n0 + 8 * g;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        if constexpr (kMode == kAdd) {
          float o[8];
          unpack8(h.res[m], o);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[8 * m + e] += o[e];
          if (more) request(m, next, next_row, h);
        }
        if constexpr (kMode == kGelu) {
          if (n0 < a.end.gelu_n) {                 // (the same for all lanes)
            const bool through = n0 + 32 * m + 8 * g < a.end.gelu_n;
#pragma unroll
            for (int e = 0; e < 8; ++e) v[8 * m + e] = through ? gelu_tanh_f(taken(v[8 * m + e])) : v[8 * m + e];
          }
        }
        if (m & 1) store_lines(row + 32 * (m - 1), a.ldo, token, a.T, a.N - (n0 + 32 * (m - 1) + 8 * g), pack8(v + 8 * m - 8), pack8(v + 8 * m), a.stream);
      }
    } else if constexpr (is_pair(kMode)) {
      const int n1 = n0 / 2;
      uint4 packed[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float gate = taken(v[16 * m + e]), up = taken(v[16 * m + 8 + e]);
          o[e] = kMode == kGlu ? clamped_glu_f(gate, up, a.end.limit, a.end.alpha, a.end.shift) : silu_f(gate) * up;
        }
        packed[m] = pack8(o);
      }
      store_lines(a.out + (int64_t)token * a.ldo + n1 + 8 * g, a.ldo, token, a.T, a.N / 2 - (n1 + 8 * g), packed[0], packed[1], a.stream);
    } else {
      if (dst == nullptr) return;
      if (norm_w != nullptr) {
        float ssq = 0.f;
#pragma unroll
        for (int e = 0; e < 32; ++e) ssq += v[e] * v[e];
        const float inv = rsqrtf(column_sum(ssq) * (1.0f / kHeadDim) + a.eps);
#pragma unroll
        for (int m = 0; m < 2; ++m) {          // dims d = 32 m + 8 g + e and d + 64
          float wl[8], wh[8];
          // (the weights stay packed between the tokens: unpacked once for all of them they would take 32 registers)
          asm volatile("" : "+v"(nw[m].x), "+v"(nw[m].y), "+v"(nw[m].z), "+v"(nw[m].w), "+v"(nw[m + 2].x), "+v"(nw[m + 2].y), "+v"(nw[m + 2].z),
                       "+v"(nw[m + 2].w));
          unpack8(nw[m], wl);
          unpack8(nw[m + 2], wh);
          const float cs[8] = {h.cs[m][0].x, h.cs[m][0].y, h.cs[m][0].z, h.cs[m][0].w, h.cs[m][1].x, h.cs[m][1].y, h.cs[m][1].z, h.cs[m][1].w};
          const float sn[8] = {h.sn[m][0].x, h.sn[m][0].y, h.sn[m][0].z, h.sn[m][0].w, h.sn[m][1].x, h.sn[m][1].y, h.sn[m][1].z, h.sn[m][1].w};
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float lo = v[8 * m + e] * (inv * wl[e]), hi = v[16 + 8 * m + e] * (inv * wh[e]);
            v[8 * m + e] = lo * cs[e] - hi * sn[e];
            v[16 + 8 * m + e] = hi * cs[e] + lo * sn[e];
          }
          if (more) request(m, next, next_row, h);
        }
      }
      bf16_t* row = dst + ((int64_t)token * heads + head_at) * kHeadDim + 8 * g;
#pragma unroll
      for (int m = 0; m < 4; m += 2)
        store_lines(row + 32 * m, (int64_t)heads * kHeadDim, token, a.T, kHeadDim, pack8(v + 8 * m), pack8(v + 8 * m + 8), a.stream);
    }
  }
};

#if defined(__HIP_DEVICE_COMPILE__)
// Per-lane constants of the asm statements: LDS offsets of the operand fragments of the two sub-steps, and the global offsets of the
// lane's 16 bytes in the wavefront's eight 1 KB blocks of either tile (lane l lands at byte 16 l of its block, row l / 8, unit slot
// l % 8, and fetches the unit that belongs there).
template <int kMode>
__device__ __forceinline__ void set_operand_registers(int lane, int wave, int ldw, int ldx) {
  int v[4];
#define MSA_GEMM_SET(TEXT) asm volatile(TEXT ::"v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]) : MSA_GEMM_CLOBBERS)
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int sw = ((s * 4 + (lane >> 4)) ^ (((lane & 15) >> 1) & 7)) * 16;
    v[s] = ((wave >> 1) * 128 + (lane & 15)) * 128 + sw;
    v[2 + s] = ((wave & 1) * 128 + (lane & 15)) * 128 + sw;
  }
  MSA_GEMM_SET(MSA_GEMM_SET_ADDR);
  auto blocks = [&](int first, bool weights) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = (wave * 8 + first + i) * 8 + (lane >> 3);
      v[i] = (weights ? weight_row<kMode>(row) * ldw : row * ldx) + ((lane & 7) ^ ((row >> 1) & 7)) * 16;
    }
  };
  blocks(0, true);
  MSA_GEMM_SET(MSA_GEMM_SET_VOFF_A0);
  blocks(4, true);
  MSA_GEMM_SET(MSA_GEMM_SET_VOFF_A1);
  blocks(0, false);
  MSA_GEMM_SET(MSA_GEMM_SET_VOFF_B0);
  blocks(4, false);
  MSA_GEMM_SET(MSA_GEMM_SET_VOFF_B1);
#undef MSA_GEMM_SET
}

// One resource per operand tile whose extent is the valid part of the tile: rows behind the last read as zero (the K displacement is
// scalar and stays inside a row).  A tile that does not exist gets an empty extent.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rows(const bf16_t* base, int ld, int row_bytes, int tile, int rows, bool valid) {
  const int n = min(kTile, rows - tile * kTile);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(base)) + (valid ? (int64_t)tile * kTile * ld : 0), 0,
                                           valid ? (n - 1) * ld + row_bytes : 0, 0x00020000);
}
#endif

template <int kMode>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_num_vgpr(kCompilerVgprs))) void tile_gemm_kernel(TileArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int per_xcd = gridDim.x / kXcds, xcd = blockIdx.x % kXcds, slot = blockIdx.x / kXcds;
  const int k_tiles = a.K * 2 / kRowBytes;
  const Share share = tile_share(a.tiles_t * a.tiles_n, per_xcd, xcd);
  Item cur, nxt{};
  if (!item_at(a, share, xcd, slot, per_xcd, k_tiles, 0, cur)) return;
  const int ldw = a.K * 2, ldx = (int)a.ldx * 2;
  set_operand_registers<kMode>(lane, wave, ldw, ldx);
  auto make_a = [&](const Item& it, bool valid) { return tile_rows(a.w, ldw, a.K * 2, it.tile_n, a.N, valid); };
  auto make_b = [&](const Item& it, bool valid) { return tile_rows(a.x, ldx, a.K * 2, it.tile_t, a.T, valid); };
  const bool single = k_tiles == 1;              // the second K tile of every tile does not exist: zeros
  int n_item = 0;
  __amdgpu_buffer_rsrc_t ra_c = make_a(cur, true), rb_c = make_b(cur, true), ra_n, rb_n;
  bool more;
  auto plan_next = [&]() {
    more = item_at(a, share, xcd, slot, per_xcd, k_tiles, ++n_item, nxt);
    ra_n = make_a(nxt, more);
    rb_n = make_b(nxt, more);
  };
  plan_next();

  const int woff = wave * 8192;
  int sa = 0, sb = 0x10000;
  {
    const __amdgpu_buffer_rsrc_t ra_2 = make_a(cur, !single), rb_2 = make_b(cur, !single);
    const int k = cur.k0 * kRowBytes;
    asm volatile(MSA_GEMM_LOAD8_B ::[dst] "s"(0x10000 + woff), [r] "s"(rb_c), [k] "s"(k) : MSA_GEMM_CLOBBERS);
    asm volatile(MSA_GEMM_LOAD8_A ::[dst] "s"(0 + woff), [r] "s"(ra_c), [k] "s"(k) : MSA_GEMM_CLOBBERS);
    asm volatile(MSA_GEMM_LOAD8_B ::[dst] "s"(0x18000 + woff), [r] "s"(rb_2), [k] "s"(k + kRowBytes) : MSA_GEMM_CLOBBERS);
    asm volatile(MSA_GEMM_LOAD8_A ::[dst] "s"(0x8000 + woff), [r] "s"(ra_2), [k] "s"(k + kRowBytes) : MSA_GEMM_CLOBBERS);
  }
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  asm volatile(MSA_GEMM_FRAGS0 ::[sa] "s"(sa), [sb] "s"(sb) : MSA_GEMM_CLOBBERS);

#define MSA_GEMM_STEP(TEXT, RA, RB, KOFF)                                                                    \
  asm volatile(TEXT : [sa] "+s"(sa), [sb] "+s"(sb)                                                           \
               : [ra] "s"(RA), [rb] "s"(RB), [k] "s"(KOFF), [woff] "s"(woff) : MSA_GEMM_CLOBBERS)
  for (;;) {
    // Step kt requests K tile kt + 2: of this item while it has one, of the next item after that (an item has two at least).
    const int k_first = cur.k0 * kRowBytes, k_end = (cur.k0 + cur.nk) * kRowBytes, k_next = nxt.k0 * kRowBytes;
    const int steps = max(cur.nk, 2);
    if (steps > 2) {
      MSA_GEMM_STEP(MSA_GEMM_KSTEP_FRESH, ra_c, rb_c, k_first + 2 * kRowBytes);
      for (int k = k_first + 3 * kRowBytes; k < k_end; k += kRowBytes) MSA_GEMM_STEP(MSA_GEMM_KSTEP, ra_c, rb_c, k);
      MSA_GEMM_STEP(MSA_GEMM_KSTEP, ra_n, rb_n, k_next);
    } else {
      MSA_GEMM_STEP(MSA_GEMM_KSTEP_FRESH, ra_n, rb_n, k_next);
    }
    if (single) {
      const __amdgpu_buffer_rsrc_t ra_2 = make_a(nxt, false), rb_2 = make_b(nxt, false);
      MSA_GEMM_STEP(MSA_GEMM_KSTEP, ra_2, rb_2, 0);
    } else {
      MSA_GEMM_STEP(MSA_GEMM_KSTEP, ra_n, rb_n, k_next + kRowBytes);
    }
    asm volatile(MSA_GEMM_SETTLE ::: "memory");

    // the finished item's accumulators, a column block (128 weight rows x 16 tokens) at a time
    const int token0 = cur.tile_t * kTile + wn * 128 + (lane & 15);
    float v[32];
#define MSA_GEMM_READ(J, H)                                                                                                        \
  asm volatile(MSA_GEMM_ACC_##J##_##H                                                                                              \
               : "=v"(v[16 * H]), "=v"(v[16 * H + 1]), "=v"(v[16 * H + 2]), "=v"(v[16 * H + 3]), "=v"(v[16 * H + 4]),               \
                 "=v"(v[16 * H + 5]), "=v"(v[16 * H + 6]), "=v"(v[16 * H + 7]), "=v"(v[16 * H + 8]), "=v"(v[16 * H + 9]),           \
                 "=v"(v[16 * H + 10]), "=v"(v[16 * H + 11]), "=v"(v[16 * H + 12]), "=v"(v[16 * H + 13]), "=v"(v[16 * H + 14]),      \
                 "=v"(v[16 * H + 15]))
    if (cur.piece < 0) {
      Finish<kMode> f(a, cur.tile_n * kTile + wm * 128, lane);
      auto table_row = [&](int j) { return kMode == kHeads ? f.table_row(token0 + 16 * j) : 0; };
      typename Finish<kMode>::Ahead ahead;
      int row = table_row(0);
#pragma unroll
      for (int m = 0; m < 4; ++m) f.request(m, token0, row, ahead);
      row = table_row(1);
#define MSA_GEMM_COLUMN(J)                                                                       \
  {                                                                                              \
    const int row2 = J < 6 ? table_row(J + 2) : 0;                                               \
    MSA_GEMM_READ(J, 0);                                                                         \
    MSA_GEMM_READ(J, 1);                                                                         \
    f.finish(token0 + 16 * J, v, ahead, J < 7, token0 + 16 * (J + 1), row);                      \
    row = row2;                                                                                  \
  }
      MSA_GEMM_COLUMN(0) MSA_GEMM_COLUMN(1) MSA_GEMM_COLUMN(2) MSA_GEMM_COLUMN(3)
      MSA_GEMM_COLUMN(4) MSA_GEMM_COLUMN(5) MSA_GEMM_COLUMN(6) MSA_GEMM_COLUMN(7)
#undef MSA_GEMM_COLUMN
    } else {
      float4* to = reinterpret_cast<float4*>(a.pieces + (int64_t)cur.piece * (kTile * kTile)) + wave * 4096 + lane;
#define MSA_GEMM_COLUMN(J)                                                                                              \
  MSA_GEMM_READ(J, 0);                                                                                                  \
  MSA_GEMM_READ(J, 1);                                                                                                  \
  _Pragma("unroll") for (int i = 0; i < 8; ++i) to[(J * 8 + i) * 64] = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
      MSA_GEMM_COLUMN(0) MSA_GEMM_COLUMN(1) MSA_GEMM_COLUMN(2) MSA_GEMM_COLUMN(3)
      MSA_GEMM_COLUMN(4) MSA_GEMM_COLUMN(5) MSA_GEMM_COLUMN(6) MSA_GEMM_COLUMN(7)
#undef MSA_GEMM_COLUMN
    }
#undef MSA_GEMM_READ
    if (!more) break;
    cur = nxt;
    ra_c = ra_n; rb_c = rb_n;
    plan_next();
  }
#undef MSA_GEMM_STEP
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#endif
}

// The same walk for ends that need nothing but the sums: a finished tile is rounded to bf16 into 128 registers while the next tile's
// first step overwrites its accumulators, and finished and stored, sixteen tokens a step, behind the MFMAs of the eight steps after that
// (gen_scan_asm.py).  A wavefront is alone on its SIMD, so whatever it does between two tiles the matrix cores wait for: storing a
// tile took it 5 us, gelu 10, against 57 us of steps at K = 2560 and 23 at K = 1024.  Whole calls, us, ends in registers and here: 32771 x
// 2560 x 19456 stored 2392 and 2238, 6001 x 2560 x 19456 with the gated unit 434 and 415, 8192 x 1024 x 4096 with gelu 88 and 60, and
// with silu-mul 2257 and 2221 (the encoding block around it 12.00 and 11.90 ms: its half output leaves less to hide).
constexpr int kFlowVgprs = 24;                 // the compiler's share of the vector registers
constexpr int kFlowSteps = 11;                 // an item of that many steps takes another tile's end: one packs, eight finish, the
                                               // last two already load for the item behind
[[maybe_unused]] constexpr int kFar = 0x7ff00000;               // behind every extent, whatever is added: nothing is stored

template <int kMode, bool kStream>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_num_vgpr(kFlowVgprs))) void tile_flow_kernel(TileArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int per_xcd = gridDim.x / kXcds, xcd = blockIdx.x % kXcds, slot = blockIdx.x / kXcds;
  const int k_tiles = a.K * 2 / kRowBytes;
  const Share share = tile_share(a.tiles_t * a.tiles_n, per_xcd, xcd);
  Item cur, nxt{};
  if (!item_at(a, share, xcd, slot, per_xcd, k_tiles, 0, cur)) return;
  const int ldw = a.K * 2, ldx = (int)a.ldx * 2;
  set_operand_registers<kMode>(lane, wave, ldw, ldx);
  if constexpr (kMode == kGelu) asm volatile(MSA_GEMM_SET_GELU ::: MSA_GEMM_FLOW_CLOBBERS);
  auto make_a = [&](const Item& it, bool valid) { return tile_rows(a.w, ldw, a.K * 2, it.tile_n, a.N, valid); };
  auto make_b = [&](const Item& it, bool valid) { return tile_rows(a.x, ldx, a.K * 2, it.tile_t, a.T, valid); };
  // the output behind a tile's first token and column
  constexpr int kCols = is_pair(kMode) ? kTile / 2 : kTile;
  const int width = is_pair(kMode) ? a.N / 2 : a.N, ldo = (int)a.ldo * 2;
  auto make_out = [&](const Item& it) {
    const int rows = min(kTile, a.T - it.tile_t * kTile), at = it.tile_n * kCols;
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<char*>(a.out) + (int64_t)it.tile_t * kTile * ldo + at * 2, 0,
                                             (rows - 1) * ldo + (width - at) * 2, 0x00020000);
  };
  // a lane's offsets in it: the columns of its group, tokens of the first eight of a column block in the lower lanes
  int so0, so1;
  auto set_offsets = [&](const Item& it) {
    const bool low = (lane & 8) == 0;
    const int col = wm * (kCols / 2) + 8 * (lane >> 4) + (low ? 0 : 32), at = it.tile_n * kCols + col;
    const int row = (wn * 128 + (lane & 7)) * ldo + col * 2;
    so0 = at < width ? row : kFar;
    so1 = at + 64 < width ? row + 128 : kFar;
  };

  int n_item = 0;
  __amdgpu_buffer_rsrc_t ra_c = make_a(cur, true), rb_c = make_b(cur, true), ra_n, rb_n, ro = make_out(cur);
  bool more;
  auto plan_next = [&]() {
    more = item_at(a, share, xcd, slot, per_xcd, k_tiles, ++n_item, nxt);
    ra_n = make_a(nxt, more);
    rb_n = make_b(nxt, more);
  };
  plan_next();
  const int woff = wave * 8192, row8 = 8 * ldo, row16 = 16 * ldo;
  int sa = 0, sb = 0x10000;
  {
    const int k = cur.k0 * kRowBytes;
    asm volatile(MSA_GEMM_LOAD8_B ::[dst] "s"(0x10000 + woff), [r] "s"(rb_c), [k] "s"(k) : MSA_GEMM_FLOW_CLOBBERS);
    asm volatile(MSA_GEMM_LOAD8_A ::[dst] "s"(0 + woff), [r] "s"(ra_c), [k] "s"(k) : MSA_GEMM_FLOW_CLOBBERS);
    asm volatile(MSA_GEMM_LOAD8_B ::[dst] "s"(0x18000 + woff), [r] "s"(rb_c), [k] "s"(k + kRowBytes) : MSA_GEMM_FLOW_CLOBBERS);
    asm volatile(MSA_GEMM_LOAD8_A ::[dst] "s"(0x8000 + woff), [r] "s"(ra_c), [k] "s"(k + kRowBytes) : MSA_GEMM_FLOW_CLOBBERS);
  }
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  asm volatile(MSA_GEMM_FRAGS0 ::[sa] "s"(sa), [sb] "s"(sb) : MSA_GEMM_FLOW_CLOBBERS);

#define MSA_GEMM_STEP(TEXT, RA, RB, KOFF)                                                                    \
  asm volatile(TEXT : [sa] "+s"(sa), [sb] "+s"(sb)                                                           \
               : [ra] "s"(RA), [rb] "s"(RB), [k] "s"(KOFF), [woff] "s"(woff) : MSA_GEMM_FLOW_CLOBBERS)
#define MSA_GEMM_ENDS                                                                                         \
  [ro] "s"(ro), [row8] "s"(row8), [row16] "s"(row16), [so0] "v"(so0), [so1] "v"(so1), [limit] "s"(a.end.limit), [rate] "s"(a.rate), \
      [shift] "s"(a.end.shift)
#define MSA_GEMM_KSTEP_END(END, J, KOFF)                                                                     \
  if constexpr (kStream)                                                                                     \
    asm volatile(MSA_GEMM_KSTEP_##END##_##J(" nt") : [sa] "+s"(sa), [sb] "+s"(sb)                             \
                 : [ra] "s"(ra_c), [rb] "s"(rb_c), [k] "s"(KOFF), [woff] "s"(woff), MSA_GEMM_ENDS : MSA_GEMM_FLOW_CLOBBERS); \
  else                                                                                                       \
    asm volatile(MSA_GEMM_KSTEP_##END##_##J("") : [sa] "+s"(sa), [sb] "+s"(sb)                                \
                 : [ra] "s"(ra_c), [rb] "s"(rb_c), [k] "s"(KOFF), [woff] "s"(woff), MSA_GEMM_ENDS : MSA_GEMM_FLOW_CLOBBERS);
#define MSA_GEMM_END(END, J)                                                                                 \
  if constexpr (kStream) asm volatile(MSA_GEMM_END_##END##_##J(" nt") ::MSA_GEMM_ENDS : MSA_GEMM_FLOW_CLOBBERS); \
  else asm volatile(MSA_GEMM_END_##END##_##J("") ::MSA_GEMM_ENDS : MSA_GEMM_FLOW_CLOBBERS);
#define MSA_GEMM_EIGHT(DO, END, ...)                                                                         \
  DO(END, 0 __VA_OPT__(, __VA_ARGS__ + 0 * kRowBytes)) DO(END, 1 __VA_OPT__(, __VA_ARGS__ + 1 * kRowBytes))  \
  DO(END, 2 __VA_OPT__(, __VA_ARGS__ + 2 * kRowBytes)) DO(END, 3 __VA_OPT__(, __VA_ARGS__ + 3 * kRowBytes))  \
  DO(END, 4 __VA_OPT__(, __VA_ARGS__ + 4 * kRowBytes)) DO(END, 5 __VA_OPT__(, __VA_ARGS__ + 5 * kRowBytes))  \
  DO(END, 6 __VA_OPT__(, __VA_ARGS__ + 6 * kRowBytes)) DO(END, 7 __VA_OPT__(, __VA_ARGS__ + 7 * kRowBytes))
#define MSA_GEMM_BY_MODE(DO, ...)                                                                            \
  if constexpr (kMode == kStore) { MSA_GEMM_EIGHT(DO, STORE __VA_OPT__(, __VA_ARGS__)) }                     \
  else if constexpr (kMode == kSiluMul) { MSA_GEMM_EIGHT(DO, SILU __VA_OPT__(, __VA_ARGS__)) }               \
  else if constexpr (kMode == kGlu) { MSA_GEMM_EIGHT(DO, GLU __VA_OPT__(, __VA_ARGS__)) }                    \
  else { MSA_GEMM_EIGHT(DO, GELU __VA_OPT__(, __VA_ARGS__)) }
  // (gelu's columns end at a multiple of a wavefront's rows: a tile's part of the wavefront is through gelu or is not)
  bool held = false, plain = false;              // a finished tile waits for its end (ro, so0, so1 are its); without gelu
  for (;;) {
    const int k_first = cur.k0 * kRowBytes, k_end = (cur.k0 + cur.nk) * kRowBytes, k_next = nxt.k0 * kRowBytes;
    int k = k_first + 3 * kRowBytes;             // what the next step requests
    if (held) {                                  // (cur.nk >= kFlowSteps)
      MSA_GEMM_STEP(MSA_GEMM_KSTEP_FRESH_PACK, ra_c, rb_c, k_first + 2 * kRowBytes);
      if (kMode == kGelu && plain) { MSA_GEMM_EIGHT(MSA_GEMM_KSTEP_END, STORE, k) }
      else { MSA_GEMM_BY_MODE(MSA_GEMM_KSTEP_END, k) }
      k += 8 * kRowBytes;
    } else if (cur.nk > 2) {
      MSA_GEMM_STEP(MSA_GEMM_KSTEP_FRESH, ra_c, rb_c, k_first + 2 * kRowBytes);
    } else {
      MSA_GEMM_STEP(MSA_GEMM_KSTEP_FRESH, ra_n, rb_n, k_next);
    }
    for (; k < k_end; k += kRowBytes) MSA_GEMM_STEP(MSA_GEMM_KSTEP, ra_c, rb_c, k);
    if (cur.nk > 2) MSA_GEMM_STEP(MSA_GEMM_KSTEP, ra_n, rb_n, k_next);
    MSA_GEMM_STEP(MSA_GEMM_KSTEP, ra_n, rb_n, k_next + kRowBytes);
    held = cur.piece < 0 && more && nxt.nk >= kFlowSteps;
    if (cur.piece >= 0) {
      const int sp = __builtin_amdgcn_readfirstlane(wave * (kPieceBytes / 4));
      const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc(
          reinterpret_cast<char*>(a.pieces) + (int64_t)cur.piece * kPieceBytes, 0, kPieceBytes, 0x00020000);
      asm volatile(MSA_GEMM_PIECE ::[rp] "s"(to), [vp] "v"(lane * 16), [sp] "s"(sp) : MSA_GEMM_FLOW_CLOBBERS);
    } else {
      ro = make_out(cur);
      set_offsets(cur);
      plain = kMode == kGelu && cur.tile_n * kTile + wm * 128 >= a.end.gelu_n;
      if (!held) {
        asm volatile(MSA_GEMM_PACK ::: MSA_GEMM_FLOW_CLOBBERS);
        if (kMode == kGelu && plain) { MSA_GEMM_EIGHT(MSA_GEMM_END, STORE) }
        else { MSA_GEMM_BY_MODE(MSA_GEMM_END) }
      }
    }
    if (!more) break;
    cur = nxt;
    ra_c = ra_n; rb_c = rb_n;
    plan_next();
  }
#undef MSA_GEMM_STEP
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#endif
}

// The tiles that were multiplied in pieces: a workgroup adds up a column block's pieces, in their order, for the four wavefronts that
// would have finished it.
template <int kMode, bool kRounded>
__global__ __launch_bounds__(kThreads) void tile_finish_kernel(TileArgs a, int per_xcd) {
  const int j = blockIdx.x & 7, xcd = (blockIdx.x >> 3) / a.max_rem, u = (blockIdx.x >> 3) % a.max_rem;
  const Share share = tile_share(a.tiles_t * a.tiles_n, per_xcd, xcd);
  if (u >= share.rem) return;
  int tile_t, tile_n;
  tile_at(a, share.first + share.rounds * per_xcd + u, tile_t, tile_n);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave >> 1, wn = wave & 1;
  const int token = tile_t * kTile + wn * 128 + 16 * j + (lane & 15);
  Finish<kMode, kRounded> f(a, tile_n * kTile + wm * 128, lane);
  typename Finish<kMode, kRounded>::Ahead ahead;
#pragma unroll
  for (int m = 0; m < 4; ++m) f.request(m, token, kMode == kHeads ? f.table_row(token) : 0, ahead);
  const float4* from = reinterpret_cast<const float4*>(a.pieces + (int64_t)(blockIdx.x >> 3) * a.split * (kTile * kTile)) + wave * 4096 + j * 512 + lane;
  float v[32] = {};
  for (int p = 0; p < a.split; ++p) {
    float4 part[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) part[i] = from[(int64_t)p * (kTile * kTile / 4) + i * 64];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[4 * i] += part[i].x; v[4 * i + 1] += part[i].y; v[4 * i + 2] += part[i].z; v[4 * i + 3] += part[i].w;
    }
  }
  f.finish(token, v, ahead, false, 0, 0);
}

struct Plan {
  int tiles_t, tiles_n, group, grid, split, max_rem;
  size_t bytes;             // of pieces
};

// How many pieces the tiles of the incomplete round are cut into.  A K tile takes a compute unit about 1.45 us; a piece is written and
// read again, 0.5 MB at about 4 TB/s for all of them, behind a launch of about 5 us.
Plan make_plan(int64_t T, int K, int N, bool may_split) {
  Plan p{};
  p.tiles_t = (int)((T + kTile - 1) / kTile);
  p.tiles_n = (N + kTile - 1) / kTile;
  p.group = std::min(4, p.tiles_t);
  p.grid = std::max(kXcds * 2, device_compute_units() / kXcds * kXcds);
  p.split = 1;
  const int per_xcd = p.grid / kXcds, k_tiles = std::max(2, K / 64);
  int rem = 0, tiles_of = 0;
  for (int x = 0; x < kXcds; ++x) {
    const int r = tile_share(p.tiles_t * p.tiles_n, per_xcd, x).rem;
    rem = std::max(rem, r);
    tiles_of += r;
  }
  p.max_rem = rem;
  if (!may_split || rem == 0) return p;
  double best = k_tiles * 1.45;
  for (int s = 2; s <= 16 && k_tiles / s >= 4 && rem * s <= 2 * per_xcd; ++s) {
    const double us = (double)((rem * s + per_xcd - 1) / per_xcd) * ((k_tiles + s - 1) / s) * 1.45 + tiles_of * s * (2.0 * kPieceBytes) / 4e6 + 5;
    if (us < best) { best = us; p.split = s; }
  }
  if (p.split > 1) p.bytes = (size_t)kXcds * rem * p.split * kPieceBytes;
  return p;
}

template <void (*kern)(TileArgs)>
int launch_tile_kernel(const TileArgs& a, const Plan& p, hipStream_t st) {
  static std::atomic<int> lds_limit_raised{0}, resources_checked{0};
  if (const int rc = check_asm_kernel_resources(resources_checked, reinterpret_cast<const void*>(kern), "tile kernel", nullptr, nullptr)) return rc;
  MSA_HIP(raise_dynamic_lds_limit(lds_limit_raised, reinterpret_cast<const void*>(kern), kLdsBytes));
  kern<<<p.grid, kThreads, kLdsBytes, st>>>(a);
  MSA_LAUNCH_CHECK();
  return MSA_OK;
}

template <int kMode, bool kRounded>
int launch_finish(const TileArgs& a, const Plan& p, hipStream_t st) {
  tile_finish_kernel<kMode, kRounded><<<kXcds * p.max_rem * 8, kThreads, 0, st>>>(a, p.grid / kXcds);
  MSA_LAUNCH_CHECK();
  return MSA_OK;
}

// An end under the next tile's steps wants tiles of kFlowSteps steps, and gelu's line between two wavefronts' rows.
bool flows(const TileArgs& a, int mode) {
  return mode != kAdd && mode != kHeads && a.K >= 64 * kFlowSteps && a.ldo < ((int64_t)1 << 21) && (mode != kGelu || a.end.gelu_n % 128 == 0);
}

// The columns that fill whole rounds, where the others are better off in block_gemm.hip's smaller tiles (N: none).  A few tiles behind the
// last whole round take a launch most of another one, whole or in pieces: `last`, fitted to 16 to 128 such tiles, 1024 and 2560 deep (less: not measured;
// more: level, 8192 x 3072 x 6176 233 and 234, x 4096 x 6176 301 and 302, 6001 x 9728 x 4608 384 and 380).  us,
// rows x K x N, all tiles and split: 8192 x 1024 x 6176 (32 columns' tiles a fourth round) 98 and 87, x 2304 52 and 42, 6001 x 1024 x 3072 50
// and 43, 8192 x 2560 x 4608 165 and 153, x 12368 442 and 431; level or behind, and not split: 8192 x 1024 x 3072 54 and 58, 6001 x 1024 x
// 6176 74 and 76, x 2560 x 8480 204 and 205, 1700 x 2560 x 19456 glu 143 and 147.  The ends round their sums alike in both kernels where the tiles' end flows.
int whole_columns(const TileArgs& a, int mode) {
  if ((mode != kStore && mode != kGelu && mode != kGlu) || (mode != kStore && !flows(a, mode)) || a.K < 1024 || a.K > 2560) return a.N;
  const int tiles_t = (a.T + kTile - 1) / kTile, tiles_n = (a.N + kTile - 1) / kTile;
  const int units = std::max(kXcds * 2, device_compute_units() / kXcds * kXcds), rounds = (int)((int64_t)tiles_t * tiles_n / units);
  const int columns = (int)((int64_t)rounds * units / tiles_t), behind = (int)((int64_t)tiles_t * tiles_n - (int64_t)rounds * units);
  if (behind == 0 || columns < 1 || columns >= tiles_n) return a.N;
  const float last = std::min(1.2f * (float)(a.K / 64), 6.f + 0.45f * (float)behind);
  return 1.35f * msa_block_linear_us(a.T, a.K, a.N - columns * kTile) < last ? columns * kTile : a.N;
}

template <int kMode>
int launch_tiles(TileArgs a, const Plan& p, hipStream_t st) {
  // Half of the memory-side cache: an output within it is still there for its reader (a 32771-token encoding block through two layers
  // takes 11.98 ms with all outputs non-temporal, 11.89 with none, 11.87 with the large ones).
  a.stream = (int64_t)a.T * a.N * (is_pair(kMode) ? 1 : 2) > (int64_t)128 << 20;
  a.tiles_t = p.tiles_t; a.tiles_n = p.tiles_n; a.group = p.group; a.split = p.split; a.max_rem = p.max_rem;
  if constexpr (kMode != kAdd && kMode != kHeads) {
    if (flows(a, kMode)) {
      a.rate = -1.4426950408889634f * a.end.alpha;
      const int rc = a.stream ? launch_tile_kernel<tile_flow_kernel<kMode, true>>(a, p, st) : launch_tile_kernel<tile_flow_kernel<kMode, false>>(a, p, st);
      return rc != MSA_OK || p.split == 1 ? rc : launch_finish<kMode, kMode != kStore>(a, p, st);
    }
  }
  const int rc = launch_tile_kernel<tile_gemm_kernel<kMode>>(a, p, st);
  return rc != MSA_OK || p.split == 1 ? rc : launch_finish<kMode, false>(a, p, st);
}

int check_operands(const char* name, const void* x, int64_t T, int64_t ldx, const void* w, int32_t K, int64_t N) {
  MSA_REQUIRE(T > 0 && T < ((int64_t)1 << 22), "%s: T=%lld out of range", name, (long long)T);
  MSA_REQUIRE(K >= 64 && K % 64 == 0 && K <= 32768, "%s: K=%d (a multiple of 64 up to 32768)", name, K);
  MSA_REQUIRE(ldx >= K && ldx % 8 == 0 && ldx < ((int64_t)1 << 21), "%s: row stride %lld", name, (long long)ldx);
  MSA_REQUIRE(N > 0 && N < ((int64_t)1 << 20), "%s: N=%lld out of range", name, (long long)N);
  MSA_REQUIRE((((uintptr_t)x | (uintptr_t)w) & 15) == 0, "%s: x / w must be 16-byte aligned", name);
  return MSA_OK;
}

}  // namespace

extern "C" size_t msa_tile_workspace_bytes(int64_t T, int32_t K, int32_t N) {
  if (T <= 0 || K < 64 || N <= 0 || T >= ((int64_t)1 << 22) || N >= (1 << 20)) return 0;
  return make_plan(T, K, N, true).bytes;
}

extern "C" int msa_tile_linear(const void* x, int64_t ldx, int64_t T, int32_t K, const void* w, int32_t N, const msa_tile_end* end, void* out,
                               int64_t ldo, void* ws, size_t ws_bytes, void* stream) {
  MSA_REQUIRE(x && w && out && end, "msa_tile_linear: null pointer");
  if (const int rc = check_operands("msa_tile_linear", x, T, ldx, w, K, N)) return rc;
  const int mode = end->mode;
  MSA_REQUIRE(mode == kStore || mode == kAdd || mode == kGelu || is_pair(mode), "msa_tile_linear: mode %d", mode);
  MSA_REQUIRE(N % (is_pair(mode) ? 16 : 8) == 0, "msa_tile_linear: N=%d", N);
  MSA_REQUIRE(mode != kGelu || (end->gelu_n >= 0 && end->gelu_n <= N && end->gelu_n % 8 == 0), "msa_tile_linear: gelu_n=%d", end->gelu_n);
  MSA_REQUIRE(ldo >= (is_pair(mode) ? N / 2 : N) && ldo % 8 == 0 && ((uintptr_t)out & 15) == 0,
              "msa_tile_linear: out must be 16-byte aligned, its row stride (%lld) a multiple of 8", (long long)ldo);
  TileArgs a{};
  a.x = static_cast<const bf16_t*>(x); a.w = static_cast<const bf16_t*>(w); a.out = static_cast<bf16_t*>(out);
  a.ldx = ldx; a.ldo = ldo; a.T = (int32_t)T; a.K = K; a.N = N; a.end = *end;
  if (const int n = whole_columns(a, mode); n < N) {
    a.N = n;
    msa_tile_end rest = *end;
    rest.gelu_n = std::max(0, end->gelu_n - n);
    a.end.gelu_n = std::min(end->gelu_n, n);
    if (const int rc = msa_block_linear(x, ldx, T, K, a.w + (int64_t)n * K, N - n, &rest, a.out + (mode == kGlu ? n / 2 : n), ldo, stream)) return rc;
  }
  Plan p = make_plan(T, K, a.N, ws != nullptr);
  if (p.bytes > ws_bytes || ((uintptr_t)ws & 15)) p = make_plan(T, K, a.N, false);
  a.pieces = static_cast<float*>(ws);
  switch (mode) {
    case kStore: return launch_tiles<kStore>(a, p, as_stream(stream));
    case kAdd: return launch_tiles<kAdd>(a, p, as_stream(stream));
    case kGelu: return launch_tiles<kGelu>(a, p, as_stream(stream));
    case kGlu: return launch_tiles<kGlu>(a, p, as_stream(stream));
    default: return launch_tiles<kSiluMul>(a, p, as_stream(stream));
  }
}

extern "C" int msa_qkv_proj_ws(const void* x, int64_t T, int32_t K, const void* w, int32_t Hq, int32_t Hkv, int32_t Hr_front,
                               int32_t Hr_back, const int64_t* positions, const void* q_norm_w, const void* k_norm_w,
                               float eps, const float* rope_cos, const float* rope_sin, int32_t rope_rows, void* q_out,
                               void* k_out, void* v_out, void* r_out, void* ws, size_t ws_bytes, void* stream) {
  MSA_REQUIRE(x && w && positions && q_norm_w && k_norm_w && rope_cos && rope_sin && q_out && k_out && v_out,
              "msa_qkv_proj: null pointer");
  MSA_REQUIRE(Hq > 0 && Hkv > 0 && Hr_front >= 0 && Hr_back >= 0, "msa_qkv_proj: bad head counts");
  const int64_t heads = (int64_t)Hq + 2 * (int64_t)Hkv + Hr_front + Hr_back;
  if (const int rc = check_operands("msa_qkv_proj", x, T, K, w, K, heads * kHeadDim)) return rc;
  MSA_REQUIRE((Hr_front + Hr_back == 0) || r_out != nullptr, "msa_qkv_proj: router heads without an output");
  MSA_REQUIRE(rope_rows > 0 && eps > 0.f, "msa_qkv_proj: rope_rows / eps");
  MSA_REQUIRE((((uintptr_t)q_norm_w | (uintptr_t)k_norm_w) & 15) == 0,
              "msa_qkv_proj: q_norm_w / k_norm_w (128 bf16 each) must be 16-byte aligned");
  MSA_REQUIRE((((uintptr_t)rope_cos | (uintptr_t)rope_sin) & 3) == 0 &&
                  (((uintptr_t)q_out | (uintptr_t)k_out | (uintptr_t)v_out | (uintptr_t)r_out) & 15) == 0,
              "msa_qkv_proj: rope tables (fp32 [rope_rows, 64]) 4-byte and outputs 16-byte aligned");
  TileArgs a{};
  a.x = static_cast<const bf16_t*>(x); a.w = static_cast<const bf16_t*>(w); a.pos = positions;
  a.q_norm_w = static_cast<const bf16_t*>(q_norm_w); a.k_norm_w = static_cast<const bf16_t*>(k_norm_w);
  a.rope_cos = rope_cos; a.rope_sin = rope_sin;
  a.q_out = static_cast<bf16_t*>(q_out); a.k_out = static_cast<bf16_t*>(k_out); a.v_out = static_cast<bf16_t*>(v_out);
  a.r_out = static_cast<bf16_t*>(r_out);
  a.T = (int32_t)T; a.K = K; a.N = (int32_t)(heads * kHeadDim); a.ldx = K;
  a.Hq = Hq; a.Hkv = Hkv; a.Hr_front = Hr_front; a.Hr_back = Hr_back; a.rope_rows = rope_rows; a.eps = eps;
  Plan p = make_plan(T, K, a.N, ws != nullptr);
  if (p.bytes > ws_bytes || ((uintptr_t)ws & 15)) p = make_plan(T, K, a.N, false);
  a.pieces = static_cast<float*>(ws);
  return launch_tiles<kHeads>(a, p, as_stream(stream));
}

extern "C" int msa_qkv_proj(const void* x, int64_t T, int32_t K, const void* w, int32_t Hq, int32_t Hkv, int32_t Hr_front,
                            int32_t Hr_back, const int64_t* positions, const void* q_norm_w, const void* k_norm_w,
                            float eps, const float* rope_cos, const float* rope_sin, int32_t rope_rows, void* q_out,
                            void* k_out, void* v_out, void* r_out, void* stream) {
  return msa_qkv_proj_ws(x, T, K, w, Hq, Hkv, Hr_front, Hr_back, positions, q_norm_w, k_norm_w, eps, rope_cos, rope_sin, rope_rows,
                         q_out, k_out, v_out, r_out, nullptr, 0, stream);
}
