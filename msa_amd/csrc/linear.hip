// Weight-streaming linear layer for a handful of rows (the decode step of the host model):
//   y[M, N] = x[M, K] . w[N, K]^T   (+ residual, or silu(gate) * up over interleaved row groups)
// with M <= 16.  The weight matrix is read from HBM exactly once, which is the whole cost: per
// decode step of a 36-layer model the projections stream ~8 GB.  The 16 rows of x are exactly one
// 16x16x32 MFMA operand, so a wavefront multiplies 16 weight rows (one row group) at a time:
//   lane (n = lane % 16, g = lane / 16), vector j = 0..J-1, loads the 16 bytes of weight row n at
//   k = unit * 32 J + 32 j + 8 g   (one load instruction covers 64 contiguous bytes of each of 16 rows),
// and the same bytes of x row n (J = 4, or 2 when the RMSNorm is folded in).  The contraction order
// inside a unit is permuted the same way on both operands, which a dot product does not see.  A workgroup owns R row groups and splits
// K over its wavefronts; partial sums meet in LDS and are added in wavefront order (deterministic).  Matrices of more than
// some 10 MB take the form of rows_ring.h instead (takes_ring).
#include <algorithm>

#include "rows_ring.h"

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4_t;
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kUnit = 128;           // K must be a multiple of this; a wavefront steps through K in units of 32 J
constexpr int kMaxWaves = 16;

enum { kEpiPlain = 0, kEpiResidual = 1, kEpiSiluMul = 2 };

// two floats -> packed bf16 pair, round to nearest even in hardware (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t pack_rne(float lo, float hi) {
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  union { bf16x2_t b; uint32_t u; } c;
  c.b = __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t);
  return c.u;
}

__device__ __forceinline__ bf16x8_t as_frag(u32x4_t v) {
  union { u32x4_t u; bf16x8_t b; } c;
  c.u = v;
  return c.b;
}

template <int R, int kEpi, bool kNorm, int J>
__global__ __launch_bounds__(kMaxWaves * 64) void skinny_linear_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const bf16_t* __restrict__ residual,
    const bf16_t* __restrict__ norm_w, float eps, bf16_t* __restrict__ y, int32_t M, int32_t N, int32_t K,
    int64_t y_row_stride, int32_t rows_per_wg) {
  constexpr int kUnitBytes = 64 * J;   // one unit = J vectors of 16 bytes per lane = 32 J elements of a row
  const int units = K / (32 * J);
  extern __shared__ __align__(16) float part[];   // [waves][R][64][4], then [waves][16] row sums of squares
  const int tid = threadIdx.x, lane = tid & 63, waves = blockDim.x >> 6;
  // the wavefront index as a scalar: every K offset below derives from it and rides in the scalar offset of the
  // buffer loads, which must be provably uniform (a value the compiler takes for divergent costs a
  // read-first-lane loop around every load)
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_l = lane & 15, g = lane >> 4;
  // a workgroup owns rows [n_base, n_base + rows_per_wg) of w, rows_per_wg <= 16 R (fewer than 16 R when the matrix
  // has too few rows to give every compute unit a full set: the rows past it read as zero and are not stored)
  const int n_base = blockIdx.x * rows_per_wg;
  const int64_t row_bytes = (int64_t)K * 2;

  // rows past N (weights) and past M (activations) read as zero through the buffer bounds
  const int rows_w = min(rows_per_wg, N - n_base);
  const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(reinterpret_cast<const char*>(w)) + (int64_t)n_base * row_bytes, 0, (int)(rows_w * row_bytes),
      0x00020000);
  const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(reinterpret_cast<const char*>(x)), 0, (int)(M * row_bytes), 0x00020000);
  const int voff = n_l * (int)row_bytes + g * 16;

  // this wavefront's share of the K units
  const int u0 = (int)((uint32_t)units * (uint32_t)wave / (uint32_t)waves);        // units * waves < 2^31: K is bounded by the host
  const int u1 = (int)((uint32_t)units * (uint32_t)(wave + 1) / (uint32_t)waves);

  floatx4_t acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = floatx4_t{0.f, 0.f, 0.f, 0.f};

  const __amdgpu_buffer_rsrc_t rs_g = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(reinterpret_cast<const char*>(kNorm ? norm_w : x)), 0, (int)row_bytes, 0x00020000);
  float ssq = 0.f;                      // this lane's share of sum(x^2) of row n_l
  u32x4_t fw[2][R][J];
  auto load_w = [&](int slot, int u) {
    const int k_off = u * kUnitBytes;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int j = 0; j < J; ++j)
        fw[slot][r][j] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, voff + r * 16 * (int)row_bytes, k_off + j * 64, 0);
  };

  {
    u32x4_t fx[2][J];
    u32x4_t fg[kNorm ? 2 : 1][J];     // norm weights of the unit (every row group shares them; they hit L1 / L2)
    auto load_unit = [&](int slot, int u) {
      const int k_off = u * kUnitBytes;
#pragma unroll
      for (int j = 0; j < J; ++j) fx[slot][j] = __builtin_amdgcn_raw_buffer_load_b128(rs_x, voff, k_off + j * 64, 0);
      if constexpr (kNorm) {
#pragma unroll
        for (int j = 0; j < J; ++j) fg[slot][j] = __builtin_amdgcn_raw_buffer_load_b128(rs_g, g * 16, k_off + j * 64, 0);
      }
      load_w(slot, u);
    };
    auto mul_unit = [&](int slot) {
      if constexpr (kNorm) {
        // RMSNorm folded in: the operand is bf16(x * norm_w); the row scale rsqrt(mean(x^2) + eps) commutes
        // with the product and is applied to the fp32 sums in the epilogue, so nothing here waits for it.
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const float lo = bf16lo(fx[slot][j][c]), hi = bf16hi(fx[slot][j][c]);
            ssq += lo * lo + hi * hi;
            fx[slot][j][c] = pack_rne(lo * bf16lo(fg[slot][j][c]), hi * bf16hi(fg[slot][j][c]));
          }
      }
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int r = 0; r < R; ++r)
          acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(fx[slot][j]), as_frag(fw[slot][r][j]), acc[r], 0, 0, 0);
    };
    // two register stages, one unit each: the loads of unit u+1 are in flight under the MFMAs of u
    if (u0 < u1) load_unit(0, u0);
    int u = u0;
    for (; u + 2 <= u1; u += 2) {
      load_unit(1, u + 1);
      mul_unit(0);
      if (u + 2 < u1) load_unit(0, u + 2);
      mul_unit(1);
    }
    if (u < u1) mul_unit(0);
  }

  // partial sums -> LDS; acc[r][e] is y[m = 4 g + e][n_base + 16 r + n_l]
#pragma unroll
  for (int r = 0; r < R; ++r) *reinterpret_cast<floatx4_t*>(&part[((wave * R + r) * 64 + lane) * 4]) = acc[r];
  float* row_ssq = part + waves * R * 256;
  if constexpr (kNorm) {
    ssq += __shfl_xor(ssq, 16);
    ssq += __shfl_xor(ssq, 32);
    if (g == 0) row_ssq[wave * 16 + n_l] = ssq;
  }
  __syncthreads();
  floatx4_t inv = floatx4_t{1.f, 1.f, 1.f, 1.f};   // row scales of this lane's four output rows
  if constexpr (kNorm) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float tot = 0.f;
      for (int wv = 0; wv < waves; ++wv) tot += row_ssq[wv * 16 + 4 * g + e];
      inv[e] = rsqrtf(tot / (float)K + eps);
    }
  }
  if (kEpi == kEpiSiluMul) {
    // every 16-row group holds gate rows [8 i, 8 i + 8) in its first half and the same up rows in its second: a
    // lane with n_l < 8 has the gate sum and takes the up sum from the lane 8 further on
    for (int r = wave; r < R; r += waves) {
      floatx4_t sum = floatx4_t{0.f, 0.f, 0.f, 0.f};
      for (int wv = 0; wv < waves; ++wv) sum += *reinterpret_cast<const floatx4_t*>(&part[((wv * R + r) * 64 + lane) * 4]);
      floatx4_t up;
#pragma unroll
      for (int e = 0; e < 4; ++e) up[e] = __shfl_xor(sum[e], 8);
      const int n = ((n_base + 16 * r) >> 1) + n_l;    // output column: a group of 16 rows folds into 8 outputs
      if (n_l >= 8 || n_base + 16 * r + 8 + n_l >= N) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = 4 * g + e;
        if (m >= M) continue;
        const float a = bf16_to_f32(f32_to_bf16(sum[e] * inv[e])), b = bf16_to_f32(f32_to_bf16(up[e] * inv[e]));
        y[(int64_t)m * y_row_stride + n] = f32_to_bf16(a / (1.f + __expf(-a)) * b);
      }
    }
    return;
  }
  for (int r = wave; r < R; r += waves) {
    floatx4_t sum = floatx4_t{0.f, 0.f, 0.f, 0.f};
    for (int wv = 0; wv < waves; ++wv) sum += *reinterpret_cast<const floatx4_t*>(&part[((wv * R + r) * 64 + lane) * 4]);
    const int n = n_base + 16 * r + n_l;
    if (n >= N || 16 * r + n_l >= rows_per_wg) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = 4 * g + e;
      if (m >= M) continue;
      float v = sum[e] * inv[e];
      if (kEpi == kEpiResidual) v = bf16_to_f32(f32_to_bf16(v)) + bf16_to_f32(residual[(int64_t)m * y_row_stride + n]);
      y[(int64_t)m * y_row_stride + n] = f32_to_bf16(v);
    }
  }
}

// The line to the form of rows_ring.h (us here and there, one / sixteen rows): 3072 x 1280 3.7 / 4.6 and 4.5 / 5.1, 6144 x 1280 5.5 / 6.1
// and 5.8 / 6.3, 4096 x 1024 3.6 / 4.3 and 3.9 / 4.3; 2560 x 2560 5.1 / 7.2 and 5.3 / 6.4, 2560 x 2048 4.7 / 5.9 and 4.5 / 5.4,
// 9728 x 1024 7.4 / 8.4 and 6.3 / 6.7.  Longer rows than kMaxResidentK have no line of their own: with sixteen
// rows, plain and ring, 6144 x 9728 32.3 and 27.4, 7168 x 5632 22.6 and 19.4, 6400 x 8192 30.4 and 23.5, 8176 x 9728 37.6 and 31.8.
constexpr int64_t kRingWeights = 5 << 20;
bool takes_ring(int32_t N, int32_t K, bool norm) {
  return K > rows_ring::kMinK && rows_ring::busy_weights(N, K) >= kRingWeights && (!norm || K <= rows_ring::kMaxResidentK);
}

// What rows_ring.h's kernel does with a product.
template <int kEpi>
struct RingEnd {
  struct Args {
    const bf16_t* residual;
    bf16_t* y;
    int64_t y_row_stride;
  };
  bf16_t add;
  __device__ __forceinline__ void begin(const Args&, int) {}
  __device__ __forceinline__ void load(const Args& a, int m, int n, bool mine, bool, int) {
    if (kEpi == kEpiResidual && mine) add = a.residual[(int64_t)m * a.y_row_stride + n];
  }
  __device__ __forceinline__ void apply(const Args& a, int m, int n, float v, bool mine, bool, int) const {
    if constexpr (kEpi == kEpiSiluMul) {
      // a 16-row group holds gate rows in its first half and the same up rows in its second, 32 lanes on
      const float gate = bf16_to_f32(f32_to_bf16(v)), up = bf16_to_f32(f32_to_bf16(__shfl_xor(v, 32)));
      if (mine && (n & 8) == 0) a.y[(int64_t)m * a.y_row_stride + (n >> 4) * 8 + (n & 7)] = f32_to_bf16(gate / (1.f + __expf(-gate)) * up);
    } else if (mine) {
      if (kEpi == kEpiResidual) v = bf16_to_f32(f32_to_bf16(v)) + bf16_to_f32(add);
      a.y[(int64_t)m * a.y_row_stride + n] = f32_to_bf16(v);
    }
  }
};

template <int kEpi>
int launch_ring(const void* x, const void* w, const void* residual, const void* norm_w, float eps, void* y, int32_t M, int32_t N,
                int32_t K, hipStream_t st) {
  rows_ring::Args r{};
  r.w = static_cast<const char*>(w);
  r.x = static_cast<const char*>(x);
  r.norm_w = static_cast<const char*>(norm_w);
  r.xs = (int64_t)K * 2;
  r.M = M;
  r.N = r.n_b = N;
  r.row_bytes = K * 2;
  r.eps = eps;
  const typename RingEnd<kEpi>::Args s{static_cast<const bf16_t*>(residual), static_cast<bf16_t*>(y), kEpi == kEpiSiluMul ? N / 2 : N};
  const int granule = kEpi == kEpiSiluMul ? 16 : 1;
  return norm_w ? rows_ring::launch<RingEnd<kEpi>, rows_ring::kNormed>(r, s, granule, st)
                : rows_ring::launch<RingEnd<kEpi>>(r, s, granule, st);
}

// ------------------------------------------------------------------------------------------------
// Tiled form for matrices with few rows and a long K (down_proj: 2560 x 9728): the matrix is cut both ways,
// workgroup (row block, K slice) owns `gpw` row groups (one per wavefront) over a slice of K.  A compute unit moves
// only about 34 GB/s whatever the source, so what counts is the weight plus activation bytes per compute unit and
// that all compute units take part: with one 16-row group per workgroup every workgroup re-reads all of x, as many
// bytes as its weights, and 160 row groups leave 96 compute units idle; a tile of ten row groups over a sixteenth of
// K reads a tenth of its weight bytes in activations and there are 256 of them.  The x slice is staged once in LDS
// in operand order; a wavefront streams its 16 weight rows of the slice (up to twenty loads in flight per lane) and
// stores its fp32 partial block; `skinny_tile_reduce_kernel` adds the K slices in order and applies the epilogue.
// K slices are runs of 32-element MFMA steps, as even as the step count allows.  (The same cut measured slower than
// the other forms for the gate/up and q/k/v matrices, which have rows enough: 29.7 vs 28.0 and 15.7 vs 12.8 us.)
// ------------------------------------------------------------------------------------------------
constexpr int kTileDepth = 20;      // weight vectors in flight per lane
constexpr int kTileMaxSlices = 16;

__global__ __launch_bounds__(kMaxWaves * 64) void skinny_tile_partial_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, float* __restrict__ part, int32_t M, int32_t N, int32_t K,
    int32_t gpw) {
  extern __shared__ __align__(16) u32x4_t xs[];     // [steps padded to kTileDepth][64] x operands of the K slice
  const int tid = threadIdx.x, lane = tid & 63, waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_l = lane & 15, g = lane >> 4;
  const int row_bytes = K * 2;
  const int rb = blockIdx.x, ks = blockIdx.y, n_slices = gridDim.y;
  const int steps_total = K / 32;
  const int s0 = (int)((int64_t)steps_total * ks / n_slices), s1 = (int)((int64_t)steps_total * (ks + 1) / n_slices);
  const int steps = s1 - s0;
  const int steps_max = (steps_total + n_slices - 1) / n_slices;
  const int steps_pad = (steps_max + kTileDepth - 1) / kTileDepth * kTileDepth;    // the host sizes LDS with this
  const int slice_off = s0 * 64;
  const int voff = n_l * row_bytes + g * 16;
  const int groups = (N + 15) >> 4;

  const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(reinterpret_cast<const char*>(x)), 0, M * row_bytes, 0x00020000);
  for (int f = wave; f < steps_pad; f += waves)      // padding steps hold zeros: their products must not be NaN
    xs[f * 64 + lane] = f < steps ? __builtin_amdgcn_raw_buffer_load_b128(rs_x, voff, slice_off + f * 64, 0)
                                  : u32x4_t{0u, 0u, 0u, 0u};
  __syncthreads();

  const int gid = rb * gpw + wave;                   // this wavefront's row group
  if (wave >= gpw || gid >= groups) return;
  const int extent = __builtin_amdgcn_readfirstlane(min(16, N - gid * 16) * row_bytes);
  const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(reinterpret_cast<const char*>(w)) + (int64_t)gid * 16 * row_bytes, 0, extent, 0x00020000);
  floatx4_t acc = floatx4_t{0.f, 0.f, 0.f, 0.f};
  for (int f0 = 0; f0 < steps; f0 += kTileDepth) {
    u32x4_t fw[kTileDepth];
#pragma unroll
    for (int i = 0; i < kTileDepth; ++i) {
      // steps past the slice read through an offset beyond the extent: zeros, no memory access, no branch
      const int vo = f0 + i < steps ? voff : 0x7fffffff - 4096;
      fw[i] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, vo, slice_off + (f0 + i) * 64, 0);
    }
#pragma unroll
    for (int i = 0; i < kTileDepth; ++i)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(xs[(f0 + i) * 64 + lane]), as_frag(fw[i]), acc, 0, 0, 0);
  }
  // acc[e] is the partial of y[m = 4 g + e][16 gid + n_l] over this K slice
  *reinterpret_cast<floatx4_t*>(part + (((int64_t)ks * groups + gid) * 64 + lane) * 4) = acc;
}

// One thread per output element in the order the partial blocks are stored (row group, lane, accumulator element),
// so the reads of every K slice are contiguous; all slices are loaded first and added in K order.
template <int kEpi>
__global__ __launch_bounds__(256) void skinny_tile_reduce_kernel(const float* __restrict__ part,
                                                                 const bf16_t* __restrict__ residual,
                                                                 bf16_t* __restrict__ y, int32_t M, int32_t N,
                                                                 int32_t n_slices) {
  const int groups = (N + 15) >> 4;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;       // (row group, lane, element)
  if (t >= groups * 256) return;
  float v[kTileMaxSlices];
#pragma unroll
  for (int s = 0; s < kTileMaxSlices; ++s) v[s] = s < n_slices ? part[(int64_t)s * groups * 256 + t] : 0.f;
  float sum = 0.f;
#pragma unroll
  for (int s = 0; s < kTileMaxSlices; ++s) sum += v[s];
  const int lane = (t >> 2) & 63;
  const int m = 4 * (lane >> 4) + (t & 3), n = 16 * (t >> 8) + (lane & 15);
  if (m >= M || n >= N) return;
  if (kEpi == kEpiResidual) sum = bf16_to_f32(f32_to_bf16(sum)) + bf16_to_f32(residual[(int64_t)m * N + n]);
  y[(int64_t)m * N + n] = f32_to_bf16(sum);
}

// The cut of the tiled form: up to 16 row groups per row block (fewer when the matrix has fewer than 256 groups), as
// many K slices as keep the launch within one workgroup per compute unit (at most 16); used when it takes at least
// 8 us less per compute unit than the plain form at ~34 GB/s (the second launch costs ~4 us).  The form of rows_ring.h reads the
// activations again once a workgroup, which is cheaper than a second launch up to fourteen of them (us there and here, nine / twelve /
// sixteen rows: 2048 x 6144 9.4 / 9.7 / 10.4 and 11.6, 2560 x 8192 11.8 / 12.5 / 13.4 and 14.2, 4096 x 9728 17.4 / 17.9 / 19.4 and 22,
// 2560 x 9728 14.3 / 15.1 / 16.4 and 15.8) and with more where this form saves no more than some 11 us by that measure, but not for a few
// hundred rows of weights, of which each workgroup there has four (1024 x 9728 11.1 / 11.1 / 11.5 and 9.8 to 10.0).
// Scratch is asked for wherever the cut form could run, the calls that rows_ring.h takes included.
constexpr int kTileMinRows = 8, kRingRows = 14, kTileLong = 7;
constexpr double kTileSaves = 8.0, kTileSavesOfRing = 11.5;
struct TilePlan {
  int n_slices, gpw, row_blocks;
  bool use, ring;                        // worth it beside the plain form, but not beside rows_ring.h
};
TilePlan plan_tile(int32_t M, int32_t N, int32_t K) {
  TilePlan t{0, 0, 0, false, false};
  const int groups = (N + 15) / 16;
  const int steps = K / 32;
  const bool is_long = K > (int64_t)kTileLong * N;
  if (K % 32 != 0 || groups > 256 || (!is_long && M <= kTileMinRows)) return t;
  t.gpw = std::min(kMaxWaves, (groups + 15) / 16);
  t.row_blocks = (groups + t.gpw - 1) / t.gpw;
  t.n_slices = std::min(std::min(kTileMaxSlices, steps), 256 / std::max(1, t.row_blocks));
  if (t.n_slices < 2) return t;
  const double plain_bytes = (16.0 + 16.0) * K * 2;                             // one row group + all of x
  const double tiled_bytes = (16.0 * t.gpw + 16.0) * ((double)K / t.n_slices) * 2;
  const double saves = (plain_bytes - tiled_bytes) / 34e3;                      // bytes / (34 GB/s) in us
  t.use = saves > kTileSaves;
  t.ring = !is_long && takes_ring(N, K, false) && (M <= kRingRows || saves <= kTileSavesOfRing);
  return t;
}

size_t tile_workspace_bytes(const TilePlan& t, int32_t N) {
  return (size_t)t.n_slices * ((N + 15) / 16) * 256 * sizeof(float);
}

template <int R, int kEpi, bool kNorm>
int launch(const void* x, const void* w, const void* residual, const void* norm_w, float eps, void* y, int32_t M,
           int32_t N, int32_t K, int waves, int rows_per_wg, hipStream_t st) {
  const int groups = (N + rows_per_wg - 1) / rows_per_wg;
  const size_t lds = (size_t)waves * (R * 256 + 16) * sizeof(float);
  const int64_t y_stride = kEpi == kEpiSiluMul ? N / 2 : N;
  // with the norm folded in a unit is 64 elements instead of 128: the extra fragments then fit 128 VGPRs
  skinny_linear_kernel<R, kEpi, kNorm, kNorm ? 2 : 4><<<groups, waves * 64, lds, st>>>(
      static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), static_cast<const bf16_t*>(residual),
      static_cast<const bf16_t*>(norm_w), eps, static_cast<bf16_t*>(y), M, N, K, y_stride, rows_per_wg);
  MSA_LAUNCH_CHECK();
  return MSA_OK;
}

}  // namespace

extern "C" int msa_skinny_linear(const void* x, const void* w, const void* residual, const void* norm_w, float eps,
                                 int32_t epilogue, int32_t dtype, int32_t M, int32_t N, int32_t K, void* y,
                                 void* stream) {
  MSA_REQUIRE(x && w && y, "msa_skinny_linear: null pointer");
  MSA_REQUIRE(dtype == MSA_BF16, "msa_skinny_linear: bf16 only");
  MSA_REQUIRE(M > 0 && M <= 16, "msa_skinny_linear: M=%d (1..16 rows)", M);
  MSA_REQUIRE(N > 0 && K > 0 && K % kUnit == 0, "msa_skinny_linear: N=%d K=%d (K must be a multiple of %d)", N, K, kUnit);
  MSA_REQUIRE((int64_t)32 * K * 2 < ((int64_t)1 << 31) && (int64_t)M * K * 2 < ((int64_t)1 << 31),
              "msa_skinny_linear: K=%d too large", K);
  MSA_REQUIRE(epilogue >= kEpiPlain && epilogue <= kEpiSiluMul, "msa_skinny_linear: epilogue %d", epilogue);
  MSA_REQUIRE((epilogue == kEpiResidual) == (residual != nullptr), "msa_skinny_linear: residual pointer and epilogue disagree");
  MSA_REQUIRE(epilogue != kEpiSiluMul || N % 16 == 0, "msa_skinny_linear: silu-mul needs N %% 16 == 0");
  MSA_REQUIRE((((uintptr_t)x | (uintptr_t)w | (uintptr_t)norm_w) & 15) == 0, "msa_skinny_linear: x / w / norm_w must be 16-byte aligned");
  const int units = K / kUnit;
  MSA_REQUIRE(norm_w == nullptr || eps > 0.f, "msa_skinny_linear: folded RMSNorm needs eps > 0");
  hipStream_t st = as_stream(stream);

  if (takes_ring(N, K, norm_w != nullptr)) {
    switch (epilogue) {
      case kEpiPlain: return launch_ring<kEpiPlain>(x, w, residual, norm_w, eps, y, M, N, K, st);
      case kEpiResidual: return launch_ring<kEpiResidual>(x, w, residual, norm_w, eps, y, M, N, K, st);
      case kEpiSiluMul: return launch_ring<kEpiSiluMul>(x, w, residual, norm_w, eps, y, M, N, K, st);
    }
  }

  // Wavefronts per workgroup: split K far enough that the launch has a few thousand wavefronts, and
  // prefer a count that divides the K units so every wavefront streams the same number of bytes.
  // Row groups per wavefront: two share one load of x (every workgroup re-reads x from L2) when N is large
  // enough to still fill the chip with workgroups.
  int R = ((int64_t)N / 32 * kMaxWaves >= 3072 || epilogue == kEpiSiluMul) ? 2 : 1;
  // Rows per workgroup: 16 R, or fewer when that leaves compute units without a workgroup (a compute unit moves
  // only ~34 GB/s, so 256 workgroups of 10 rows beat 160 of 16 on a 2560-row matrix); the silu epilogue needs whole
  // gate / up groups.
  int rows_per_wg = 16 * R;
  if (epilogue != kEpiSiluMul && (N + 16 * R - 1) / (16 * R) < 256) {
    const int spread = std::max(8, (N + 255) / 256);
    if (spread > 16 * (R - 1) && spread < 16 * R) rows_per_wg = spread;
  }
  const int groups = (N + rows_per_wg - 1) / rows_per_wg;
  int want = (int)std::min<int64_t>(kMaxWaves, std::max<int64_t>(1, (4096 + groups - 1) / groups));
  want = std::max(1, std::min(want, units));
  int waves = want;
  for (int cand = want; cand >= std::max(1, want / 2); --cand)
    if (units % cand == 0) { waves = cand; break; }

#define MSA_LIN(R_, E_)                                                                              \
  (norm_w ? launch<R_, E_, true>(x, w, residual, norm_w, eps, y, M, N, K, waves, rows_per_wg, st)    \
          : launch<R_, E_, false>(x, w, residual, norm_w, eps, y, M, N, K, waves, rows_per_wg, st))
  switch (epilogue * 8 + R) {
    case kEpiPlain * 8 + 1: return MSA_LIN(1, kEpiPlain);
    case kEpiPlain * 8 + 2: return MSA_LIN(2, kEpiPlain);
    case kEpiResidual * 8 + 1: return MSA_LIN(1, kEpiResidual);
    case kEpiResidual * 8 + 2: return MSA_LIN(2, kEpiResidual);
    case kEpiSiluMul * 8 + 2: return MSA_LIN(2, kEpiSiluMul);
  }
#undef MSA_LIN
  msa_set_error("msa_skinny_linear: no kernel for epilogue %d with %d row groups", epilogue, R);
  return MSA_EINVAL;
}

extern "C" size_t msa_skinny_linear_workspace_bytes(int32_t M, int32_t N, int32_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const TilePlan t = plan_tile(M, N, K);
  return t.use ? tile_workspace_bytes(t, N) : 0;
}

extern "C" int msa_skinny_linear_ws(const void* x, const void* w, const void* residual, const void* norm_w, float eps,
                                    int32_t epilogue, int32_t dtype, int32_t M, int32_t N, int32_t K, void* y,
                                    void* workspace, size_t workspace_bytes, void* stream) {
  const bool fits = x && w && y && dtype == MSA_BF16 && M > 0 && M <= 16 && N > 0 && K > 0 && K % kUnit == 0 &&
                    norm_w == nullptr && (epilogue == kEpiPlain || epilogue == kEpiResidual) &&
                    (epilogue == kEpiResidual) == (residual != nullptr) && (int64_t)M * K * 2 < ((int64_t)1 << 31) &&
                    (int64_t)32 * K * 2 < ((int64_t)1 << 31) &&
                    (((uintptr_t)x | (uintptr_t)w | (uintptr_t)workspace) & 15) == 0;
  const TilePlan t = fits ? plan_tile(M, N, K) : TilePlan{0, 0, 0, false, false};
  if (!fits || !t.use || t.ring || workspace == nullptr || workspace_bytes < tile_workspace_bytes(t, N))
    return msa_skinny_linear(x, w, residual, norm_w, eps, epilogue, dtype, M, N, K, y, stream);   // it reports bad arguments
  hipStream_t st = as_stream(stream);
  const int groups = (N + 15) / 16;
  const int steps_max = (K / 32 + t.n_slices - 1) / t.n_slices;
  const int steps_pad = (steps_max + kTileDepth - 1) / kTileDepth * kTileDepth;
  const size_t lds = (size_t)steps_pad * 64 * 16;
  MSA_REQUIRE(lds <= 64 * 1024, "msa_skinny_linear_ws: a K slice of %d steps does not fit LDS", steps_max);
  float* part = static_cast<float*>(workspace);
  skinny_tile_partial_kernel<<<dim3(t.row_blocks, t.n_slices), t.gpw * 64, lds, st>>>(
      static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), part, M, N, K, t.gpw);
  MSA_LAUNCH_CHECK();
  if (epilogue == kEpiResidual)
    skinny_tile_reduce_kernel<kEpiResidual><<<groups, 256, 0, st>>>(part, static_cast<const bf16_t*>(residual),
                                                                   static_cast<bf16_t*>(y), M, N, t.n_slices);
  else
    skinny_tile_reduce_kernel<kEpiPlain><<<groups, 256, 0, st>>>(part, nullptr, static_cast<bf16_t*>(y), M, N, t.n_slices);
  MSA_LAUNCH_CHECK();
  return MSA_OK;
}
