// Weight-streaming linear for the rows of a decode step (M <= 16, bf16), with the recurrent decoder's element-wise work in
// the epilogue: gelu, clamped gated units, softcap, the gated residual with the next norm and token shift, the causal convolution, the minimal
// gated recurrence.  Like the skinny linear of the attention model a workgroup owns a few 16-row groups of the weights and
// splits K over its wavefronts (16x16x32 MFMA: the 16 activation rows are exactly one operand); partial sums meet in LDS
// and are added in wavefront order.  Everything behind the sums is element-wise in this model (dynamic tanh has no row
// statistics), so a layer's chain of launches is one per weight matrix plus the state-space / attention step.  Large matrices take
// the form of rows_ring.h with the same ends; this file's kernel is left with small ones, short rows and per-head products.
#include <algorithm>

#include "rows_ring.h"
#include "seq_mfma.h"

namespace {

constexpr int kMaxWaves = 16;
constexpr int kGruGroup = 16;
// A workgroup of rows_ring.h takes 48 rows of the recurrence at least, which leaves compute units without work in small matrices
// (4096 x 1024, 16 rows: 7.5 us against 6.8; 10240 x 2560: 13.8 against 17.5).
constexpr int64_t kGruRingWeights = 8 << 20;

// Units of 32 J elements of K (J 16-byte vectors per lane): shorter when three row groups share the registers.
template <int R>
constexpr int kVectors = R == 3 ? 2 : 4;

// The element-wise end of product (m, n), `col` its column in the output.  What it reads besides the product is fetched by
// `load`, which the kernels call before they multiply, so that it arrives with the weights instead of behind the sums; `begin`
// fetches what the row alone tells, `touches` is whether column n takes any of it: in front of rows_linear_kernel's products nothing
// may be fetched that is not used there, or it is waited for before the weights are requested (3232 x 640: 4.3 us instead of 4.0).
template <int EPI>
struct Finish {
  __device__ __forceinline__ static bool touches(const msa_rows_args&, int) { return true; }
  __device__ __forceinline__ void begin(const msa_rows_args&, int) {}
  __device__ __forceinline__ void load(const msa_rows_args& a, int m, int n) {}
  __device__ __forceinline__ void apply(const msa_rows_args& a, int m, int n, int64_t col, float v) const {
    if constexpr (EPI == MSA_ROWS_F32) {
      if (a.cap > 0.f) v = a.cap * tanh_f(v / a.cap);
      if (a.add) v += a.add[col];
      static_cast<float*>(a.out)[m * a.out_stride + col] = v;
    } else {
      if (EPI == MSA_ROWS_PLAIN && n < a.gelu_n) v = gelu_tanh_f(v);
      static_cast<bf16_t*>(a.out)[m * a.out_stride + col] = f32_to_bf16(v);
    }
  }
};

template <>
struct Finish<MSA_ROWS_MAMBA> {
  static constexpr int kTaps = 4;            // more taps than this are read when they are needed
  float keep[kTaps - 1], tap[kTaps], bias;
  int32_t slot;
  __device__ __forceinline__ static bool touches(const msa_rows_args& a, int n) { return n >= a.conv_lo && n - a.conv_lo < a.conv_n; }
  __device__ __forceinline__ void begin(const msa_rows_args& a, int m) { slot = m < a.M ? a.slot[m] : 0; }
  __device__ __forceinline__ void load(const msa_rows_args& a, int m, int n) {
    const int c = n - a.conv_lo;
    if (c < 0 || c >= a.conv_n) return;
    const float* kp = a.conv_state + (int64_t)slot * (a.conv_k - 1) * a.conv_n + c;
    const float* tp = a.taps + (int64_t)c * a.conv_k;
    bias = a.conv_bias ? a.conv_bias[c] : 0.f;
#pragma unroll
    for (int j = 0; j < kTaps; ++j) {
      if (j + 1 < a.conv_k && j < kTaps - 1) keep[j] = kp[(int64_t)j * a.conv_n];
      if (j < a.conv_k) tap[j] = tp[j];
    }
  }
  __device__ __forceinline__ void apply(const msa_rows_args& a, int m, int n, int64_t col, float v) const {
    const int c = n - a.conv_lo;
    if (c >= 0 && c < a.conv_n) {
      float* kp = a.conv_state + (int64_t)slot * (a.conv_k - 1) * a.conv_n + c;
      float y = bias;
      if (a.conv_k <= kTaps) {
#pragma unroll
        for (int j = 0; j < kTaps; ++j) {
          if (j + 1 < a.conv_k && j < kTaps - 1) {
            y += tap[j] * keep[j];
            if (j > 0) kp[(int64_t)(j - 1) * a.conv_n] = keep[j];
          }
          if (j + 1 == a.conv_k) y += tap[j] * v;
        }
      } else {
        const float* tp = a.taps + (int64_t)c * a.conv_k;
        for (int j = 0; j + 1 < a.conv_k; ++j) {
          const float old = kp[(int64_t)j * a.conv_n];
          y += tp[j] * old;
          if (j > 0) kp[(int64_t)(j - 1) * a.conv_n] = old;
        }
        y += tp[a.conv_k - 1] * v;
      }
      if (a.conv_k > 1) kp[(int64_t)(a.conv_k - 2) * a.conv_n] = v;
      v = silu_f(y);
    }
    static_cast<bf16_t*>(a.out)[m * a.out_stride + col] = f32_to_bf16(v);
  }
};

template <>
struct Finish<MSA_ROWS_RESIDUAL> {
  float x, bias, w, b, mix, before;
  bf16_t gate;
  int32_t slot;
  __device__ __forceinline__ static bool touches(const msa_rows_args&, int) { return true; }
  __device__ __forceinline__ void begin(const msa_rows_args& a, int m) { slot = a.shift && m < a.M ? a.slot[m] : 0; }
  __device__ __forceinline__ void load(const msa_rows_args& a, int m, int n) {
    x = a.x_in[(int64_t)m * a.N + n];
    gate = static_cast<const bf16_t*>(a.gate)[m * a.gate_stride + n];
    bias = a.gate_bias[n];
    if (!a.norm.w) return;
    w = a.norm.w[n];
    b = a.norm.b[n];
    if (!a.shift) return;
    mix = a.shift[n];
    before = a.prev[(int64_t)slot * a.N + n];
  }
  __device__ __forceinline__ void apply(const msa_rows_args& a, int m, int n, int64_t, float v) const {
    const int64_t at = (int64_t)m * a.N + n;
    const float y = x + sigmoid_f(bf16_to_f32(gate) + bias) * v;
    a.x_out[at] = y;
    if (!a.norm.w) return;
    const float h = tanh_f(a.norm.alpha * y) * w + b;
    if (a.h) static_cast<bf16_t*>(a.h)[at] = f32_to_bf16(h);
    if (!a.shift) return;
    a.prev[(int64_t)slot * a.N + n] = h;
    static_cast<bf16_t*>(a.h_shift)[at] = f32_to_bf16(h + (before - h) * mix);
  }
};

// A (gate, up) pair of neighbouring columns, in the lane of the even one.
template <>
struct Finish<MSA_ROWS_GLU> {
  __device__ __forceinline__ static bool touches(const msa_rows_args&, int) { return false; }
  __device__ __forceinline__ void begin(const msa_rows_args&, int) {}
  __device__ __forceinline__ void load(const msa_rows_args& a, int m, int n) {}
  __device__ __forceinline__ void apply(const msa_rows_args& a, int m, int n, float gate, float up) const {
    if (n & 1) return;
    static_cast<bf16_t*>(a.out)[m * a.out_stride + (n >> 1)] = f32_to_bf16(clamped_glu_f(gate, up, a.glu_limit, a.glu_alpha, a.glu_shift));
  }
};

template <int EPI, int R>
__device__ __forceinline__ void rows_linear(const msa_rows_args& a, int32_t rows_per_wg) {
  constexpr int J = kVectors<R>, kUnit = 32 * J;
  extern __shared__ __align__(16) float part[];   // [waves][R][64][4]
  const int tid = threadIdx.x, lane = tid & 63, waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_l = lane & 15, g = lane >> 4;
  const int n_base = blockIdx.x * rows_per_wg, grp = blockIdx.y;
  const int row_bytes = a.K * 2;
  const int rows_w = min(rows_per_wg, a.N - n_base);
  const bool second = n_base >= a.n_b;
  const int64_t xs = second ? a.x_b_stride : a.x_stride;
  const char* xbase = static_cast<const char*>(second ? a.x_b : a.x) + (int64_t)grp * row_bytes;
  const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(static_cast<const char*>(a.w)) + ((int64_t)grp * a.N + n_base) * row_bytes, 0, rows_w * row_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(xbase), 0, (int)((a.M - 1) * xs * 2 + row_bytes), 0x00020000);
  const int voff_w = n_l * row_bytes + g * 16, voff_x = n_l * (int)(xs * 2) + g * 16;
  constexpr int kFar = 0x7ff00000;          // past every extent, whatever is added: reads zeros
  const int units = (a.K + kUnit - 1) / kUnit;
  const int u0 = units * wave / waves, u1 = units * (wave + 1) / waves;

  // output i of a row group: lane i / 4, element i % 4 of its accumulator
  auto row_of = [](int i) { return 4 * (i >> 6) + (i & 3); };
  auto col_of = [](int i) { return (i >> 2) & 15; };
  Finish<EPI> fin;                          // of this thread's first output
  {
    const int m = row_of(tid & 255), nr = 16 * (tid >> 8) + col_of(tid & 255);
    if (tid < R * 256 && m < a.M && nr < rows_w && fin.touches(a, n_base + nr)) {
      fin.begin(a, m);
      fin.load(a, m, n_base + nr);
    }
  }

  floatx4_t acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  u32x4_t fw[2][R][J], fx[2][J];
  auto load_unit = [&](int slot, int u) {
    const int k_off = u * kUnit * 2;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const bool in = k_off + j * 64 + g * 16 < row_bytes;        // pieces behind K read as zero
      fx[slot][j] = __builtin_amdgcn_raw_buffer_load_b128(rs_x, in ? voff_x : kFar, k_off + j * 64, 0);
#pragma unroll
      for (int r = 0; r < R; ++r)
        fw[slot][r][j] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, in ? voff_w + r * 16 * row_bytes : kFar, k_off + j * 64, 0);
    }
  };
  auto mul_unit = [&](int slot) {
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int r = 0; r < R; ++r)
        acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, fx[slot][j]),
                                                         __builtin_bit_cast(bf16x8_t, fw[slot][r][j]), acc[r], 0, 0, 0);
  };
  if (u0 < u1) load_unit(0, u0);
  int u = u0;
  for (; u + 2 <= u1; u += 2) {
    load_unit(1, u + 1);
    mul_unit(0);
    if (u + 2 < u1) load_unit(0, u + 2);
    mul_unit(1);
  }
  if (u < u1) mul_unit(0);

#pragma unroll
  for (int r = 0; r < R; ++r) *reinterpret_cast<floatx4_t*>(&part[((wave * R + r) * 64 + lane) * 4]) = acc[r];
  __syncthreads();

  auto total = [&](int r, int i) {
    float v = 0.f;
    for (int w = 0; w < waves; ++w) v += part[(w * R + r) * 256 + i];
    return v;
  };
  if constexpr (EPI == MSA_ROWS_GRU) {
    if (!second) {
      for (int i = tid; i < 256; i += blockDim.x) {
        const int m = row_of(i), c = n_base / (3 * kGruGroup) * kGruGroup + col_of(i);
        if (m >= a.M || c >= a.gru_n) continue;
        float* st = a.gru_state + (int64_t)a.slot[m] * a.gru_n + c;
        const float before = *st, zb = a.z_bias[c], ub = a.u_bias[c];
        const float z = sigmoid_f(total(0, i) + zb), uu = total(1, i) + ub, gt = total(2, i);
        const float S = (1.0f - z) * before + z * (uu >= 0.f ? uu + 0.5f : sigmoid_f(uu));
        *st = S;
        static_cast<bf16_t*>(a.out2)[(int64_t)m * a.gru_n + c] = f32_to_bf16(S * silu_f(gt));
      }
      return;
    }
  }
  for (int o = tid; o < R * 256; o += blockDim.x) {
    const int r = o >> 8, i = o & 255;
    const int m = row_of(i), nr = 16 * r + col_of(i), n = n_base + nr;
    if (m >= a.M || nr >= rows_w) continue;
    if constexpr (EPI == MSA_ROWS_GLU) {    // (rows come in pairs: the neighbouring column is in this wavefront, four lanes on)
      const float v = total(r, i), up = __shfl_xor(v, 4);
      fin.apply(a, m, n, v, up);
    } else {
      if (o != tid && fin.touches(a, n)) {
        fin.begin(a, m);
        fin.load(a, m, n);
      }
      fin.apply(a, m, n, (int64_t)grp * a.N + n, total(r, i));
    }
  }
}

template <int EPI, int R>
__global__ __launch_bounds__(kMaxWaves * 64) void rows_linear_kernel(msa_rows_args a, int32_t rows_per_wg) {
  rows_linear<EPI, R>(a, rows_per_wg);
}

// The same beside the appending of the rows' latents, which needs nothing of the products: the last column of workgroups does that.
template <int R>
__global__ __launch_bounds__(kMaxWaves * 64) void rows_append_kernel(msa_rows_args a, int32_t rows_per_wg, msa_rows_append p, msa_seq_batch b) {
  if (blockIdx.x + 1 < gridDim.x) return rows_linear<MSA_ROWS_PLAIN, R>(a, rows_per_wg);
  const int waves = blockDim.x >> 6;
  for (int row = blockIdx.y * waves + (threadIdx.x >> 6); row < b.rows; row += gridDim.y * waves)
    append_latent<bf16_t, 8>(static_cast<const bf16_t*>(p.in), p.in_stride, p.w, p.eps, p.rank, static_cast<bf16_t*>(p.cache), p.Lcap, b, row);
}

// What rows_ring.h's kernel does with a product: the same ends, and the minimal gated recurrence, whose three sums of a channel
// are three consecutive items of a workgroup.
template <int EPI>
struct RingEnd {
  using Args = msa_rows_args;
  Finish<EPI> fin;
  __device__ __forceinline__ void begin(const Args& a, int m) { fin.begin(a, m); }
  __device__ __forceinline__ void load(const Args& a, int m, int n, bool mine, bool, int) {
    if (mine) fin.load(a, m, n);
  }
  __device__ __forceinline__ void apply(const Args& a, int m, int n, float v, bool mine, bool, int) const {
    if constexpr (EPI == MSA_ROWS_GLU) {
      const float up = __shfl_xor(v, 4);
      if (mine) fin.apply(a, m, n, v, up);
    } else if (mine) {
      fin.apply(a, m, n, n, v);
    }
  }
};

template <>
struct RingEnd<MSA_ROWS_GRU> {
  using Args = msa_rows_args;
  float before = 0.f, zb = 0.f, ub = 0.f, z = 0.f, u = 0.f;
  int32_t slot;
  __device__ __forceinline__ void begin(const Args& a, int m) { slot = m < a.M ? a.slot[m] : 0; }
  __device__ __forceinline__ static int channel(int n) { return n / (3 * kGruGroup) * kGruGroup + n % kGruGroup; }
  __device__ __forceinline__ void load(const Args& a, int m, int n, bool mine, bool second, int item) {
    const int c = channel(n);
    if (second || !mine || item % 3 != 0 || c >= a.gru_n) return;
    before = a.gru_state[(int64_t)slot * a.gru_n + c];
    zb = a.z_bias[c];
    ub = a.u_bias[c];
  }
  __device__ __forceinline__ void apply(const Args& a, int m, int n, float v, bool mine, bool second, int item) {
    if (!mine) return;
    if (second) {
      static_cast<bf16_t*>(a.out)[m * a.out_stride + n] = f32_to_bf16(v);
      return;
    }
    const int c = channel(n), part = item % 3;
    if (c >= a.gru_n) return;
    z = part == 0 ? sigmoid_f(v + zb) : z;
    u = part == 1 ? v + ub : u;
    if (part < 2) return;
    const float S = (1.0f - z) * before + z * (u >= 0.f ? u + 0.5f : sigmoid_f(u));
    a.gru_state[(int64_t)slot * a.gru_n + c] = S;
    static_cast<bf16_t*>(a.out2)[(int64_t)m * a.gru_n + c] = f32_to_bf16(S * silu_f(v));
  }
};

// The weight ring's part of the calls (us without and with it, one / sixteen rows: 2560 x 1536 4.2 / 5.2 and 4.5 / 5.2, 3072 x 1280 4.0 /
// 4.9 and 4.6 / 5.1, 2048 x 1024 3.5 / 4.2 and 3.6 / 4.2; 4096 x 1024 4.1 / 4.6 and 4.0 / 4.3, 1024 x 3072 5.3 / 7.2 and 5.1 / 6.9; with
// fp32 results 512 x 6144 7.0 and 7.4, 768 x 3584 5.3 and 5.6).  From 2048 elements on this file's kernel is short of wavefronts.
constexpr int64_t kRingWeights = 3 << 20, kLongRingWeights = 3 << 19, kLongK = 2048;
bool takes_ring(const msa_rows_args& a, int32_t epilogue) {
  if (a.groups != 1 || a.K <= rows_ring::kMinK) return false;
  if (epilogue == MSA_ROWS_GRU) return (int64_t)a.N * a.K >= kGruRingWeights;
  return rows_ring::busy_weights(a.N, a.K) >= kRingWeights || (epilogue != MSA_ROWS_F32 && a.K >= kLongK && (int64_t)a.N * a.K >= kLongRingWeights);
}

template <int EPI, int kPro = rows_ring::kPlain>
int launch_ring(const msa_rows_args& a, hipStream_t st, const msa_rows_post* post = nullptr, const float* next_w = nullptr,
                const msa_rows_embed* embed = nullptr) {
  rows_ring::Args r{};
  r.post_next = next_w;
  if (embed) {
    r.tokens = embed->tokens;
    r.vocab = embed->vocab;
    r.post_out = embed->x_out;
  }
  if (post) {
    r.post_x = post->x_in;
    r.post_w = post->w;
    r.post_out = post->x_out;
    r.eps = post->eps;
  }
  r.w = static_cast<const char*>(a.w);
  r.x = static_cast<const char*>(a.x);
  r.x_b = static_cast<const char*>(a.x_b);
  r.xs = a.x_stride * 2;
  r.xbs = a.x_b_stride * 2;
  r.M = a.M;
  r.N = a.N;
  r.n_b = a.n_b;
  r.row_bytes = a.K * 2;
  return rows_ring::launch<RingEnd<EPI>, kPro>(r, a, EPI == MSA_ROWS_GRU ? 3 * kGruGroup : EPI == MSA_ROWS_GLU ? 2 : 1, st);
}

template <int EPI, int R>
int launch_rows(const msa_rows_args& a, int waves, int rows_per_wg, hipStream_t st, const msa_rows_append* append = nullptr) {
  const size_t lds = (size_t)waves * R * 256 * sizeof(float);       // at most 48 KB
  if (EPI == MSA_ROWS_PLAIN && append)
    rows_append_kernel<R><<<dim3((a.N + rows_per_wg - 1) / rows_per_wg + 1, a.groups), waves * 64, lds, st>>>(a, rows_per_wg, *append, *append->batch);
  else
    rows_linear_kernel<EPI, R><<<dim3((a.N + rows_per_wg - 1) / rows_per_wg, a.groups), waves * 64, lds, st>>>(a, rows_per_wg);
  MSA_LAUNCH_CHECK();
  return MSA_OK;
}

}  // namespace

namespace {
int rows_entry(const msa_rows_args& a, int32_t epilogue, const msa_rows_post* post, void* stream, const float* next_w = nullptr,
               const msa_rows_embed* embed = nullptr, const msa_rows_append* append = nullptr) {
  MSA_REQUIRE(a.x && a.w && a.M > 0 && a.M <= 16 && a.N > 0 && a.K > 0 && a.K % 8 == 0 && a.groups > 0 && a.groups <= 65535,
              "msa_rows_linear: M=%d (1..16) N=%d K=%d (a multiple of 8) groups=%d", a.M, a.N, a.K, a.groups);
  MSA_REQUIRE(a.x_stride >= (int64_t)a.K * a.groups && a.x_stride % 8 == 0 && a.x_stride * 32 < ((int64_t)1 << 30) &&
                  (int64_t)64 * a.K * 2 < ((int64_t)1 << 30), "msa_rows_linear: x_stride=%lld K=%d", (long long)a.x_stride, a.K);
  const bool two = a.n_b < a.N;
  MSA_REQUIRE(a.n_b > 0 && (!two || (a.x_b && a.groups == 1 && a.x_b_stride >= a.K && a.x_b_stride % 8 == 0 &&
                                     a.x_b_stride * 32 < ((int64_t)1 << 30))), "msa_rows_linear: second operand");
  MSA_REQUIRE((((uintptr_t)a.x | (uintptr_t)a.x_b | (uintptr_t)a.w) & 15) == 0, "msa_rows_linear: x / x_b / w must be 16-byte aligned");
  switch (epilogue) {
    case MSA_ROWS_PLAIN:
    case MSA_ROWS_F32:
      MSA_REQUIRE(a.out && a.out_stride >= (int64_t)a.N * a.groups, "msa_rows_linear: output");
      break;
    case MSA_ROWS_RESIDUAL:
      MSA_REQUIRE(a.x_in && a.x_out && a.gate && a.gate_bias && a.gate_stride >= a.N && a.groups == 1 && !two, "msa_rows_linear: residual arguments");
      MSA_REQUIRE(!a.norm.w || (a.norm.b && (a.h || a.shift)), "msa_rows_linear: norm arguments");
      MSA_REQUIRE(!a.shift || (a.norm.w && a.prev && a.h_shift && a.slot), "msa_rows_linear: shift arguments");
      break;
    case MSA_ROWS_MAMBA:
      MSA_REQUIRE(a.out && a.out_stride >= a.N && a.groups == 1 && a.taps && a.slot && a.conv_k >= 1 && a.conv_lo >= 0 &&
                      a.conv_n > 0 && a.conv_lo + a.conv_n <= a.n_b && (a.conv_k == 1 || a.conv_state), "msa_rows_linear: convolution arguments");
      break;
    case MSA_ROWS_GLU:
      MSA_REQUIRE(a.out && a.N % 2 == 0 && a.out_stride >= a.N / 2 && a.groups == 1 && !two, "msa_rows_linear: gated unit arguments");
      break;
    case MSA_ROWS_GRU:
      MSA_REQUIRE(a.out2 && a.z_bias && a.u_bias && a.gru_state && a.slot && a.groups == 1 && a.gru_n > 0 &&
                      a.n_b == (a.gru_n + kGruGroup - 1) / kGruGroup * 3 * kGruGroup && (!two || (a.out && a.out_stride >= a.N)),
                  "msa_rows_linear: recurrence arguments");
      break;
    default:
      msa_set_error("msa_rows_linear: epilogue %d", epilogue);
      return MSA_EINVAL;
  }
  // Row groups per workgroup: two when N alone fills the chip (the activations are then read half as often); fewer than 16
  // rows when that leaves compute units without a workgroup.  Wavefronts: a few thousand in the launch, and a share of K each.
  const bool gru = epilogue == MSA_ROWS_GRU;
  int R = gru ? 3 : ((int64_t)a.N * a.groups >= 6144 && (!two || a.n_b % 32 == 0) && a.N >= 32) ? 2 : 1;
  int rows_per_wg = 16 * R;
  MSA_REQUIRE(!two || a.n_b % rows_per_wg == 0, "msa_rows_linear: n_b=%d must be a multiple of %d", a.n_b, rows_per_wg);
  if (R == 1 && !two && a.groups == 1 && (a.N + 15) / 16 < device_compute_units())
    rows_per_wg = std::min(16, std::max(8, (a.N + device_compute_units() - 1) / device_compute_units()));
  if (epilogue == MSA_ROWS_GLU) rows_per_wg = (rows_per_wg + 1) & ~1;
  const int64_t wgs = (int64_t)((a.N + rows_per_wg - 1) / rows_per_wg) * a.groups;
  const int kUnit = 32 * (R == 3 ? kVectors<3> : kVectors<1>);
  const int units = (a.K + kUnit - 1) / kUnit;
  int waves = (int)std::min<int64_t>(kMaxWaves, std::max<int64_t>(1, (4096 + wgs - 1) / wgs));
  waves = std::max(1, std::min(waves, units));
  for (int cand = waves; cand >= std::max(1, waves / 2); --cand)
    if (units % cand == 0) { waves = cand; break; }
  hipStream_t st = as_stream(stream);
  if (takes_ring(a, epilogue)) {
    if (embed && epilogue == MSA_ROWS_MAMBA) return launch_ring<MSA_ROWS_MAMBA, rows_ring::kEmbed>(a, st, nullptr, nullptr, embed);
    if (embed) return launch_ring<MSA_ROWS_PLAIN, rows_ring::kEmbed>(a, st, nullptr, nullptr, embed);
    if (post && next_w) return launch_ring<MSA_ROWS_F32, rows_ring::kFinal>(a, st, post, next_w);
    if (post) {
      switch (epilogue) {
        case MSA_ROWS_PLAIN: return launch_ring<MSA_ROWS_PLAIN, rows_ring::kPost>(a, st, post);
        case MSA_ROWS_MAMBA: return launch_ring<MSA_ROWS_MAMBA, rows_ring::kPost>(a, st, post);
        case MSA_ROWS_GLU: return launch_ring<MSA_ROWS_GLU, rows_ring::kPost>(a, st, post);
      }
    }
    switch (epilogue) {
      case MSA_ROWS_PLAIN: return launch_ring<MSA_ROWS_PLAIN>(a, st);
      case MSA_ROWS_F32: return launch_ring<MSA_ROWS_F32>(a, st);
      case MSA_ROWS_RESIDUAL: return launch_ring<MSA_ROWS_RESIDUAL>(a, st);
      case MSA_ROWS_MAMBA: return launch_ring<MSA_ROWS_MAMBA>(a, st);
      case MSA_ROWS_GLU: return launch_ring<MSA_ROWS_GLU>(a, st);
      case MSA_ROWS_GRU: return launch_ring<MSA_ROWS_GRU>(a, st);
    }
  }
  switch (epilogue * 4 + R) {
    case MSA_ROWS_PLAIN * 4 + 1: return launch_rows<MSA_ROWS_PLAIN, 1>(a, waves, rows_per_wg, st, append);
    case MSA_ROWS_PLAIN * 4 + 2: return launch_rows<MSA_ROWS_PLAIN, 2>(a, waves, rows_per_wg, st, append);
    case MSA_ROWS_F32 * 4 + 1: return launch_rows<MSA_ROWS_F32, 1>(a, waves, rows_per_wg, st);
    case MSA_ROWS_F32 * 4 + 2: return launch_rows<MSA_ROWS_F32, 2>(a, waves, rows_per_wg, st);
    case MSA_ROWS_RESIDUAL * 4 + 1: return launch_rows<MSA_ROWS_RESIDUAL, 1>(a, waves, rows_per_wg, st);
    case MSA_ROWS_RESIDUAL * 4 + 2: return launch_rows<MSA_ROWS_RESIDUAL, 2>(a, waves, rows_per_wg, st);
    case MSA_ROWS_MAMBA * 4 + 1: return launch_rows<MSA_ROWS_MAMBA, 1>(a, waves, rows_per_wg, st);
    case MSA_ROWS_MAMBA * 4 + 2: return launch_rows<MSA_ROWS_MAMBA, 2>(a, waves, rows_per_wg, st);
    case MSA_ROWS_GLU * 4 + 1: return launch_rows<MSA_ROWS_GLU, 1>(a, waves, rows_per_wg, st);
    case MSA_ROWS_GLU * 4 + 2: return launch_rows<MSA_ROWS_GLU, 2>(a, waves, rows_per_wg, st);
    case MSA_ROWS_GRU * 4 + 3: return launch_rows<MSA_ROWS_GRU, 3>(a, waves, rows_per_wg, st);
  }
  msa_set_error("msa_rows_linear: no kernel for epilogue %d with %d row groups", epilogue, R);
  return MSA_EINVAL;
}
}  // namespace

extern "C" int msa_rows_linear(const msa_rows_args* args, int32_t epilogue, void* stream) {
  MSA_REQUIRE(args != nullptr, "msa_rows_linear: null arguments");
  return rows_entry(*args, epilogue, nullptr, stream);
}

// One launch for the latents and the products of the queries with the heads' matrices, which follow one another in a step but need nothing
// of each other (whole steps, us: one sequence of the 1b size 165.0 and 161.6, eight 183.4 and 180.3, sixteen of the 4b size 434 and 430).
extern "C" int msa_rows_linear_append(const msa_rows_args* args, const msa_rows_append* append, void* stream) {
  MSA_REQUIRE(args && append, "msa_rows_linear_append: null arguments");
  const msa_rows_append& p = *append;
  MSA_CHECK_BATCH(p.batch, "msa_rows_linear_append");
  MSA_REQUIRE(p.in && p.w && p.cache && p.rank > 0 && p.in_stride >= p.rank && p.Lcap > 0, "msa_rows_linear_append: bad arguments");
  if (!takes_ring(*args, MSA_ROWS_PLAIN) && vec_ok(8, {p.in, p.w, p.cache}, {p.in_stride, p.rank})) return rows_entry(*args, MSA_ROWS_PLAIN, nullptr, stream, nullptr, nullptr, append);
  if (const int rc = msa_seq_latent_append(p.in, p.in_stride, p.w, p.eps, MSA_BF16, p.rank, p.cache, p.Lcap, p.batch, stream); rc != MSA_OK) return rc;
  return rows_entry(*args, MSA_ROWS_PLAIN, nullptr, stream);
}

// The residual step is folded where its operands are few: every workgroup reads all of them, six bytes an element where the product
// alone reads two, and waits for a second reduction.  That is worth less than a launch up to 8192 elements in rows of one unit a
// wavefront, and in longer ones up to 6144 if the product is no short one itself (with the product, us, folded against separate: 1 and 8
// rows of 1024 with 3104 x 1024 6.0 / 6.4 and 6.7 / 6.7, 3 of 2048 with 6144 x 2048 9.7 / 9.9, 2 of 2560 with 6144 x 2560 11.5 / 11.8; but
// 3 of 2560 with 3104 x 2560 10.2 / 8.9, 4 of 2048 with 1024 x 2048 8.3 / 7.6, 5 of 1280 with 6144 x 1280 and the convolution 10.3 / 9.7,
// 16 of 2560 28.0 / 22.7).  The separate launch also works in place and takes rows that the ring's registers do not hold.
constexpr int kMaxPostElements = 8192, kMaxLongPostElements = 6144, kPostRow = rows_ring::kWaves * rows_ring::kUnitBytes / 2;
constexpr int64_t kMinLongPostWeights = 12 << 20;
bool worth_folding(const msa_rows_args& a) {
  const int64_t elements = a.M * (int64_t)a.K;
  return a.K <= kPostRow ? elements <= kMaxPostElements : elements <= kMaxLongPostElements && (int64_t)a.N * a.K >= kMinLongPostWeights;
}
// What the residual step asks of its operands to be formed on the way.
static bool post_fits(const msa_rows_args& a, const msa_rows_post* post) {
  return a.K % 8 == 0 && a.K <= rows_ring::kMaxPost * rows_ring::kWaves * rows_ring::kUnitBytes / 2 &&
         (((uintptr_t)post->x_in | (uintptr_t)post->x_out | (uintptr_t)post->w) & 15) == 0;
}
// Likewise in front of the head, in the same limits (steps of one, 4 and 8 rows of 1024: 180.3, 185.9 and 196.6 us separate, 179.2, 184.9
// and 195.3 folded: of the launch's 5 us a second reduction, behind the first and while the whole ring waits, costs most).
extern "C" int msa_rows_linear_final(const msa_rows_args* args, const msa_rows_post* post, const float* next_w, void* stream) {
  MSA_REQUIRE(args && post && next_w && post->x_in && post->w && post->h && post->eps >= 0.f, "msa_rows_linear_final: null arguments");
  msa_rows_args a = *args;
  MSA_REQUIRE(a.x && a.M > 0 && a.M <= 16 && a.K > 0 && a.groups == 1 && a.x_stride >= a.K && a.n_b >= a.N,
              "msa_rows_linear_final: M=%d (1..16) K=%d groups=%d n_b=%d", a.M, a.K, a.groups, a.n_b);
  if (takes_ring(a, MSA_ROWS_F32) && worth_folding(a) && post_fits(a, post) && ((uintptr_t)next_w & 15) == 0) return rows_entry(a, MSA_ROWS_F32, post, stream, next_w);
  MSA_REQUIRE(post->x_out, "msa_rows_linear_final: the separate launch needs x_out");
  if (const int rc = msa_seq_rms_residual(post->x_in, a.x, a.x_stride, post->w, post->eps, post->x_out, next_w, post->h, MSA_BF16, a.M, a.K, stream); rc != MSA_OK) return rc;
  a.x = post->h;
  a.x_stride = a.K;
  return rows_entry(a, MSA_ROWS_F32, nullptr, stream);
}
// The lookup is folded wherever the ring's registers hold the rows and 32-bit offsets reach the table: every workgroup reads the same bytes
// as without, one latency (the tokens') later.  Whole decode steps of four layers, us, with the launch of its own and without: one row of
// 1024 179.7 and 176.2, 4 rows 185.1 and 180.9, one of 2560 384.3 and 380.8, 16 of them 485.7 and 481.4.
extern "C" int msa_rows_linear_embed(const msa_rows_args* args, int32_t epilogue, const msa_rows_embed* embed, void* stream) {
  MSA_REQUIRE(args && embed && embed->tokens && embed->table && embed->x_out && embed->h, "msa_rows_linear_embed: null arguments");
  msa_rows_args a = *args;
  MSA_REQUIRE(a.M > 0 && a.M <= 16 && a.K > 0 && a.K % 8 == 0 && a.groups == 1 && a.n_b >= a.N && embed->vocab > 0 &&
                  (((uintptr_t)embed->table | (uintptr_t)embed->x_out | (uintptr_t)embed->h) & 15) == 0,
              "msa_rows_linear_embed: M=%d (1..16) K=%d groups=%d n_b=%d, 16-byte alignment", a.M, a.K, a.groups, a.n_b);
  a.x = embed->table;
  a.x_stride = a.K;
  if ((epilogue == MSA_ROWS_PLAIN || epilogue == MSA_ROWS_MAMBA) && takes_ring(a, epilogue) && a.K <= rows_ring::kMaxResidentK &&
      embed->vocab <= rows_ring::kFar / (a.K * 2))
    return rows_entry(a, epilogue, nullptr, stream, nullptr, embed);
  if (const int rc = msa_embed_rows(embed->tokens, a.M, embed->table, embed->vocab, 1, a.K, MSA_BF16, embed->h, embed->x_out, stream); rc != MSA_OK) return rc;
  a.x = embed->h;
  return rows_entry(a, epilogue, nullptr, stream);
}
extern "C" int msa_rows_linear_post(const msa_rows_args* args, int32_t epilogue, const msa_rows_post* post, void* stream) {
  MSA_REQUIRE(args && post && post->x_in && post->x_out && post->w && post->h && post->eps >= 0.f, "msa_rows_linear_post: null arguments");
  msa_rows_args a = *args;
  MSA_REQUIRE(a.x && a.M > 0 && a.M <= 16 && a.K > 0 && a.groups == 1 && a.x_stride >= a.K && a.n_b >= a.N,
              "msa_rows_linear_post: M=%d (1..16) K=%d groups=%d n_b=%d", a.M, a.K, a.groups, a.n_b);
  const bool folds = (epilogue == MSA_ROWS_PLAIN || epilogue == MSA_ROWS_MAMBA || epilogue == MSA_ROWS_GLU) && takes_ring(a, epilogue) && worth_folding(a) && post_fits(a, post) &&
                     post->x_in != post->x_out;
  if (folds) return rows_entry(a, epilogue, post, stream);
  if (const int rc = msa_seq_rms_residual(post->x_in, a.x, a.x_stride, post->w, post->eps, post->x_out, nullptr, post->h, MSA_BF16, a.M, a.K, stream); rc != MSA_OK) return rc;
  a.x = post->h;
  a.x_stride = a.K;
  return rows_entry(a, epilogue, nullptr, stream);
}
