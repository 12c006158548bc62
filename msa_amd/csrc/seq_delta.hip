// Delta rule with a decay per key channel, token by token: the form for decoding, short portions and fp32 (the chunked
// matrix-core form is in seq_delta_chunk.hip).
//
// A workgroup owns (sequence, head, up to 128 value columns): lane = column, and the wavefronts of a column group share the
// state's rows, which they keep in registers.  A few tokens are staged at a time (unit vectors, decays, step sizes in LDS).  Both
// sums over the rows are taken from the decayed state in one pass, since
//   o = (S + k u^T)^T q = S^T q + (k . q) u,
// so a token costs one exchange and one barrier.  When the workgroup has all of a head's columns it also finishes the output
// (norm and gate); otherwise head_norm_gate_kernel does.
#include <algorithm>

#include "seq_mfma.h"

namespace {

constexpr int kTok = 8;                  // tokens per stage

template <typename T, int NI, int RW, int CW>
__global__ __launch_bounds__(RW * CW * 64) void delta_scan_kernel(msa_delta_args a, msa_seq_batch b) {
  constexpr int kD = NI * RW, kCols = CW * 64, kWaves = RW * CW;
  __shared__ __align__(16) float ks[kTok][kD], qs[kTok][kD], gs[kTok][kD];
  __shared__ float beta[kTok], kq[kTok];
  __shared__ float2 part[2][RW][kCols];
  __shared__ float os[kTok][kCols];
  const int s = blockIdx.z, head = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), cw = wave % CW, rw = wave / CW;
  const int col0 = blockIdx.x * kCols, cl = cw * 64 + lane, col = col0 + cl;
  const bool live = col < a.E, whole = gridDim.x == 1;
  const int lo = b.cu[s], n_tok = b.cu[s + 1] - lo, kvh = head / (a.H / a.G);
  float* st = a.state + (((int64_t)b.slot[s] * a.H + head) * a.D + rw * NI) * a.E + col;
  const float rate = -expf(a.A_log[head]), q_scale = 1.0f / sqrtf((float)a.D);
  const float* bias = a.dt_bias + (int64_t)head * a.D;
  const T* qkv = static_cast<const T*>(a.qkv) + (int64_t)lo * a.qkv_stride;
  const T* qp = qkv + (int64_t)kvh * a.D;
  const T* kp = qp + (int64_t)a.G * a.D;
  const T* vp = qkv + 2LL * a.G * a.D + (int64_t)head * a.E;
  const T* ap = static_cast<const T*>(a.a) + (int64_t)lo * a.a_stride + (int64_t)head * a.D;
  const T* bp = static_cast<const T*>(a.b) + (int64_t)lo * a.b_stride + head;
  const T* gp = static_cast<const T*>(a.gate) + (int64_t)lo * a.gate_stride + (int64_t)head * a.E;
  constexpr int kEach = (kD + 63) / 64, kMine = (kTok + kWaves - 1) / kWaves;    // values of a lane, tokens of a wavefront in a stage
  // What a stage reads is requested together, and the first one's in front of the state: loads arrive in the order they are made,
  // and the vectors are ready by the time the state is there.
  float k[kMine][kEach], q[kMine][kEach], x[kMine][kEach], bv[kMine], v[kTok], db[kEach];
#pragma unroll
  for (int j = 0; j < kEach; ++j) db[j] = lane + 64 * j < a.D ? bias[lane + 64 * j] : 0.f;
  auto fetch = [&](int t0) {
    const int rows = min(kTok, n_tok - t0);
#pragma unroll
    for (int m = 0; m < kMine; ++m) {
      const int r = wave + m * kWaves;
      const int64_t t = t0 + min(r, rows - 1);
#pragma unroll
      for (int j = 0; j < kEach; ++j) {
        const int i = lane + 64 * j;
        const bool in = i < a.D;
        k[m][j] = in ? to_f32<T>(kp[t * a.qkv_stride + i]) : 0.f;
        q[m][j] = in ? to_f32<T>(qp[t * a.qkv_stride + i]) : 0.f;
        x[m][j] = in ? to_f32<T>(ap[t * a.a_stride + i]) : 0.f;
      }
      bv[m] = to_f32<T>(bp[t * a.b_stride]);
    }
#pragma unroll
    for (int r = 0; r < kTok; ++r) v[r] = live && r < rows ? to_f32<T>(vp[(t0 + r) * a.qkv_stride + col]) : 0.f;
  };
  fetch(0);
  const float out_w = live && whole ? a.norm[col] : 0.f;
  const float gate0 = live && whole ? to_f32<T>(gp[col]) : 0.f;        // of the first token, all there is when decoding
  float S[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) S[i] = live && rw * NI + i < a.D ? st[(int64_t)i * a.E] : 0.f;
  for (int t0 = 0; t0 < n_tok; t0 += kTok) {
    const int rows = min(kTok, n_tok - t0);
    if (t0 > 0) fetch(t0);
#pragma unroll
    for (int m = 0; m < kMine; ++m) {                    // a wavefront per token
      const int r = wave + m * kWaves;
      if (r >= rows) break;
      float kk = 0.f, qq = 0.f, dot = 0.f;
#pragma unroll
      for (int j = 0; j < kEach; ++j) {
        const int i = lane + 64 * j;
        if (i < kD) gs[r][i] = i < a.D ? expf(rate * softplus_f(x[m][j] + db[j])) : 0.f;
        kk += k[m][j] * k[m][j];
        qq += q[m][j] * q[m][j];
        dot += k[m][j] * q[m][j];
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        kk += __shfl_xor(kk, o);
        qq += __shfl_xor(qq, o);
        dot += __shfl_xor(dot, o);
      }
      const float ki = 1.0f / sqrtf(kk + 1e-6f), qi = q_scale / sqrtf(qq + 1e-6f);
#pragma unroll
      for (int j = 0; j < kEach; ++j) {
        const int i = lane + 64 * j;
        if (i < kD) {
          ks[r][i] = k[m][j] * ki;
          qs[r][i] = q[m][j] * qi;
        }
      }
      if (lane == 0) {
        kq[r] = dot * ki * qi;
        beta[r] = sigmoid_f(bv[m]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kTok; ++r) {
      if (r >= rows) break;
      float rec = 0.f, read = 0.f;
#pragma unroll
      for (int i = 0; i < NI; i += 4) {
        const float4 g4 = *reinterpret_cast<const float4*>(&gs[r][rw * NI + i]);
        const float4 k4 = *reinterpret_cast<const float4*>(&ks[r][rw * NI + i]);
        const float4 q4 = *reinterpret_cast<const float4*>(&qs[r][rw * NI + i]);
        S[i] *= g4.x; rec += S[i] * k4.x; read += S[i] * q4.x;
        S[i + 1] *= g4.y; rec += S[i + 1] * k4.y; read += S[i + 1] * q4.y;
        S[i + 2] *= g4.z; rec += S[i + 2] * k4.z; read += S[i + 2] * q4.z;
        S[i + 3] *= g4.w; rec += S[i + 3] * k4.w; read += S[i + 3] * q4.w;
      }
      if constexpr (RW > 1) {
        part[r & 1][rw][cl] = make_float2(rec, read);
        __syncthreads();
        rec = read = 0.f;
#pragma unroll
        for (int w = 0; w < RW; ++w) {
          const float2 x = part[r & 1][w][cl];
          rec += x.x;
          read += x.y;
        }
      }
      const float u = beta[r] * (v[r] - rec);
      if (rw == 0) os[r][cl] = read + kq[r] * u;
#pragma unroll
      for (int i = 0; i < NI; i += 4) {
        const float4 k4 = *reinterpret_cast<const float4*>(&ks[r][rw * NI + i]);
        S[i] += k4.x * u;
        S[i + 1] += k4.y * u;
        S[i + 2] += k4.z * u;
        S[i + 3] += k4.w * u;
      }
    }
    __syncthreads();
    if (whole && n_tok == 1) {                           // decoding: every thread of the first row share finishes its column
      float ssq = 0.f;
#pragma unroll
      for (int c = lane; c < kCols; c += 64) ssq += c < a.E ? os[0][c] * os[0][c] : 0.f;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) ssq += __shfl_xor(ssq, o);
      if (rw == 0 && live)
        static_cast<T*>(a.out)[((int64_t)lo * a.H + head) * a.E + col] =
            from_f32<T>(os[0][cl] * (1.0f / sqrtf(ssq / (float)a.E + a.eps)) * out_w * sigmoid_f(gate0));
    } else {
      for (int r = wave; r < rows; r += kWaves) {        // outputs, a wavefront per token
        const int64_t row = lo + t0 + r;
        T* dst = static_cast<T*>(a.out) + (row * a.H + head) * a.E + col0;
        float inv = 1.f;
        if (whole) {
          float ssq = 0.f;
#pragma unroll
          for (int c = lane; c < kCols; c += 64) ssq += c < a.E ? os[r][c] * os[r][c] : 0.f;
#pragma unroll
          for (int o = 32; o > 0; o >>= 1) ssq += __shfl_xor(ssq, o);
          inv = 1.0f / sqrtf(ssq / (float)a.E + a.eps);
        }
        const T* gate = gp + (int64_t)(t0 + r) * a.gate_stride;
#pragma unroll
        for (int c = lane; c < kCols; c += 64) {
          if (col0 + c >= a.E) break;
          float y = os[r][c];
          if (whole) y *= inv * a.norm[c] * sigmoid_f(to_f32<T>(gate[c]));
          dst[c] = from_f32<T>(y);
        }
      }
    }
    // (the next stage's first barrier stands between these reads of `os` and its being written again)
  }
#pragma unroll
  for (int i = 0; i < NI; ++i)
    if (live && rw * NI + i < a.D) st[(int64_t)i * a.E] = S[i];
}

// ---- One token a sequence, the decays' and the gate's operands through a low rank whose second product is formed here.
//
// A workgroup owns (sequence, head).  What it reads is cold, the state and the head's D + E weight rows 3 us away, and everything else is a
// chain of a few sums: what bounds it is how soon all of that is requested, so no load stands in a branch (what lies outside a buffer reads
// zero) or waits for more than the slot's number, and the code is one token's.  As the scan above with the low rank in front of it, unrolled
// for eight tokens, 3400 cycles lay between its first request and the state's.  us, so and now: 1 / 16 sequences of 16 heads of 64 x 128, rank
// 64, 10.6 / 13.2 and 6.3 / 8.4; 1 / 8 of 32 heads of 128 x 128, rank 128, 13.2 / 19.0 and 8.1 / 12.0 (twice the wavefronts, 16 rows each, 8.4 /
// 12.0).  Whole steps with the low rank's product a launch of its own and here: 16 sequences 478 and 464 (4b), 242 and 221 (1b), 4 412 and 389.
template <int kCtrl>
__device__ __forceinline__ float add_moved(float v) {
  return v + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), kCtrl, 0xf, 0xf, false));
}
// The sum over sixteen lanes, and over a wavefront, in every lane.
__device__ __forceinline__ float row_sum(float v) { return add_moved<0x140>(add_moved<0x141>(add_moved<0x4E>(add_moved<0xB1>(v)))); }
__device__ __forceinline__ float wave_sum(float v) { return lanes_sum(row_sum(v)); }
// One 16-byte chunk's products of a weight row and its operand.
__device__ __forceinline__ float dot8(const u32x4_t& w, const u32x4_t& x, float s) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    s += bf16lo(w[i]) * bf16lo(x[i]);
    s += bf16hi(w[i]) * bf16hi(x[i]);
  }
  return s;
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t bytes_rsrc(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
__device__ __forceinline__ float load_bf16(__amdgpu_buffer_rsrc_t rs, int at) { return bf16_to_f32(__builtin_amdgcn_raw_buffer_load_b16(rs, at, 0, 0)); }
__device__ __forceinline__ float load_f32(__amdgpu_buffer_rsrc_t rs, int at) { return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, at, 0, 0)); }

// NI state rows a thread, RW wavefronts' shares of the rows, CW wavefronts of 64 value columns.
template <int NI, int RW, int CW>
__global__ __launch_bounds__(RW * CW * 64) void delta_step_kernel(msa_delta_args a, msa_seq_batch b, msa_delta_low low) {
  constexpr int kD = NI * RW, kCols = CW * 64, kRows = RW * CW * 4;                       // kRows: weight rows at a time, sixteen lanes each
  constexpr int kEach = (kD + 63) / 64, kTurnsA = (kD + kRows - 1) / kRows, kTurnsG = (kCols + kRows - 1) / kRows;
  __shared__ __align__(16) float ks[kD], qs[kD], gs[kD];
  __shared__ float low_out[kD + kCols], beta_kq[2];
  __shared__ float2 part[RW][kCols];
  const int head = blockIdx.x, s = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), cw = wave % CW, rw = wave / CW, col = cw * 64 + lane;
  // (as many rows as sequences, none with more than one: nothing to look up in front of the first loads)
  const bool dense = b.rows == b.n_seq;
  const int row = dense ? s : b.cu[s], kvh = head / (a.H / a.G);
  if (!dense && b.cu[s + 1] == row) return;
  const int slot = b.slot[s];
  float* const st = a.state + ((int64_t)slot * a.H + head) * a.D * a.E;
  const bf16_t* const qkv = static_cast<const bf16_t*>(a.qkv) + row * a.qkv_stride;

  const __amdgpu_buffer_rsrc_t rs_w = bytes_rsrc(static_cast<const bf16_t*>(low.w) + (int64_t)head * a.D * low.rank, a.D * low.rank * 2);
  const __amdgpu_buffer_rsrc_t rs_g = bytes_rsrc(static_cast<const bf16_t*>(low.w) + (low.n_a + (int64_t)head * a.E) * low.rank, a.E * low.rank * 2);
  const __amdgpu_buffer_rsrc_t rs_xa = bytes_rsrc(static_cast<const bf16_t*>(low.a_low) + row * low.a_stride, low.rank * 2);
  const __amdgpu_buffer_rsrc_t rs_xg = bytes_rsrc(static_cast<const bf16_t*>(low.g_low) + row * low.g_stride, low.rank * 2);
  u32x4_t wa[kTurnsA], wg[kTurnsG], xa, xg;
  auto fetch_low = [&](int unit) {
    // (a row's end, not the next row; rows behind the head's own by the vector offset, which is what the range check compares)
    const int at = unit * 8 < low.rank ? (tid >> 4) * low.rank * 2 + unit * 16 : kOutside, turn = kRows * low.rank * 2;
    xa = __builtin_amdgcn_raw_buffer_load_b128(rs_xa, unit * 16, 0, 0);
    xg = __builtin_amdgcn_raw_buffer_load_b128(rs_xg, unit * 16, 0, 0);
#pragma unroll
    for (int i = 0; i < kTurnsA; ++i) wa[i] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, at + i * turn, 0, 0);
#pragma unroll
    for (int i = 0; i < kTurnsG; ++i) wg[i] = __builtin_amdgcn_raw_buffer_load_b128(rs_g, at + i * turn, 0, 0);
  };
  // ---- everything is requested, once the slot and all arguments are there (else they are waits in between)
  asm volatile("" ::"s"(slot));
  __builtin_amdgcn_sched_barrier(0);
  float k[kEach], q[kEach], bias = 0.f;
  const __amdgpu_buffer_rsrc_t rs_q = bytes_rsrc(qkv + (int64_t)kvh * a.D, a.D * 2), rs_k = bytes_rsrc(qkv + (int64_t)(a.G + kvh) * a.D, a.D * 2);
#pragma unroll
  for (int j = 0; j < kEach; ++j) {                        // (every wavefront: cheaper than a branch)
    k[j] = load_bf16(rs_k, (lane + 64 * j) * 2);
    q[j] = load_bf16(rs_q, (lane + 64 * j) * 2);
  }
  const float v = load_bf16(bytes_rsrc(qkv + 2LL * a.G * a.D + (int64_t)head * a.E, a.E * 2), col * 2);
  const float bv = load_bf16(bytes_rsrc(static_cast<const bf16_t*>(a.b) + row * a.b_stride + head, 2), 0);
  fetch_low(tid & 15);
  bias = load_f32(bytes_rsrc(a.dt_bias + (int64_t)head * a.D, a.D * 4), tid * 4);
  const float out_w = load_f32(bytes_rsrc(a.norm, a.E * 4), col * 4);
  const __amdgpu_buffer_rsrc_t rs_s = bytes_rsrc(st, a.D * a.E * 4);
  const int s_at = col < a.E ? (rw * NI * a.E + col) * 4 : kOutside;
  float S[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) S[i] = load_f32(rs_s, s_at + i * a.E * 4);
  __builtin_amdgcn_sched_barrier(0);
  const float rate = -expf(a.A_log[head]);

  // ---- unit vectors, and the low rank's second product
  if (wave == 0) {
    float kk = 0.f, qq = 0.f, dot = 0.f;
#pragma unroll
    for (int j = 0; j < kEach; ++j) {
      kk += k[j] * k[j];
      qq += q[j] * q[j];
      dot += k[j] * q[j];
    }
    const float ki = 1.0f / sqrtf(wave_sum(kk) + 1e-6f), qi = 1.0f / (sqrtf((float)a.D) * sqrtf(wave_sum(qq) + 1e-6f));
    dot = wave_sum(dot);
#pragma unroll
    for (int j = 0; j < kEach; ++j) {
      const int i = lane + 64 * j;
      if (i < kD) {
        ks[i] = k[j] * ki;
        qs[i] = q[j] * qi;
      }
    }
    if (lane == 0) {
      beta_kq[0] = sigmoid_f(bv);
      beta_kq[1] = dot * ki * qi;
    }
  }
  float sum[kTurnsA + kTurnsG] = {};
  for (int u0 = 0;;) {
#pragma unroll
    for (int i = 0; i < kTurnsA; ++i) sum[i] = dot8(wa[i], xa, sum[i]);
#pragma unroll
    for (int i = 0; i < kTurnsG; ++i) sum[kTurnsA + i] = dot8(wg[i], xg, sum[kTurnsA + i]);
    if ((u0 += 16) >= low.rank / 8) break;
    fetch_low(u0 + (tid & 15));
  }
#pragma unroll
  for (int i = 0; i < kTurnsA + kTurnsG; ++i) {
    const float x = row_sum(sum[i]);
    const int r = (i < kTurnsA ? i : i - kTurnsA) * kRows + (tid >> 4);
    if ((tid & 15) == 0 && r < (i < kTurnsA ? kD : kCols)) low_out[(i < kTurnsA ? 0 : kD) + r] = x;
  }
  __syncthreads();
  if (tid < kD) gs[tid] = tid < a.D ? expf(rate * softplus_f(low_out[tid] + bias)) : 0.f;
  __syncthreads();

  // ---- the rule
  float rec = 0.f, read = 0.f;
#pragma unroll
  for (int i = 0; i < NI; i += 4) {
    const float4 g4 = *reinterpret_cast<const float4*>(&gs[rw * NI + i]);
    const float4 k4 = *reinterpret_cast<const float4*>(&ks[rw * NI + i]);
    const float4 q4 = *reinterpret_cast<const float4*>(&qs[rw * NI + i]);
    S[i] *= g4.x; rec += S[i] * k4.x; read += S[i] * q4.x;
    S[i + 1] *= g4.y; rec += S[i + 1] * k4.y; read += S[i + 1] * q4.y;
    S[i + 2] *= g4.z; rec += S[i + 2] * k4.z; read += S[i + 2] * q4.z;
    S[i + 3] *= g4.w; rec += S[i + 3] * k4.w; read += S[i + 3] * q4.w;
  }
  part[rw][col] = make_float2(rec, read);
  __syncthreads();
  rec = read = 0.f;
#pragma unroll
  for (int w = 0; w < RW; ++w) {
    const float2 x = part[w][col];
    rec += x.x;
    read += x.y;
  }
  const float beta = beta_kq[0], kq = beta_kq[1], u = beta * (v - rec), o = read + kq * u;
#pragma unroll
  for (int i = 0; i < NI; i += 4) {
    const float4 k4 = *reinterpret_cast<const float4*>(&ks[rw * NI + i]);
    S[i] += k4.x * u;
    S[i + 1] += k4.y * u;
    S[i + 2] += k4.z * u;
    S[i + 3] += k4.w * u;
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(S[i]), rs_s, s_at + i * a.E * 4, 0, 0);

  // ---- norm and gate of the output: the columns' sums of squares by the first share's wavefronts
  __shared__ float squares[CW];
  const float ssq = wave_sum(col < a.E ? o * o : 0.f);
  if (CW > 1) {
    if (rw == 0 && lane == 0) squares[cw] = ssq;
    __syncthreads();
  }
  if (rw == 0 && col < a.E) {
    float total = ssq;
    if (CW > 1) {
      total = squares[0];
#pragma unroll
      for (int w = 1; w < CW; ++w) total += squares[w];
    }
    static_cast<bf16_t*>(a.out)[((int64_t)row * a.H + head) * a.E + col] =
        f32_to_bf16(o * (1.0f / sqrtf(total / (float)a.E + a.eps)) * out_w * sigmoid_f(low_out[kD + col]));
  }
}

// Value columns of a workgroup.
int column_block(int32_t D, int32_t E) { return E <= 64 || D > 256 ? 64 : 128; }

template <typename T, int NI, int RW>
void launch_scan(const msa_delta_args& a, const msa_seq_batch& b, hipStream_t st) {
  const int cols = column_block(a.D, a.E);
  const dim3 grid((a.E + cols - 1) / cols, a.H, b.n_seq);
  if (cols == 64) delta_scan_kernel<T, NI, RW, 1><<<grid, RW * 64, 0, st>>>(a, b);
  else if constexpr (NI * RW <= 256) delta_scan_kernel<T, NI, RW, 2><<<grid, RW * 128, 0, st>>>(a, b);
}

template <typename T>
int launch_scan(const msa_delta_args& a, const msa_seq_batch& b, hipStream_t st) {
  if (a.D <= 16) launch_scan<T, 4, 4>(a, b, st);
  else if (a.D <= 32) launch_scan<T, 8, 4>(a, b, st);
  else if (a.D <= 64) launch_scan<T, 16, 4>(a, b, st);
  else if (a.D <= 128 && (int64_t)a.H * b.n_seq <= device_compute_units() / 2) launch_scan<T, 16, 8>(a, b, st);    // (twice the wavefronts when compute units are free)
  else if (a.D <= 128) launch_scan<T, 32, 4>(a, b, st);
  else if (a.D <= 256) launch_scan<T, 32, 8>(a, b, st);
  else launch_scan<T, 64, 8>(a, b, st);
  MSA_LAUNCH_CHECK();
  return MSA_OK;
}

template <int NI, int RW>
void launch_step(const msa_delta_args& a, const msa_delta_low& low, const msa_seq_batch& b, hipStream_t st) {
  const dim3 grid(a.H, b.n_seq);
  if (a.E <= 64) delta_step_kernel<NI, RW, 1><<<grid, RW * 64, 0, st>>>(a, b, low);
  else delta_step_kernel<NI, RW, 2><<<grid, RW * 128, 0, st>>>(a, b, low);
}

}  // namespace

extern "C" int msa_seq_delta_step(const msa_delta_args* args, const msa_delta_low* low, const msa_seq_batch* batch, void* stream) {
  MSA_CHECK_BATCH(batch, "msa_seq_delta_step");
  MSA_REQUIRE(args && low && args->qkv && args->b && args->A_log && args->dt_bias && args->norm && args->state && args->out && low->a_low &&
                  low->g_low && low->w, "msa_seq_delta_step: null pointer");
  const msa_delta_args& a = *args;
  MSA_REQUIRE(batch->max_rows == 1, "msa_seq_delta_step: one token a sequence, got %d", batch->max_rows);
  MSA_REQUIRE(a.H > 0 && a.H <= 65535 && a.G > 0 && a.H % a.G == 0 && a.D > 0 && a.D <= 128 && a.E > 0 && a.E <= 128 && batch->n_seq <= 65535,
              "msa_seq_delta_step: H=%d G=%d D=%d E=%d (both up to 128)", a.H, a.G, a.D, a.E);
  MSA_REQUIRE(a.qkv_stride >= 2LL * a.G * a.D + (int64_t)a.H * a.E && a.b_stride >= a.H, "msa_seq_delta_step: strides");
  MSA_REQUIRE(low->rank > 0 && low->rank % 8 == 0 && low->a_stride >= low->rank && low->g_stride >= low->rank && low->a_stride % 8 == 0 &&
                  low->g_stride % 8 == 0 && low->n_a >= a.H * a.D &&
                  (((uintptr_t)low->a_low | (uintptr_t)low->g_low | (uintptr_t)low->w) & 15) == 0,
              "msa_seq_delta_step: rank=%d (a multiple of 8, 16-byte aligned rows)", low->rank);
  hipStream_t st = as_stream(stream);
  if (a.D <= 16) launch_step<4, 4>(a, *low, *batch, st);
  else if (a.D <= 32) launch_step<8, 4>(a, *low, *batch, st);
  else if (a.D <= 64) launch_step<8, 8>(a, *low, *batch, st);
  else launch_step<32, 4>(a, *low, *batch, st);
  MSA_LAUNCH_CHECK();
  return MSA_OK;
}

extern "C" int msa_seq_delta_scan(const msa_delta_args* args, int32_t dtype, const msa_seq_batch* batch, void* stream) {
  MSA_CHECK_BATCH(batch, "msa_seq_delta_scan");
  MSA_CHECK_DTYPE(dtype, "msa_seq_delta_scan");
  MSA_REQUIRE(args && args->qkv && args->a && args->b && args->gate && args->A_log && args->dt_bias && args->norm && args->state && args->out,
              "msa_seq_delta_scan: null pointer");
  const msa_delta_args& a = *args;
  MSA_REQUIRE(a.H > 0 && a.H <= 65535 && a.G > 0 && a.H % a.G == 0 && a.D > 0 && a.D <= 512 && a.E > 0 && batch->n_seq <= 65535,
              "msa_seq_delta_scan: H=%d G=%d D=%d (up to 512) E=%d", a.H, a.G, a.D, a.E);
  MSA_REQUIRE(a.qkv_stride >= 2LL * a.G * a.D + (int64_t)a.H * a.E && a.a_stride >= (int64_t)a.H * a.D && a.b_stride >= a.H &&
                  a.gate_stride >= (int64_t)a.H * a.E, "msa_seq_delta_scan: strides");
  hipStream_t st = as_stream(stream);
  const int rc = dtype == MSA_BF16 ? launch_scan<bf16_t>(a, *batch, st) : launch_scan<float>(a, *batch, st);
  if (rc != MSA_OK || a.E <= column_block(a.D, a.E)) return rc;
  return msa_seq_head_norm_gate(a.out, a.gate, a.gate_stride, a.norm, a.eps, dtype, batch->rows, a.H, a.E, stream);
}
