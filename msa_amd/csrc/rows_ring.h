// Weight-streaming product of up to 16 bf16 rows, y[m, n] = x[m, :K] . w[n, :K]: the decode steps' matrices, read from HBM
// exactly once, which is the whole cost.
//
// One workgroup of 16 wavefronts per compute unit stays for the whole launch and owns a contiguous range of weight rows (equal
// shares of all rows), taken 16 at a time.  K is cut into units of 64 elements (128 bytes, a cache line) dealt round the
// wavefronts; a wavefront requests a unit of the 16 rows as two direct-to-LDS loads of eight whole lines each into a ring of
// two slots of its own, so no wavefront waits for another's data, and the next unit is always in flight.  The 16-byte pieces of a
// line are stored XORed with the row, which spreads the operand reads over the banks.  The 16 activation rows are one operand of
// the 16x16x32 MFMA and stay in registers up to K = 5120; longer rows pass the ring beside the weights, as whole lines.  The
// wavefronts' partial sums meet in LDS behind one barrier per 16 rows (two for long rows, whose ring leaves no room to take planes
// in turn) and are added in a fixed order.
//
// What bounds it is HBM where a workgroup has several rounds, and the launch, the first loads' latency and the activations (every
// workgroup reads all of them from its L2) where it has one.
//
// Why not through registers: an MFMA operand load touches 16 rows in 64-byte pieces, so a line is fetched by two instructions,
// and with non-temporal loads (10 % more bandwidth) even twice from memory.  Whole lines into LDS take non-temporal loads, and
// need no registers for what is in flight.  Measured in graphs over operands larger than the caches, launches included, against
// the register forms before, us with 1 / 16 rows: 151936 x 2560 fp32 out 120 / 131 against 154 / 177 (6.5 / 5.9 TB/s); 151936 x
// 1024 48 / 56 against 74 / 77; 19456 x 2560 gated units 17.6 / 18.9 against 23.8 / 26.5; 14944 x 2560 with convolution 15.3 /
// 18.0 against 20.5 / 25.8; 2560 x 4096 6.5 / 8.0 against 7.3 / 9.6; 4096 x 1024 4.0 / 4.3 against 4.1 / 4.7.  A
// third slot changes nothing, except with a folded norm, whose arithmetic it hides (6144 x 2560: 9.3 / 10.3 against 9.9 / 11.0 with
// two).  Long rows of activations held the weights up when they were loaded as the operand wants them (us with 1 / 4 / 16 rows, then and
// through the ring: 2560 x 9728 12.4 / 13.9 / 18.4 and 12.5 / 13.9 / 16.5, 5120 x 8192 19.9 / 20.7 / 27.2 and 20.3 / 20.3 / 21.9,
// 1024 x 9728 10.8 / 11.1 / 15.0 and 10.9 / 10.9 / 11.3; three or four slots of weights instead were 5 to 20 % slower).  An item of the loop must not wait for its own output's store or for what the epilogue reads.
#pragma once

#include "common.h"

namespace rows_ring {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4_t;
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kWaves = 16, kUnitBytes = 128, kUnitSlab = 16 * kUnitBytes;
constexpr int kPlane = 272;                        // floats between two wavefronts' partial blocks: four adders hit distinct banks
constexpr int kMaxResident = 5;                    // units per wavefront whose activations stay in registers
constexpr int kMaxResidentK = kMaxResident * kWaves * kUnitBytes / 2;
// The line between the two forms: small matrices are done within the launch's own time, rows of up to 512 elements leave half of the
// sixteen wavefronts without work, and so do some longer ones in their last round: what counts is the weights times the share of the
// wavefronts at work.  Each library's products have a line of their own.
constexpr int kMinK = 512, kMinRows = 4;
static inline int64_t busy_weights(int64_t N, int64_t K) {
  const int64_t units = (K * 2 + kUnitBytes - 1) / kUnitBytes, rounds = (units + kWaves - 1) / kWaves;
  return N * K * units / (rounds * kWaves);
}
constexpr int kFar = 0x7ff00000;                   // past every extent, whatever is added: reads zeros, touches no memory
// What happens to the activations in front of the products: nothing, an RMSNorm, or a residual step with the norm of its own (one
// launch less, but all workgroups read its fp32 operands: seq_rows.hip has the line), or that and the norm behind it (the head);
// or they are rows of an embedding table, found by their tokens.
enum { kPlain, kNormed, kPost, kFinal, kEmbed };
constexpr int kMaxPost = 3;                        // units per wavefront that the residual step takes: what its registers hold
constexpr int slots(int pro) { return pro ? 3 : 2; }              // of a wavefront's ring
// Rows too long for the registers (nu = 0): the activations' unit lies behind the weights' in its slot, and there is room for one plane
// of partial sums instead of two in turn.
constexpr int planes(int nu) { return nu == 0 ? 1 : 2; }
constexpr int slab(int nu) { return nu == 0 ? 2 * kUnitSlab : kUnitSlab; }
constexpr int lds_bytes(int pro, int nu) {
  return planes(nu) * kWaves * kPlane * 4 + kWaves * slots(pro) * slab(nu) + (pro == kFinal ? 2 : pro == kPlain || pro == kEmbed ? 0 : 1) * kWaves * 16 * 4;
}
static_assert(kMaxPost * 2 * kUnitBytes <= 1024 && kMaxResident * kUnitBytes <= 1024, "one request for a wavefront's part of the norm's weights");
static_assert(kPlane * 4 >= 1024 && kPlane % 4 == 0, "which lies where the wavefront's first partial sums will");
static_assert(lds_bytes(kNormed, 1) <= 160 * 1024 && lds_bytes(kPlain, 0) <= 160 * 1024 && lds_bytes(kFinal, 1) <= 160 * 1024);
constexpr int kNonTemporal = 2;                    // a step reads a weight once

// vmcnt(n), the other counters not waited for
constexpr int wait_vm(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

// the value of the lane 1 (0xB1) or 2 (0x4E) away in the group of four
template <int kPerm>
__device__ __forceinline__ float quad_xor(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), kPerm, 0xf, 0xf, false));
}

__device__ __forceinline__ uint32_t lds_offset(const void* p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p; }
__device__ __forceinline__ u32x4_t lds_read16(uint32_t at) {
  u32x4_t v;
  asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(v) : "v"(at) : "memory");
  return v;
}

struct Args {
  const char *w, *x, *x_b, *norm_w;
  const float *post_x, *post_w;                    // kPost: the operand is post_x + rms_norm(x) * post_w, which one workgroup
  float* post_out;                                 // leaves in post_out (rows of K); kFinal: rms_norm(that) * post_next
  const float* post_next;
  const int64_t* tokens;                           // kEmbed: the operand's row m is row tokens[m] of x (vocab rows of row_bytes); also left in post_out
  int64_t vocab;
  int64_t xs, xbs;                                 // bytes between activation rows
  int32_t M, N, n_b, row_bytes;                    // weight rows from n_b on multiply x_b
  int32_t wgs_a, granule, qa, ra, qb, rb;  // workgroup i < wgs_a: its share of the granules of the rows before n_b
  float eps;
};

// Epi: `begin(s, m)` first of all (m, the wavefront's output row, is uniform), `load(s, m, n, mine, second, item)` before an
// item's products, `apply(s, m, n, v, mine, second, item)` behind them, in every lane: four neighbouring lanes hold output
// (m, n), neighbouring columns are four lanes apart, `mine` in the first lane of each output that exists.  `load` must not wait
// for what it requests: loads return in order, so that would wait for the weights in front of it.
template <class Epi, int NU, int kPro>
__global__ __launch_bounds__(kWaves * 64) void rows_ring_kernel(Args a, typename Epi::Args s) {
  constexpr bool kResident = NU > 0, kNorm = kPro == kNormed, kPosts = kPro == kPost || kPro == kFinal;
  constexpr int kSlots = slots(kPro), kPlanes = planes(NU), kSlab = slab(NU);
  extern __shared__ __align__(16) char lds[];
  float(*part)[kWaves][kPlane] = reinterpret_cast<float(*)[kWaves][kPlane]>(lds);
  float* row_ssq = reinterpret_cast<float*>(lds + kPlanes * kWaves * kPlane * 4 + kWaves * kSlots * kSlab);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  char* ring = lds + kPlanes * kWaves * kPlane * 4 + wave * kSlots * kSlab;
  const int wg = blockIdx.x, n_l = lane & 15, g = lane >> 4;
  const bool second = wg >= a.wgs_a;
  const int i = second ? wg - a.wgs_a : wg, q = second ? a.qb : a.qa, rem = second ? a.rb : a.ra;
  const int gran = second ? 1 : a.granule, first = i * q + min(i, rem), end = second ? a.N : min(a.n_b, a.N);
  const int r0 = (second ? a.n_b : 0) + first * gran, r1 = min(end, r0 + (q + (i < rem)) * gran);
  const int items = (r1 - r0 + 15) >> 4;
  const int row_bytes = a.row_bytes, units = (row_bytes + kUnitBytes * kWaves - 1) / (kUnitBytes * kWaves);

  const int m = wave, quarter = lane & 3, nr = lane >> 2, at = (m & 3) * 64 + (m >> 2) * 16 + nr;      // this thread's output
  Epi epi;
  epi.begin(s, m);

  // ---- requests: unit u of the rows from `base` on, into the next slot
  const int l_row = lane >> 3, col = wave * kUnitBytes + ((lane & 7) ^ (l_row & 7)) * 16;
  const int off0 = l_row * row_bytes + col, off1 = off0 + 8 * row_bytes;
  const int64_t xs = second ? a.xbs : a.xs;
  const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(second ? a.x_b : a.x), 0,
                                                                        (int)(kPro == kEmbed ? a.vocab * row_bytes : (a.M - 1) * xs + row_bytes), 0x00020000);
  const int xoff0 = l_row * (int)xs + col, xoff1 = xoff0 + 8 * (int)xs;      // of the activations, likewise
  int req_item = 0, slot_in = 0;
  __amdgpu_buffer_rsrc_t rs;
  auto point = [&]() {
    // (the clamp compiles to a vector instruction: the extent has to come back into a scalar register, or every load gets a loop
    // over descriptors)
    const int base = r0 + 16 * req_item, rows = __builtin_amdgcn_readfirstlane(max(0, min(16, r1 - base)));
    rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.w) + (int64_t)(rows > 0 ? base : r0) * row_bytes, 0, rows * row_bytes, 0x00020000);
  };
  auto request = [&](int u) {
    const int so = u * (kUnitBytes * kWaves);
    char* dst = ring + slot_in * kSlab;
    int v0 = off0, v1 = off1, x0 = xoff0, x1 = xoff1;
    if (so + kUnitBytes * kWaves > row_bytes) {    // a row's last units can leave it
      const bool in = col + so < row_bytes;
      v0 = in ? off0 : kFar;
      v1 = in ? off1 : kFar;
      x0 = in ? xoff0 : kFar;
      x1 = in ? xoff1 : kFar;
    }
    MSA_LOAD_TO_LDS(rs, dst, v0, so, kNonTemporal);
    MSA_LOAD_TO_LDS(rs, dst + kUnitSlab / 2, v1, so, kNonTemporal);
    if constexpr (!kResident) {
      MSA_LOAD_TO_LDS(rs_x, dst + kUnitSlab, x0, so, 0);
      MSA_LOAD_TO_LDS(rs_x, dst + kUnitSlab * 3 / 2, x1, so, 0);
    }
    slot_in = slot_in + 1 == kSlots ? 0 : slot_in + 1;
  };
  const int x_col = wave * kUnitBytes + g * 16;
  const int x_row = kPro == kEmbed ? (int)embed_row(a.tokens[min(n_l, a.M - 1)], a.vocab, true) * row_bytes : n_l * (int)xs;
  auto load_x = [&](u32x4_t (&x)[2], int u) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int so = u * (kUnitBytes * kWaves) + h * 64;
      x[h] = __builtin_amdgcn_raw_buffer_load_b128(rs_x, x_col + so < row_bytes ? x_row + x_col : kFar, so, 0);
    }
  };
  const int rd0 = n_l * kUnitBytes + ((g ^ (n_l & 7)) * 16), rd1 = n_l * kUnitBytes + (((g + 4) ^ (n_l & 7)) * 16);
  int slot_out = 0;
  auto multiply = [&](u32x4_t (&x)[2], floatx4_t acc) {
    const char* src = ring + slot_out * kSlab;
    const u32x4_t w0 = *reinterpret_cast<const u32x4_t*>(src + rd0), w1 = *reinterpret_cast<const u32x4_t*>(src + rd1);
    if constexpr (!kResident) {
      x[0] = *reinterpret_cast<const u32x4_t*>(src + kUnitSlab + rd0);
      x[1] = *reinterpret_cast<const u32x4_t*>(src + kUnitSlab + rd1);
    }
    slot_out = slot_out + 1 == kSlots ? 0 : slot_out + 1;
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, x[0]), __builtin_bit_cast(bf16x8_t, w0), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, x[1]), __builtin_bit_cast(bf16x8_t, w1), acc, 0, 0, 0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the slot may be requested again
    return acc;
  };

  // The ring is filled ahead of the loop, in front of which only the activations are waited for (a register the compiler
  // believes outstanding there would be waited for, with everything behind it, in every round).
  const int rounds = kResident ? NU : (units + kSlots - 1) / kSlots * kSlots;      // (units behind a row's last read zeros)
  constexpr int kX = kResident ? NU : kSlots;
  u32x4_t xf[kX][2];
  if constexpr (kResident) {
#pragma unroll
    for (int u = 0; u < NU; ++u) load_x(xf[u], u);
  }
  // The norm's weights, alike for all rows, through LDS (in registers, five units of them spill: 2560 x 5120 with one row took 13.9
  // us instead of 8.8): where the wavefront's own partial sums will lie, which it writes behind its reads
  char *norm_lds = reinterpret_cast<char*>(part[0][wave]), *next_lds = reinterpret_cast<char*>(part[kPlanes - 1][wave]);
  if constexpr (kNorm) {
    const __amdgpu_buffer_rsrc_t rs_g = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.norm_w), 0, row_bytes, 0x00020000);
    MSA_LOAD_TO_LDS(rs_g, norm_lds, (lane >> 3) * (kUnitBytes * kWaves) + wave * kUnitBytes + (lane & 7) * 16, 0, 0);
  }
  // The residual step's other operands: the fp32 rows into registers, the weights likewise
  u32x4_t px[kPosts ? NU : 1][2][2];
  if constexpr (kPosts) {
    const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.post_w), 0, 2 * row_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rs_p = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.post_x), 0, a.M * 2 * row_bytes, 0x00020000);
    MSA_LOAD_TO_LDS(rs_w, norm_lds, (lane >> 4) * (2 * kUnitBytes * kWaves) + wave * 2 * kUnitBytes + (lane & 15) * 16, 0, 0);
    if constexpr (kPro == kFinal) {
      const __amdgpu_buffer_rsrc_t rs_n = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.post_next), 0, 2 * row_bytes, 0x00020000);
      MSA_LOAD_TO_LDS(rs_n, next_lds, (lane >> 4) * (2 * kUnitBytes * kWaves) + wave * 2 * kUnitBytes + (lane & 15) * 16, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int so = u * (kUnitBytes * kWaves) + h * 64, at = x_col + so < row_bytes ? n_l * 2 * row_bytes + 2 * x_col : kFar;
#pragma unroll
        for (int i = 0; i < 2; ++i) px[u][h][i] = __builtin_amdgcn_raw_buffer_load_b128(rs_p, at + 16 * i, 2 * so, 0);
      }
  }
  constexpr bool kLate = kPosts && NU == kMaxPost;    // (no registers for it in front of the residual step)
  if (!kLate) epi.load(s, m, r0 + nr, quarter == 0 && m < a.M && r0 + nr < r1, second, 0);
  asm volatile("" ::: "memory");                             // (not to be sunk behind the requests)
  point();
#pragma unroll
  for (int i = 0; i < kSlots; ++i) {
    if (kResident && i > 0 && i % kX == 0) {
      ++req_item;
      point();
    }
    request(i % kX);
  }
  __builtin_amdgcn_sched_barrier(0);                         // (nothing is computed before everything is requested)
  // What a norm reads of LDS it reads by hand: the compiler would wait for the ring in front of it, and nor does it wait for the
  // weights: what the ring has requested by now, 2 kSlots loads, is all that may be outstanding then.  The build checks that.
  if constexpr (kNorm) {
    // RMSNorm folded in: the operand is bf16(x * norm_w); the row's factor commutes with the product and joins at the end
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kSlots) : "memory");
    float ssq = 0.f;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      u32x4_t gw[2];
      asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:64\n\ts_waitcnt lgkmcnt(0)"
                   : "=&v"(gw[0]), "=&v"(gw[1]) : "v"(lds_offset(norm_lds) + u * kUnitBytes + g * 16) : "memory");
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float lo = bf16lo(xf[u][h][c]), hi = bf16hi(xf[u][h][c]);
          ssq += lo * lo + hi * hi;
          xf[u][h][c] = pack_bf16x2(lo * bf16lo(gw[h][c]), hi * bf16hi(gw[h][c]));
        }
      asm volatile("" : "+v"(xf[u][0]), "+v"(xf[u][1]), "+v"(ssq));      // (one unit unpacked at a time)
    }
    ssq = lanes_sum(ssq);
    if (g == 0) row_ssq[wave * 16 + n_l] = ssq;              // read behind the first barrier
  }
  if constexpr (kPro == kEmbed) {                            // (each row by one workgroup)
    const bool writes = n_l < a.M && n_l % gridDim.x == wg;
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int at = x_col + u * (kUnitBytes * kWaves) + h * 64;
        if (!writes || at >= row_bytes) continue;
        float4* to = reinterpret_cast<float4*>(a.post_out + (int64_t)n_l * (row_bytes / 2) + at / 2);
        to[0] = make_float4(bf16lo(xf[u][h][0]), bf16hi(xf[u][h][0]), bf16lo(xf[u][h][1]), bf16hi(xf[u][h][1]));
        to[1] = make_float4(bf16lo(xf[u][h][2]), bf16hi(xf[u][h][2]), bf16lo(xf[u][h][3]), bf16hi(xf[u][h][3]));
      }
  }
  if constexpr (kPosts) {
    // x + rms_norm(y) * w as the operand, the sums as in the launch of its own
    float ssq = 0.f;
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float lo = bf16lo(xf[u][h][c]), hi = bf16hi(xf[u][h][c]);
          ssq += lo * lo + hi * hi;
        }
    ssq = lanes_sum(ssq);
    const uint32_t row_at = lds_offset(row_ssq + n_l * 16);
    auto row_total = [&](uint32_t row_at) {
      u32x4_t p[4];
      if constexpr (NU < kMaxPost)
        asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:16\n\tds_read_b128 %2, %4 offset:32\n\tds_read_b128 %3, %4 offset:48\n\t"
                     "s_waitcnt lgkmcnt(0)" : "=&v"(p[0]), "=&v"(p[1]), "=&v"(p[2]), "=&v"(p[3]) : "v"(row_at) : "memory");
      float total = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (NU == kMaxPost) p[i] = lds_read16(row_at + 16 * i);                  // (no registers for all of them)
        total += (__uint_as_float(p[i][0]) + __uint_as_float(p[i][1])) + (__uint_as_float(p[i][2]) + __uint_as_float(p[i][3]));
      }
      return 1.0f / sqrtf(total / (float)(row_bytes / 2) + a.eps);
    };
    if constexpr (kPro == kFinal) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kSlots) : "memory");      // (the second weights' wait as well)
    asm volatile("ds_write_b32 %0, %1\n\ts_waitcnt vmcnt(%2) lgkmcnt(0)\n\ts_barrier" ::"v"(row_at + 4 * wave), "v"(ssq), "n"(2 * kSlots) : "memory");
    const float post_inv = row_total(row_at);
    float next_ssq = 0.f;
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int so = u * (kUnitBytes * kWaves) + h * 64;
        float v[8];
        u32x4_t w[2];
        const uint32_t w_at = lds_offset(norm_lds) + u * 2 * kUnitBytes + h * 128 + g * 32;
        if constexpr (NU < kMaxPost)
          asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:16\n\ts_waitcnt lgkmcnt(0)" : "=&v"(w[0]), "=&v"(w[1]) : "v"(w_at) : "memory");
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          if constexpr (NU == kMaxPost) w[i] = lds_read16(w_at + 16 * i);
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const uint32_t y = xf[u][h][2 * i + (c >> 1)];
            v[4 * i + c] = __uint_as_float(px[u][h][i][c]) + (c & 1 ? bf16hi(y) : bf16lo(y)) * post_inv * __uint_as_float(w[i][c]);
          }
        }
        if constexpr (kPro == kFinal) {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            next_ssq += v[e] * v[e];
            px[u][h][e >> 2][e & 3] = __float_as_uint(v[e]);
          }
          continue;
        }
        if (wg == 0 && n_l < a.M && x_col + so < row_bytes) {
          float4* to = reinterpret_cast<float4*>(a.post_out + (int64_t)n_l * (row_bytes / 2) + (x_col + so) / 2);
          to[0] = make_float4(v[0], v[1], v[2], v[3]);
          to[1] = make_float4(v[4], v[5], v[6], v[7]);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) xf[u][h][c] = pack_bf16x2(v[2 * c], v[2 * c + 1]);
      }
    if constexpr (kPro == kFinal) {
      next_ssq = lanes_sum(next_ssq);
      const uint32_t next_at = row_at + kWaves * 16 * 4;
      asm volatile("ds_write_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::"v"(next_at + 4 * wave), "v"(next_ssq) : "memory");
      const float next_inv = row_total(next_at);
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const u32x4_t w = lds_read16(lds_offset(next_lds) + u * 2 * kUnitBytes + h * 128 + g * 32 + 16 * i);
            float v[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = __uint_as_float(px[u][h][i][c]) * next_inv * __uint_as_float(w[c]);
            xf[u][h][2 * i] = pack_bf16x2(v[0], v[1]);
            xf[u][h][2 * i + 1] = pack_bf16x2(v[2], v[3]);
          }
    }
  }

  float inv = 1.f;
  if constexpr (kResident) {
#pragma unroll
    for (int u = 0; u < NU; ++u) asm volatile("" : "+v"(xf[u][0]), "+v"(xf[u][1]));
  }
  for (int item = 0; item < items; ++item) {
    const int n = r0 + 16 * item + nr;
    const bool mine = quarter == 0 && m < a.M && n < r1;
    floatx4_t acc = floatx4_t{0.f, 0.f, 0.f, 0.f};
    // one unit: its data, the product, the request of the unit kSlots ahead (`next`) into the slot it leaves
    auto round = [&](u32x4_t (&x)[2], int next, bool wraps, bool first) {
      __builtin_amdgcn_s_waitcnt(wait_vm((kResident ? 2 : 4) * (kSlots - 1)));
      asm volatile("" ::: "memory");
      if (first && (kLate || item > 0)) epi.load(s, m, n, mine, second, item);
      acc = multiply(x, acc);
      if (wraps) {
        ++req_item;
        point();
      }
      request(next);
    };
    if constexpr (kResident) {
#pragma unroll
      for (int u = 0; u < NU; ++u) round(xf[u], (u + kSlots) % NU, (u + kSlots) % NU == 0, u == 0);
    } else {
      for (int u = 0; u < rounds; u += kSlots) {
        const bool wraps = u + kSlots >= rounds;
#pragma unroll
        for (int h = 0; h < kSlots; ++h) round(xf[h], wraps ? h : u + kSlots + h, wraps && h == 0, h == 0 && u == 0);
      }
    }
    // acc[e] is (m = 4 g + e, n_l) over this wavefront's share of K
    float(*buf)[kPlane] = part[kPlanes == 2 ? item & 1 : 0];
#pragma unroll
    for (int e = 0; e < 4; ++e) buf[wave][e * 64 + lane] = acc[e];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    float v = (buf[quarter][at] + buf[quarter + 4][at]) + (buf[quarter + 8][at] + buf[quarter + 12][at]);
    v += quad_xor<0xB1>(v);
    v += quad_xor<0x4E>(v);
    if constexpr (kNorm) {
      if (item == 0) {
        float total = 0.f;
        for (int w = 0; w < kWaves; ++w) total += row_ssq[w * 16 + m];
        inv = rsqrtf(total / (float)(row_bytes / 2) + a.eps);
      }
      v *= inv;
    }
    if (kPlanes == 1 && item + 1 < items) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");    // (the block is read by all)
    epi.apply(s, m, n, v, mine, second, item);
  }
  __builtin_amdgcn_s_waitcnt(wait_vm(0));                    // nothing may still be writing LDS when the workgroup ends
}

// Shares: workgroups for the rows of either operand in proportion to their number, at most one per compute unit together, each
// with at least kMinRows rows; `granule` rows of the first operand's stay together.
static inline int plan(Args& a, int granule) {
  const int cus = device_compute_units(), na = a.n_b < a.N ? a.n_b : a.N, nb = a.N - na;
  const int ga = (na + granule - 1) / granule;
  auto lim = [](int v, int lo, int hi) { return v < lo ? lo : v > hi ? hi : v; };
  auto most = [&](int rows, int g) { return lim(rows / (kMinRows > g ? kMinRows : g), 1, cus); };
  int wa = nb ? lim((int)((int64_t)cus * na / a.N), 1, cus - 1) : cus;
  wa = lim(wa, 1, most(na, granule) < ga ? most(na, granule) : ga);
  if (granule > 1) wa = (ga + (ga + wa - 1) / wa - 1) / ((ga + wa - 1) / wa);
  const int wb = nb ? lim(cus - wa, 1, most(nb, 1)) : 0;
  a.granule = granule;
  a.wgs_a = wa;
  a.qa = ga / wa;
  a.ra = ga % wa;
  a.qb = wb ? nb / wb : 0;
  a.rb = wb ? nb % wb : 0;
  return wa + wb;
}

template <class Epi, int NU, int kPro>
int start(const Args& a, const typename Epi::Args& s, int wgs, hipStream_t st) {
  static std::atomic<int> lds_limit_raised{0};
  MSA_HIP(raise_dynamic_lds_limit(lds_limit_raised, reinterpret_cast<const void*>(rows_ring_kernel<Epi, NU, kPro>), lds_bytes(kPro, NU)));
  rows_ring_kernel<Epi, NU, kPro><<<wgs, kWaves * 64, lds_bytes(kPro, NU), st>>>(a, s);
  MSA_LAUNCH_CHECK();
  return MSA_OK;
}

template <class Epi, int kPro = kPlain>
int launch(Args a, const typename Epi::Args& s, int granule, hipStream_t st) {
  const int wgs = plan(a, granule);
  const int units = (a.row_bytes + kUnitBytes * kWaves - 1) / (kUnitBytes * kWaves);
  if (units <= 1) return start<Epi, 1, kPro>(a, s, wgs, st);
  if (units <= 2) return start<Epi, 2, kPro>(a, s, wgs, st);
  if (units <= 3) return start<Epi, 3, kPro>(a, s, wgs, st);
  if constexpr (kPro != kPost && kPro != kFinal) {
    if (units <= 4) return start<Epi, 4, kPro>(a, s, wgs, st);
    if (units <= kMaxResident) return start<Epi, kMaxResident, kPro>(a, s, wgs, st);
  }
  if constexpr (kPro != kPlain) {
    msa_set_error("rows_ring: a folded norm takes rows of at most %d bytes, not %d", (kPro == kNormed || kPro == kEmbed ? kMaxResident : kMaxPost) * kUnitBytes * kWaves, a.row_bytes);
    return MSA_EINVAL;
  } else {
    return start<Epi, 0, kPlain>(a, s, wgs, st);
  }
}

}  // namespace rows_ring
