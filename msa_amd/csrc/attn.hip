// GQA attention of ragged query rows over per-sample KV ranges (decode and stage-2 prefill).
//
// Split-KV: workgroup (query row, KV head, split) streams its slice of K and V once and serves all G query heads of that KV head from
// the same loads; splits are merged by a second kernel.  K / V rows are [Hkv, 128].  Two forms: bf16 rows go through a ring in LDS and
// the matrix cores (attn_ring_kernel, below), fp32 rows and some bf16 rows of one and two heads through the vector units
// (attn_partial_kernel; takes_ring in attn_internal.h has the line).  In the latter a wavefront takes 4 keys per step (16 lanes per
// key, 8 head-dim elements per lane: dim_of); every (key slot, dim slice) lane keeps an online-softmax state (m, l, acc[G][8]) of its own that
// is merged across slots and wavefronts.
#include "attn_internal.h"

namespace {

// 2^x by the bare hardware instruction: the library exp2f wraps it in a range fix-up for results below
// 2^-126 (five more VALU operations per call); softmax arguments are <= 0 and such tails may flush to zero.
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }


constexpr int kMaxG = 8;

// 16 bytes of K or V with the non-temporal hint: a decode step reads every cache row exactly once, so the rows
// should not displace anything in L2 (the whole decode step runs 3 % faster with the hint).
typedef unsigned int u32x4_stream_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 ld16_stream(const void* p) {
  // (memory, said outright: of a pointer that may be one of two the compiler makes flat loads, which also wait for LDS)
  const u32x4_stream_t w = __builtin_nontemporal_load((const __attribute__((address_space(1))) u32x4_stream_t*)(uintptr_t)p);
  return make_uint4(w.x, w.y, w.z, w.w);
}

__device__ __forceinline__ void ld8(const bf16_t* p, float (&x)[8]) {
  const uint4 w = ld16_stream(p);
  x[0] = bf16lo(w.x); x[1] = bf16hi(w.x); x[2] = bf16lo(w.y); x[3] = bf16hi(w.y);
  x[4] = bf16lo(w.z); x[5] = bf16hi(w.z); x[6] = bf16lo(w.w); x[7] = bf16hi(w.w);
}
__device__ __forceinline__ void ld8(const float* p, float (&x)[8]) {
  const uint4 a = ld16_stream(p), b = ld16_stream(p + kHeadDim / 2);
  x[0] = __uint_as_float(a.x); x[1] = __uint_as_float(a.y); x[2] = __uint_as_float(a.z); x[3] = __uint_as_float(a.w);
  x[4] = __uint_as_float(b.x); x[5] = __uint_as_float(b.y); x[6] = __uint_as_float(b.z); x[7] = __uint_as_float(b.w);
}

// Lane j of the 16 that share a key holds eight of its dimensions, in the pieces of 16 bytes that it loads: neighbours in bf16; of an fp32
// row four in either half, so that the lanes' pieces are whole cache lines (eight neighbours are two loads that touch every second piece:
// with non-temporal loads a line came twice from memory, 16 samples of 2926 to 4388 keys 140 -> 105 us).
template <typename T>
__device__ __forceinline__ constexpr int dim_of(int j, int i) {
  return sizeof(T) == 2 ? 8 * j + i : 4 * j + (i & 3) + (i >> 2) * (kHeadDim / 2);
}

// The same of any float: the rotary tables need not be aligned.
__device__ __forceinline__ void ld8_any(const float* p, float (&x)[8]) {
  typedef float f32x4_any_t __attribute__((ext_vector_type(4), aligned(4)));
  const f32x4_any_t a = *reinterpret_cast<const f32x4_any_t*>(p), b = *reinterpret_cast<const f32x4_any_t*>(p + 4);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[i] = a[i];
    x[4 + i] = b[i];
  }
}

// Finds the sample owning query row `row` in cu_q (B is small: linear scan is fine and uniform).
__device__ __forceinline__ int find_sample(const int32_t* cu_q, int B, int row) {
  int b = 0;
  while (b + 1 < B && cu_q[b + 1] <= row) ++b;
  return b;
}

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a), __builtin_bit_cast(bf16x2_t, b), c, false);
}

// sum over the 16 lanes of a DPP row (the lanes sharing one key); every lane gets the total
__device__ __forceinline__ float row16_allsum(float d) {
  d += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, d), 0x128, 0xf, 0xf, false));
  d += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, d), 0x124, 0xf, 0xf, false));
  d += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, d), 0x122, 0xf, 0xf, false));
  d += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, d), 0x121, 0xf, 0xf, false));
  return d;
}

__device__ const uint4 kZeros[(kHeadDim / 2 + 4) / 4] = {};             // what ld8 reaches of a float

// Streams keys first, first + stride, ... < key1 of one KV head through the running softmax state of this
// lane (key slot = lane / 16, dims 8 j .. 8 j + 8).  Keys go in batches of kBatch steps: all K / V loads of a
// batch are issued before any arithmetic (bytes in flight), scores are reduced over the 16 lanes of a key with
// DPP row rotations, and the running softmax is rescaled once per batch.  `lane_off` is the element offset of
// key 0's slice for this lane.
template <typename T, int G, int kBatch>
__device__ __forceinline__ void attend_keys(const T* __restrict__ k, const T* __restrict__ v, int64_t lane_off,
                                            int row_elems, int first, int key1, int stride, const float (&qv)[G][8],
                                            float (&m)[G], float (&l)[G], float (&acc)[G][8]) {
  for (int kb = first; kb < key1; kb += stride * kBatch) {
    float kx[kBatch][8], vx[kBatch][8];
    bool ok[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int kk = kb + u * stride;
      ok[u] = kk < key1;
      const int64_t off = lane_off + (int64_t)(ok[u] ? kk : kb) * row_elems;   // clamp: always in range
      ld8(k + off, kx[u]);
      ld8(ok[u] ? v + off : reinterpret_cast<const T*>(kZeros), vx[u]);   // (an infinite value with the weight zero would be NaN)
    }
#pragma unroll
    for (int h = 0; h < G; ++h) {
      float s[kBatch];
      float mb = m[h];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        float d = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) d += qv[h][i] * kx[u][i];
        d = row16_allsum(d);
        s[u] = ok[u] ? d : -INFINITY;
        mb = fmaxf(mb, s[u]);
      }
      // mb is finite here: the batch's first key is always valid
      const float alpha = fast_exp2(m[h] - mb);
      float psum = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[h][i] *= alpha;
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const float pu = fast_exp2(s[u] - mb);
        psum += pu;
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[h][i] += pu * vx[u][i];
      }
      l[h] = l[h] * alpha + psum;
      m[h] = mb;
    }
  }
}

// ------------------------------------------------------------------------------------------------
// bf16 single rows: keys and values of one KV head through a ring in LDS, products on the matrix cores.
//
// A workgroup has four wavefronts, each with 8 KB for a step's 32 keys and 8 KB for their values, and every fourth step, so that
// nothing waits for another wavefront until the end.  K is requested again as soon as its products are read, under the softmax, V
// behind the second product: 8 to 16 KB a wavefront are in flight, and two workgroups a compute unit cover each other's ends.  Rows
// of 256 bytes arrive by direct-to-LDS loads, four whole rows an instruction, non-temporal (a decode step reads every cache row
// once), their 16-byte units XORed with the row against bank conflicts.  S^T = K Q^T (16 keys x 16 heads, of which G exist) leaves
// the scores where P^T is wanted as the operand of O^T = V^T P^T; V^T comes by transposing LDS reads.  What bounds it is HBM for long
// contexts (decode steps, 8 KV heads of four: 16 samples of 32768 keys 354 us, 6.1 TB/s; 16 of 2194 to 4388 keys 53.0 -> 47.8 us; one
// of 4388 18.1 -> 12.6) and the chain lengths - first step - sums - combining launch for short ones (one sample of 256 keys 11.2 -> 9.7
// us): the form before held K and V in registers and took packed dot products on the vector units, 350 instructions per 8 KB.
// ------------------------------------------------------------------------------------------------
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4_t;
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
constexpr int kRingWaves = 4, kRingKeys = 32, kRowBytes = kHeadDim * 2, kSlab = kRingKeys * kRowBytes;
constexpr int kParts = kRingWaves + 1, kSumStride = kHeadDim + 4;      // a wavefront each, and the new token's
[[maybe_unused]] constexpr int kNonTemporal = 2;
constexpr int kRingLds = kRingWaves * 2 * kSlab;
constexpr int wait_vm(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }   // vmcnt(n) alone

__device__ __forceinline__ uint32_t lds_offset(const void* p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p; }
// 16 bytes of LDS that no ring writes: the compiler's own accesses would wait for what the rings have in flight.
__device__ __forceinline__ uint4 lds_read16(const uint4* p) {
  u32x4_t v;
  asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(v) : "v"(lds_offset(p)) : "memory");
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void lds_write16(uint4* p, uint4 v) {
  asm volatile("ds_write_b128 %0, %1" : : "v"(lds_offset(p)), "v"(u32x4_t{v.x, v.y, v.z, v.w}) : "memory");
}

// What one wavefront (or the new token) knows of its keys, per head: reference maximum, sum, un-normalised output.  A wavefront's
// lie where its ring was, the new token's behind the rings.
struct HeadSums {
  float m[kMaxG], l[kMaxG], o[kMaxG][kSumStride];
};
static_assert(sizeof(HeadSums) <= 2 * kSlab, "sums take a ring's place");
__device__ __forceinline__ HeadSums& sums_of(char* lds, int part) { return *reinterpret_cast<HeadSums*>(lds + part * 2 * kSlab); }

// Keys key0 .. key1 (`k` / `v`: the head's columns of key 0, `row_bytes` between keys).  `start` requests this wavefront's first
// step; `run` leaves its sums where its ring was.
struct Ring {
  const bf16_t *k, *v;
  char *kt, *vt;
  int row_bytes, key0, key1, steps, wave, off[4];
  __device__ __forceinline__ Ring(const bf16_t* k_, const bf16_t* v_, int row_bytes_, int key0_, int key1_, int wave_, int lane, char* lds)
      : k(k_), v(v_), kt(lds + wave_ * 2 * kSlab), vt(kt + kSlab), row_bytes(row_bytes_), key0(key0_), key1(key1_),
        steps(key1_ > key0_ ? (key1_ - key0_ + kRingKeys - 1) / kRingKeys : 0), wave(wave_) {
    // lane's place in four rows: row lane / 16, where unit (lane % 16) ^ row lies; rows 4 i .. further on change the unit's high bits
#pragma unroll
    for (int i = 0; i < 4; ++i) off[i] = (4 * i + (lane >> 4)) * row_bytes + (((lane & 15) ^ (4 * i + (lane >> 4))) * 16);
  }
  __device__ __forceinline__ void request(const bf16_t* src, char* dst, int step) const {
    const int64_t at = (int64_t)(key0 + (step < steps ? step : 0) * kRingKeys) * row_bytes;
    const int rows = __builtin_amdgcn_readfirstlane(step < steps ? min(kRingKeys, key1 - key0 - step * kRingKeys) : 0);
    const int extent = rows > 0 ? (rows - 1) * row_bytes + kRowBytes : 0;       // rows behind the range read as zeros
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(reinterpret_cast<const char*>(src) + at), 0, extent, 0x00020000);
#pragma unroll
    for (int i = 0; i < 8; ++i) MSA_LOAD_TO_LDS(rs, dst + i * 1024, off[i & 3], (i >> 2) * 16 * row_bytes, kNonTemporal);
  }
  __device__ __forceinline__ void start() const {
    request(k, kt, wave);
    request(v, vt, wave);
  }
  template <int kWeightParts>
  __device__ __forceinline__ void run(int lane, int G, const bf16x8_t (&qf)[4], float scale_log2e, char* lds) const;
};

// Two bf16 values with zeros in the place of infinities and NaN.
__device__ __forceinline__ uint32_t finite_pair(uint32_t w) {
  return ((w & 0x7f80u) == 0x7f80u ? 0u : w & 0xffffu) | ((w & 0x7f800000u) == 0x7f800000u ? 0u : w & 0xffff0000u);
}

// The weights go to the matrix cores as kWeightParts bf16 parts, the first the weight rounded, the others what is left of it: one
// alone would depend on which keys share a reference maximum, two hold 16 bits of the weight, three all 24.
template <int kWeightParts>
__device__ __forceinline__ void Ring::run(int lane, int G, const bf16x8_t (&qf)[4], float scale_log2e, char* lds) const {
  const int l16 = lane & 15, g = lane >> 4;
  // V^T operands: eight bytes of row 4 g + l16 / 4 (and of the row 16 further on): lanes 4 r .. 4 r + 3 of 16 name the pieces of
  // row r, column block c's 32 bytes of it being units 2 c and 2 c + 1
  uint32_t v_at[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const int row = 4 * g + (l16 >> 2);
    v_at[c] = lds_offset(vt) + row * kRowBytes + (l16 & 1) * 8 + (((2 * c + ((l16 & 3) >> 1)) ^ row) * 16);
  }
  // A second pass, if there are NaN, in which the weights' low parts see finite values alone: a low part of zero or below against an
  // infinite value makes NaN where the weight itself leaves the infinity.
  floatx4_t o[8];
  float m, l;                            // of head l16: m the same in its four lanes, l each lane's own keys
  for (bool finite_only = false;;) {
#pragma unroll
    for (int c = 0; c < 8; ++c) o[c] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    m = -INFINITY;
    l = 0.f;
    for (int step = wave; step < steps; step += kRingWaves) {
      __builtin_amdgcn_s_waitcnt(wait_vm(8));                // K: only V is younger
      asm volatile("" ::: "memory");
      floatx4_t sc[2] = {floatx4_t{0.f, 0.f, 0.f, 0.f}, floatx4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const bf16x8_t kf = *reinterpret_cast<const bf16x8_t*>(kt + (16 * t + l16) * kRowBytes + ((4 * kk + g) ^ l16) * 16);
          sc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[kk], sc[t], 0, 0, 0);
        }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // K may be requested again
      request(k, kt, step + kRingWaves);
      // sc[t][e] is head l16's score of key 16 t + 4 g + e
      const int valid = key1 - key0 - step * kRingKeys;
      float x[2][4], mx = m;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[t][e] = 16 * t + 4 * g + e < valid ? sc[t][e] * scale_log2e : -INFINITY;
          mx = fmaxf(mx, x[t][e]);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      if (__any(mx > m)) {
        const float alpha = mx == -INFINITY ? 1.f : fast_exp2(m - mx);
        l *= alpha;
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) o[c][e] *= alpha;
        m = mx;
      }
      const float ref = m == -INFINITY ? 0.f : m;            // (scores of -inf alone: every weight is 0)
      uint32_t part[kWeightParts][4];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          float p0 = fast_exp2(x[t][e] - ref), p1 = fast_exp2(x[t][e + 1] - ref);
          l += p0 + p1;
#pragma unroll
          for (int i = 0; i < kWeightParts; ++i) {
            const uint32_t w = part[i][2 * t + e / 2] = pack_bf16x2(p0, p1);
            p0 -= bf16lo(w);
            p1 -= bf16hi(w);
          }
        }
      __builtin_amdgcn_s_waitcnt(wait_vm(8));                // V: only the next K is younger
      asm volatile("" ::: "memory");
      // (the transposing reads are written out, wait included: in front of its own the compiler waits for the next K too, 4 us in 50)
      u32x2_t vr[16];
      asm volatile(
          "ds_read_b64_tr_b16 %0, %16\n\tds_read_b64_tr_b16 %1, %16 offset:4096\n\t"
          "ds_read_b64_tr_b16 %2, %17\n\tds_read_b64_tr_b16 %3, %17 offset:4096\n\t"
          "ds_read_b64_tr_b16 %4, %18\n\tds_read_b64_tr_b16 %5, %18 offset:4096\n\t"
          "ds_read_b64_tr_b16 %6, %19\n\tds_read_b64_tr_b16 %7, %19 offset:4096\n\t"
          "ds_read_b64_tr_b16 %8, %20\n\tds_read_b64_tr_b16 %9, %20 offset:4096\n\t"
          "ds_read_b64_tr_b16 %10, %21\n\tds_read_b64_tr_b16 %11, %21 offset:4096\n\t"
          "ds_read_b64_tr_b16 %12, %22\n\tds_read_b64_tr_b16 %13, %22 offset:4096\n\t"
          "ds_read_b64_tr_b16 %14, %23\n\tds_read_b64_tr_b16 %15, %23 offset:4096\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(vr[0]), "=&v"(vr[1]), "=&v"(vr[2]), "=&v"(vr[3]), "=&v"(vr[4]), "=&v"(vr[5]), "=&v"(vr[6]), "=&v"(vr[7]),
            "=&v"(vr[8]), "=&v"(vr[9]), "=&v"(vr[10]), "=&v"(vr[11]), "=&v"(vr[12]), "=&v"(vr[13]), "=&v"(vr[14]), "=&v"(vr[15])
          : "v"(v_at[0]), "v"(v_at[1]), "v"(v_at[2]), "v"(v_at[3]), "v"(v_at[4]), "v"(v_at[5]), "v"(v_at[6]), "v"(v_at[7])
          : "memory");
      request(v, vt, step + kRingWaves);                     // (V has been read)
#pragma unroll
      for (int i = 0; i < kWeightParts; ++i) {
        if (i == 1 && finite_only) {
#pragma unroll
          for (int c = 0; c < 16; ++c) vr[c] = u32x2_t{finite_pair(vr[c].x), finite_pair(vr[c].y)};
        }
        const bf16x8_t w8 = __builtin_bit_cast(bf16x8_t, make_uint4(part[i][0], part[i][1], part[i][2], part[i][3]));
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, make_uint4(vr[2 * c].x, vr[2 * c].y, vr[2 * c + 1].x, vr[2 * c + 1].y));
          o[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, w8, o[c], 0, 0, 0);
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(wait_vm(0));                  // nothing may still be writing LDS when the sums go there
    asm volatile("" ::: "memory");
    bool nan = false;
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) nan |= o[c][e] != o[c][e];
    if (finite_only || !__any(nan)) break;
    finite_only = true;
    start();
  }
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if (l16 >= G) return;
  HeadSums& out = sums_of(lds, wave);
#pragma unroll
  for (int c = 0; c < 8; ++c) *reinterpret_cast<floatx4_t*>(&out.o[l16][16 * c + 4 * g]) = o[c];
  if (g == 0) {
    out.m[l16] = m;
    out.l[l16] = l;
  }
}

// Folds the first `parts` sums of a head; thread (h, d).
__device__ __forceinline__ void fold_sums(char* lds, int parts, int h, int d, float& m, float& l, float& o) {
  m = -INFINITY;
  for (int w = 0; w < parts; ++w) m = fmaxf(m, sums_of(lds, w).m[h]);
  l = o = 0.f;
  for (int w = 0; w < parts; ++w) {
    const HeadSums& s = sums_of(lds, w);
    const float a = s.m[h] == -INFINITY ? 0.f : fast_exp2(s.m[h] - m);
    l += s.l[h] * a;
    o += s.o[h][d] * a;
  }
}

// bf16 rows: workgroup (row, KV head, split) as in attn_partial_kernel below.
template <int kWeightParts>
__global__ __launch_bounds__(kRingWaves * 64) void attn_ring_kernel(
    const bf16_t* __restrict__ q, const int32_t* __restrict__ cu_q, const bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
    const int64_t* __restrict__ kv_off, const int32_t* __restrict__ kv_len, int32_t B, int32_t Hq, int32_t Hkv, float scale_log2e,
    int32_t causal, int32_t n_split, float* __restrict__ part_ml, float* __restrict__ part_acc, bf16_t* __restrict__ out) {
  extern __shared__ __align__(16) char lds[];
  const int row = blockIdx.x, g = blockIdx.y, split = blockIdx.z, G = Hq / Hkv;
  const int b = cu_q ? find_sample(cu_q, B, row) : row;
  const int q_first = cu_q ? cu_q[b] : row, sq = cu_q ? cu_q[b + 1] - q_first : 1;
  const int L = kv_len[b], visible = causal ? max(0, L - sq + (row - q_first) + 1) : L;
  // balanced splits of this sample's own length (the host only knows an upper bound of it)
  const int per_split = (L + n_split - 1) / n_split, key0 = split * per_split, key1 = min(visible, key0 + per_split);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t at = kv_off[b] * Hkv * kHeadDim + g * kHeadDim;
  const Ring ring(k + at, v + at, Hkv * kRowBytes, key0, key1, wave, lane, lds);
  bf16x8_t qf[4];
  const uint4* q16 = reinterpret_cast<const uint4*>(q + ((int64_t)row * Hq + g * G) * kHeadDim);
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)                           // lane l16 holds head l16, zeros behind the last
    qf[kk] = __builtin_bit_cast(bf16x8_t, (lane & 15) < G ? q16[(lane & 15) * 16 + 4 * kk + (lane >> 4)] : make_uint4(0, 0, 0, 0));
  asm volatile("" ::: "memory");                           // (the ring counts what is younger)
  ring.start();
  ring.run<kWeightParts>(lane, G, qf, scale_log2e, lds);
  __syncthreads();
  for (int idx = tid; idx < G * kHeadDim; idx += kRingWaves * 64) {
    const int h = idx / kHeadDim, d = idx % kHeadDim;
    float mn, lt, at_d;
    fold_sums(lds, kRingWaves, h, d, mn, lt, at_d);
    const int64_t o = ((int64_t)row * Hq + g * G + h) * n_split + split;
    if (n_split == 1) {                                    // nothing to merge: the output itself (a launch of 4 us less)
      out[o * kHeadDim + d] = f32_to_bf16(lt > 0.f ? at_d / lt : 0.f);          // a row that sees no key yields zeros
      continue;
    }
    part_acc[o * kHeadDim + d] = at_d;
    if (d == 0) { part_ml[o * 2] = mn; part_ml[o * 2 + 1] = lt; }
  }
}

// The softmax states of two lanes kBit apart become their merger in both.
template <int kBit>
__device__ __forceinline__ void merge_slots(float& m, float& l, float (&acc)[8]) {
  auto both = [](float x, float& lower, float& upper) {
    const uint32_t u = __float_as_uint(x);
    if constexpr (kBit == 16) {
      const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
      lower = __uint_as_float(r[0]); upper = __uint_as_float(r[1]);
    } else {
      const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
      lower = __uint_as_float(r[0]); upper = __uint_as_float(r[1]);
    }
  };
  float m0, m1, x0, x1;
  both(m, m0, m1);
  m = fmaxf(m0, m1);
  const float a0 = m == -INFINITY ? 0.f : fast_exp2(m0 - m), a1 = m == -INFINITY ? 0.f : fast_exp2(m1 - m);
  both(l, x0, x1);
  l = x0 * a0 + x1 * a1;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    both(acc[i], x0, x1);
    acc[i] = x0 * a0 + x1 * a1;
  }
}

// fp32 rows, and bf16 rows of groups of one and two heads where takes_ring says so.  A workgroup serves G heads, of a group of G or of a
// larger one whose rows are then read once a workgroup.
template <typename T, int G, int kAttnWaves>
__global__ __launch_bounds__(kAttnWaves * 64) void attn_partial_kernel(
    const T* __restrict__ q, const int32_t* __restrict__ cu_q, const T* __restrict__ k, const T* __restrict__ v,
    const int64_t* __restrict__ kv_off, const int32_t* __restrict__ kv_len, int32_t B, int32_t Hq, int32_t Hkv,
    float scale_log2e, int32_t causal, int32_t n_split, float* __restrict__ part_ml,
    float* __restrict__ part_acc, T* __restrict__ out) {
  __shared__ float sm_m[kAttnWaves][G], sm_l[kAttnWaves][G];
  __shared__ float sm_acc[kAttnWaves][G][kHeadDim];

  // (fp32: with one head twice the bytes in flight are worth their registers, 16 samples of 3000 keys 98 -> 75 us; with four they cost
  // a wavefront a SIMD, 16 of 4388 131 -> 158)
  constexpr int kBatch = sizeof(T) == 4 && G == 1 && kAttnWaves <= 8 ? 8 : 4;
  const int row = blockIdx.x, h0 = blockIdx.y * G, g = h0 / (Hq / Hkv), split = blockIdx.z;
  const int b = cu_q ? find_sample(cu_q, B, row) : row;
  const int q_first = cu_q ? cu_q[b] : row;
  const int sq = cu_q ? cu_q[b + 1] - q_first : 1;
  const int L = kv_len[b];
  const int visible = causal ? max(0, L - sq + (row - q_first) + 1) : L;
  // balanced splits of this sample's own length (the host only knows an upper bound of it)
  const int per_split = (L + n_split - 1) / n_split;
  const int key0 = split * per_split;
  const int key1 = min(visible, key0 + per_split);

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int slot = lane >> 4, j = lane & 15;
  const int64_t base = kv_off[b];
  const int row_elems = Hkv * kHeadDim;

  float m[G], l[G], acc[G][8];
#pragma unroll
  for (int h = 0; h < G; ++h) {
    m[h] = -INFINITY; l[h] = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[h][i] = 0.f;
  }
  const int64_t lane_off = base * row_elems + g * kHeadDim + dim_of<T>(j, 0);     // this lane's slice of key 0
  const T* q_lane = q + ((int64_t)row * Hq + h0) * kHeadDim + dim_of<T>(j, 0);
  float qv[G][8];
#pragma unroll
  for (int h = 0; h < G; ++h) {
    ld8(q_lane + h * kHeadDim, qv[h]);
#pragma unroll
    for (int i = 0; i < 8; ++i) qv[h][i] *= scale_log2e;      // scores in log2 units: exp2f below
  }
  attend_keys<T, G, kBatch>(k, v, lane_off, row_elems, key0 + wave * 4 + slot, key1, kAttnWaves * 4, qv, m, l, acc);

  // merge the 4 key slots of the wavefront (lanes differing in bits 4 and 5): a swap leaves both lanes' values in both, without LDS
#pragma unroll
  for (int h = 0; h < G; ++h) {
    merge_slots<16>(m[h], l[h], acc[h]);
    merge_slots<32>(m[h], l[h], acc[h]);
  }
  if (slot == 0) {
#pragma unroll
    for (int h = 0; h < G; ++h) {
      if (j == 0) { sm_m[wave][h] = m[h]; sm_l[wave][h] = l[h]; }
#pragma unroll
      for (int i = 0; i < 8; ++i) sm_acc[wave][h][dim_of<T>(j, i)] = acc[h][i];
    }
  }
  __syncthreads();

  // merge the wavefronts; thread (h, d) for h < G
  for (int idx = tid; idx < G * kHeadDim; idx += kAttnWaves * 64) {
    const int h = idx / kHeadDim, d = idx % kHeadDim;
    float mn = -INFINITY;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) mn = fmaxf(mn, sm_m[w][h]);
    float lt = 0.f, at = 0.f;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) {
      const float a = mn == -INFINITY ? 0.f : fast_exp2(sm_m[w][h] - mn);
      lt += sm_l[w][h] * a;
      at += sm_acc[w][h][d] * a;
    }
    const int64_t o = ((int64_t)row * Hq + h0 + h) * n_split + split;
    if (n_split == 1) {                                  // nothing to merge: the output itself (a launch of 4 us less)
      const float y = lt > 0.f ? at / lt : 0.f;          // a row that sees no key yields zeros
      if constexpr (sizeof(T) == 2) out[o * kHeadDim + d] = f32_to_bf16(y);
      else out[o * kHeadDim + d] = y;
      continue;
    }
    part_acc[o * kHeadDim + d] = at;
    if (d == 0) { part_ml[o * 2] = mn; part_ml[o * 2 + 1] = lt; }
  }
}

// ------------------------------------------------------------------------------------------------
// Decode step with the q / k RMSNorm, the rotary embedding and the cache append folded into the attention launch
// (bf16, one new token per sample, groups of 4 or 8 query heads).  Row b of `qkv` is the fused projection output
// [Hq q heads | Hkv k heads | Hkv v heads].  A workgroup normalises and rotates the q heads of its group (16 lanes per head, 8 dims
// per lane, the same arithmetic as the stand-alone kernel) and shares them through LDS; the workgroup with a sample's last keys
// also prepares the new token's k / v row of its KV head, writes it to the cache at [b][kv_len[b]] and folds it in as one more
// key.  kv_len is only read here: the combine kernel that follows advances it.  A full cache drops the new row (and the token
// then does not see itself).
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ float row16_ror8(float v) {  // value of the lane 8 places away in the 16-lane row
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x128, 0xf, 0xf, false));
}

// RMSNorm over a head's 128 dims (fp32) times the norm weight, then half-split rotary, 16 lanes a head and 8 dims a lane.  What it
// takes from memory is requested apart from what is done with it: the ring's requests go between the two.
struct NormRope {
  uint4 x, w;
  float cs[8], sn[8];
  __device__ __forceinline__ void load(const bf16_t* src, const bf16_t* weight) {            // this lane's 8 elements
    x = *reinterpret_cast<const uint4*>(src);
    w = *reinterpret_cast<const uint4*>(weight);
  }
  __device__ __forceinline__ void load_rotary(const float* cos_row, const float* sin_row, int j) {
    ld8_any(cos_row + 8 * (j & 7), cs);
    ld8_any(sin_row + 8 * (j & 7), sn);
  }
  __device__ __forceinline__ uint4 result(float eps, int j) const {
    const uint32_t xs[4] = {x.x, x.y, x.z, x.w}, ws[4] = {w.x, w.y, w.z, w.w};
    float v[8], wt[8], ssq = 0.f, out[8];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      v[2 * c] = bf16lo(xs[c]); v[2 * c + 1] = bf16hi(xs[c]);
      wt[2 * c] = bf16lo(ws[c]); wt[2 * c + 1] = bf16hi(ws[c]);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) ssq += v[i] * v[i];
    const float inv = rsqrtf(row16_allsum(ssq) * (1.0f / kHeadDim) + eps);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float y = v[i] * inv * wt[i];
      const float other = row16_ror8(y);        // the paired dim (d + 64 for j < 8, d - 64 for j >= 8)
      out[i] = j < 8 ? y * cs[i] - other * sn[i] : y * cs[i] + other * sn[i];
    }
    return make_uint4(pack_bf16x2(out[0], out[1]), pack_bf16x2(out[2], out[3]), pack_bf16x2(out[4], out[5]), pack_bf16x2(out[6], out[7]));
  }
};

// kPaired (up to 64 samples): the pieces of samples of different lengths dealt so that two beside one another are about as long as any two.  The
// host knows the caches' capacity only: where no sample has `worth` keys the pieces are `few`, in the launch's own order, as without kPaired, and
// the other workgroups leave empty sums.  us, 8 KV heads, both launches, without kPaired, always paired and so: 16 samples of 100 keys in caches of 4388
// 8.4, 10.0 and 8.7, of 1000 17.6, 17.8 and 17.9, 8 of 1000 in 4160 12.3, 14.3 and 12.7, 32 of 300 in 2048 13.1, 14.7 and 13.3.
constexpr int kDecodeUnits = 256;
struct Pairing {
  int32_t worth, few;
};
template <bool kPaired>
__global__ __launch_bounds__(kRingWaves * 64) void attn_decode_fused_kernel(
    const bf16_t* __restrict__ qkv, int64_t row_stride, int32_t Hq, int32_t Hkv, const int64_t* __restrict__ pos,
    const bf16_t* __restrict__ qw, const bf16_t* __restrict__ kw, float eps, const float* __restrict__ cos_t,
    const float* __restrict__ sin_t, int32_t rope_rows, bf16_t* __restrict__ kcache, bf16_t* __restrict__ vcache,
    int32_t Lcap, const int32_t* __restrict__ kv_len, float scale_log2e, int32_t n_split,
    float* __restrict__ part_ml, float* __restrict__ part_acc, Pairing pairing) {
  extern __shared__ __align__(16) char lds[];
  HeadSums& new_token = sums_of(lds, kRingWaves);
  uint4* sm_q = reinterpret_cast<uint4*>(lds + kRingLds + sizeof(HeadSums));        // [G][16]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), G = Hq / Hkv;
  int b = blockIdx.x, g = blockIdx.y, split = blockIdx.z, pieces = n_split, L_old;
  int64_t position;
  const int j = lane & 15, hq = tid >> 4;                  // 16 lanes a head: the group's q heads, and behind them the new key
  NormRope head;
  uint4 v_new;
  auto load_row = [&]() {
    const bf16_t* row = qkv + (int64_t)b * row_stride + 8 * j;
    head.load(row + (int64_t)(hq < G ? g * G + hq : Hq + g) * kHeadDim, (hq < G ? qw : kw) + 8 * j);
    v_new = *reinterpret_cast<const uint4*>(row + (int64_t)(Hq + Hkv + g) * kHeadDim);
  };
  if constexpr (kPaired) {
    // Units in the order of the workgroups, the longest samples first in each of their rounds, the second round (of those a compute unit has
    // two places for) backwards: whoever has a long piece gets a short one beside it.
    const int B = gridDim.x, total = B * Hkv * n_split, second = min(2 * kDecodeUnits, total);
    const int len = lane < B ? kv_len[lane] : 0;
    const int64_t at = lane < B ? pos[lane] : 0;
    load_row();                                            // (of the launch's own order, under the lengths' way here)
    if (__any(len >= pairing.worth)) {
      int unit = b + B * (g + Hkv * split);
      if (unit >= kDecodeUnits && unit < second) unit = kDecodeUnits + second - 1 - unit;
      const int row_of = unit / B, place = unit - row_of * B;
      split = row_of / Hkv;
      g = row_of - split * Hkv;
      // a sample's place by length; no two keys are equal, and those of absent lanes come last
      const uint32_t key = (uint32_t)min(max(len, 0), (1 << 25) - 1) * 64 + (63 - lane);
      int rank = 0;
      for (int i0 = 0; i0 < B; i0 += 16)
#pragma unroll
        for (int i = 0; i < 16; ++i) rank += (uint32_t)__builtin_amdgcn_readlane((int)key, i0 + i) > key;
      b = __builtin_ctzll(__ballot(rank == place));
      load_row();
    } else {
      pieces = pairing.few;
      if (split >= pieces) {
        for (int idx = tid; idx < G * kHeadDim; idx += kRingWaves * 64) {
          const int64_t o = ((int64_t)b * Hq + g * G + idx / kHeadDim) * n_split + split;
          part_acc[o * kHeadDim + idx % kHeadDim] = 0.f;
          if (idx % kHeadDim == 0) { part_ml[o * 2] = -INFINITY; part_ml[o * 2 + 1] = 0.f; }
        }
        return;
      }
    }
    L_old = __builtin_amdgcn_readlane(len, b);
    position = (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)((uint64_t)at >> 32), b) << 32 | (uint32_t)__builtin_amdgcn_readlane((int)at, b));
  } else {
    L_old = kv_len[b];
    position = pos[b];
    load_row();
  }
  const int64_t p = min((int64_t)max((int64_t)0, position), (int64_t)rope_rows - 1);
  head.load_rotary(cos_t + p * 64, sin_t + p * 64, j);

  const bool has_new = L_old < Lcap;
  const int per_split = (L_old + pieces - 1) / pieces, key0 = split * per_split, key1 = min(L_old, key0 + per_split);
  const int64_t column = ((int64_t)b * Lcap * Hkv + g) * kHeadDim;
  const Ring ring(kcache + column, vcache + column, Hkv * kRowBytes, key0, key1, wave, lane, lds);
  asm volatile("" ::: "memory");                           // (the requests above stay above: loads return in order)
  ring.start();                                            // in flight under the queries' preparation

  const uint4 prepared = head.result(eps, j);
  if (hq < G) lds_write16(sm_q + hq * 16 + j, prepared);
  // the new token: the first 16 lanes of the last wavefront of the last split
  const bool takes_new = has_new && split == pieces - 1, owner = takes_new && wave == kRingWaves - 1 && lane < 16;
  if (owner) {
    const int64_t at = (((int64_t)b * Lcap + L_old) * Hkv + g) * kHeadDim + 8 * j;
    *reinterpret_cast<uint4*>(kcache + at) = prepared;
    *reinterpret_cast<uint4*>(vcache + at) = v_new;
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");         // (a full fence would wait for the ring)

  bf16x8_t qf[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    const uint4 u = lds_read16(sm_q + (j < G ? j : 0) * 16 + 4 * kk + (lane >> 4));
    qf[kk] = __builtin_bit_cast(bf16x8_t, j < G ? u : make_uint4(0, 0, 0, 0));
  }
  ring.run<2>(lane, G, qf, scale_log2e, lds);
  if (owner) {
    // one more key, straight from registers: its weight against itself is 1
    const uint32_t vs[4] = {v_new.x, v_new.y, v_new.z, v_new.w};
    for (int h = 0; h < G; ++h) {
      const uint4 q4 = lds_read16(sm_q + h * 16 + j);
      float d = dot2_bf16(q4.x, prepared.x, 0.f);
      d = dot2_bf16(q4.y, prepared.y, d);
      d = dot2_bf16(q4.z, prepared.z, d);
      d = dot2_bf16(q4.w, prepared.w, d);
      d = row16_allsum(d);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        new_token.o[h][8 * j + 2 * c] = bf16lo(vs[c]);
        new_token.o[h][8 * j + 2 * c + 1] = bf16hi(vs[c]);
      }
      if (j == 0) {
        new_token.m[h] = d * scale_log2e;
        new_token.l[h] = 1.f;
      }
    }
  }
  __syncthreads();
  for (int idx = tid; idx < G * kHeadDim; idx += kRingWaves * 64) {
    const int h = idx / kHeadDim, d = idx % kHeadDim;
    float mn, lt, at_d;
    fold_sums(lds, takes_new ? kParts : kRingWaves, h, d, mn, lt, at_d);
    const int64_t o = ((int64_t)b * Hq + g * G + h) * n_split + split;
    part_acc[o * kHeadDim + d] = at_d;
    if (d == 0) { part_ml[o * 2] = mn; part_ml[o * 2 + 1] = lt; }
  }
}

// One workgroup of 128 threads per (query row, head): merges the row's partials and normalises.  The partials are requested sixteen
// at a time (one after the other, each waited for the one before: 32 of them took 16 us), four or eight at a time where there are no more.  With `kv_len` (decode: rows = samples)
// the workgroup of head 0 also advances the sample's cache length, unless the cache was full and the new row was dropped.
template <typename T, int kBatch>
__global__ __launch_bounds__(kHeadDim) void attn_combine_kernel(const float* __restrict__ part_ml,
                                                                const float* __restrict__ part_acc, int32_t n_split,
                                                                T* __restrict__ out, int32_t* __restrict__ kv_len,
                                                                int32_t Lcap, int32_t Hq) {
  const int64_t rh = blockIdx.x;   // row * Hq + head
  const int d = threadIdx.x;
  if (kv_len != nullptr && d == 0 && rh % Hq == 0) {
    const int32_t len = kv_len[rh / Hq];
    if (len < Lcap) kv_len[rh / Hq] = len + 1;
  }
  float mn = -INFINITY, lt = 0.f, at = 0.f;
  for (int s0 = 0; s0 < n_split; s0 += kBatch) {
    float ms[kBatch], ls[kBatch], as[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int64_t p = rh * n_split + min(s0 + i, n_split - 1);
      ms[i] = part_ml[p * 2];
      ls[i] = part_ml[p * 2 + 1];
      as[i] = part_acc[p * kHeadDim + d];
    }
    float mb = mn;
#pragma unroll
    for (int i = 0; i < kBatch; ++i) mb = s0 + i < n_split ? fmaxf(mb, ms[i]) : mb;
    const float keep = mn == -INFINITY ? 0.f : fast_exp2(mn - mb);
    lt *= keep;
    at *= keep;
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const bool in = s0 + i < n_split;                  // (an infinity in the last partial would be NaN in the places behind it)
      const float a = ms[i] != -INFINITY ? fast_exp2(ms[i] - mb) : 0.f;
      lt += in ? ls[i] * a : 0.f;
      at += in ? as[i] * a : 0.f;
    }
    mn = mb;
  }
  const float o = lt > 0.f ? at / lt : 0.f;     // a row that sees no key yields zeros
  if constexpr (sizeof(T) == 2) out[rh * kHeadDim + d] = f32_to_bf16(o);
  else out[rh * kHeadDim + d] = o;
}

template <typename T>
int launch_combine(const float* part_ml, const float* part_acc, int64_t rows, int32_t n_split, void* out, hipStream_t st,
                   int32_t* kv_len = nullptr, int32_t Lcap = 0, int32_t Hq = 1) {
  const auto kernel = n_split <= 4 ? attn_combine_kernel<T, 4> : n_split <= 8 ? attn_combine_kernel<T, 8> : attn_combine_kernel<T, 16>;
  kernel<<<(unsigned)rows, kHeadDim, 0, st>>>(part_ml, part_acc, n_split, static_cast<T*>(out), kv_len, Lcap, Hq);
  MSA_LAUNCH_CHECK();
  return MSA_OK;
}

// Heads a workgroup of fp32 rows where whole groups would leave most of the chip idle; 0: whole groups.  A group's workgroups read its rows
// again, from the caches, which costs less than its heads one after another as long as the workgroups do not outnumber the compute units
// (`head_splits`: with one head each; twice as many with two).  More than two splits are short already.  us, 8 KV heads of four, groups
// / two heads / one: one row of 192 keys 11.4 / 9.0 / 8.1, 8 rows 12.5 / 8.6 / 7.3, 16 rows 13.5 / 9.5 / 12.2, 32 rows 15.3 / 15.4 /
// 21.9; 2 rows of 400 keys in two splits 14.5 / 11.3 / 11.2, of 1000 in four 15.2 / 12.2 / 14.8, of 2000 in eight 16.2 / 15.6 / 25.3; 4 rows
// of 2000 19.3 / 26.8 / 32.8.  Groups of one and two are in four wavefronts then, which is as many as few keys keep busy (eight, so and now: one head,
// 16 rows of 100 keys 7.1 / 6.1, 25 of 43 6.2 / 4.3; two, 4 rows of 82 6.4 / 4.7, one of 100 6.2 / 5.1, but 8 of 110 6.6 / 7.5).
int spread_heads(int64_t head_splits, int G, int n_split, int max_kv) {
  constexpr int kUnits = 256;
  if (G != 1 && G != 2 && G != 4 && G != 8) return 0;       // (two heads of a group of three would be of two groups; launch_attn refuses these)
  if ((G == 1 && max_kv <= 128) || (G == 2 && max_kv <= 104)) return 0;
  if (head_splits <= kUnits && n_split <= 2) return 1;
  return G >= 2 && head_splits <= 2 * kUnits ? 2 : 0;
}

template <typename T>
int launch_attn(const void* q, const int32_t* cu_q, const void* k, const void* v, const int64_t* kv_off,
                    const int32_t* kv_len, int32_t B, int32_t total_q, int32_t Hq, int32_t Hkv, float scale,
                    int32_t causal, SplitPlan plan, void* out, float* part_ml, float* part_acc, hipStream_t st, int spread = 0) {
  const int n_split = plan.n_split;
  const int G = spread ? spread : Hq / Hkv;
  dim3 grid((unsigned)total_q, (unsigned)(Hq / G), (unsigned)n_split);
  const float sl2 = scale * 1.4426950408889634f;
#define MSA_ATTN_CASE(GG, WW)                                                                                      \
  case GG:                                                                                                         \
    attn_partial_kernel<T, GG, WW><<<grid, WW * 64, 0, st>>>(                                                      \
        static_cast<const T*>(q), cu_q, static_cast<const T*>(k), static_cast<const T*>(v), kv_off, kv_len, B, Hq, \
        Hkv, sl2, causal, n_split, part_ml, part_acc, static_cast<T*>(out));                                       \
    return MSA_OK;
  const auto first = [&] {
    if constexpr (sizeof(T) == 4) {
      if (spread) switch (G) {
          MSA_ATTN_CASE(1, 8)
          MSA_ATTN_CASE(2, 8)
        }
    }
    switch (G) {
      MSA_ATTN_CASE(1, 4)
      MSA_ATTN_CASE(2, 4)
    }
    if constexpr (sizeof(T) == 4) {
      switch (G) {
        MSA_ATTN_CASE(4, 8)
        MSA_ATTN_CASE(8, 8)
      }
    }
    msa_set_error("msa_sparse_attn: GQA group size %d unsupported (1, 2, 4, 8)", G);
    return MSA_EINVAL;
  };
#undef MSA_ATTN_CASE
  if (const int rc = first(); rc != MSA_OK) return rc;
  MSA_LAUNCH_CHECK();
  if (n_split == 1) return MSA_OK;
  return launch_combine<T>(part_ml, part_acc, (int64_t)total_q * Hq, n_split, out, st);
}

constexpr int kFusedLds = kRingLds + (int)sizeof(HeadSums) + kMaxG * 16 * (int)sizeof(uint4);
static_assert(2 * kFusedLds <= 160 * 1024, "two workgroups a compute unit");

template <int kWeightParts>
int launch_attn_ring(const void* q, const int32_t* cu_q, const void* k, const void* v, const int64_t* kv_off,
                     const int32_t* kv_len, int32_t B, int32_t total_q, int32_t Hq, int32_t Hkv, float scale,
                     int32_t causal, SplitPlan plan, void* out, float* part_ml, float* part_acc, hipStream_t st) {
  const int n_split = plan.n_split;
  static std::atomic<int> lds_limit_raised{0};
  MSA_HIP(raise_dynamic_lds_limit(lds_limit_raised, reinterpret_cast<const void*>(attn_ring_kernel<kWeightParts>), kRingLds));
  attn_ring_kernel<kWeightParts><<<dim3((unsigned)total_q, (unsigned)Hkv, (unsigned)n_split), kRingWaves * 64, kRingLds, st>>>(
      static_cast<const bf16_t*>(q), cu_q, static_cast<const bf16_t*>(k), static_cast<const bf16_t*>(v), kv_off, kv_len, B, Hq, Hkv,
      scale * 1.4426950408889634f, causal, n_split, part_ml, part_acc, static_cast<bf16_t*>(out));
  MSA_LAUNCH_CHECK();
  if (n_split == 1) return MSA_OK;
  return launch_combine<bf16_t>(part_ml, part_acc, (int64_t)total_q * Hq, n_split, out, st);
}

int launch_attn_bf16(const void* q, const int32_t* cu_q, const void* k, const void* v, const int64_t* kv_off,
                     const int32_t* kv_len, int32_t B, int32_t total_q, int32_t max_kv, int32_t Hq, int32_t Hkv, float scale,
                     int32_t causal, SplitPlan plan, void* out, float* part_ml, float* part_acc, hipStream_t st) {
  const int G = Hq / Hkv;
  if (!takes_ring(total_q, Hkv, max_kv, G))
    return launch_attn<bf16_t>(q, cu_q, k, v, kv_off, kv_len, B, total_q, Hq, Hkv, scale, causal, plan, out, part_ml, part_acc, st);
  const auto launch = G <= 2 ? launch_attn_ring<3> : launch_attn_ring<2>;
  return launch(q, cu_q, k, v, kv_off, kv_len, B, total_q, Hq, Hkv, scale, causal, plan, out, part_ml, part_acc, st);
}

int rows_splits(int32_t total_q, int32_t Hkv, int32_t max_kv) {
  return std::max(plan_splits(total_q, Hkv, max_kv).n_split, plan_splits_rows(total_q, Hkv, max_kv, true).n_split);
}
size_t partials_bytes(int32_t total_q, int32_t Hq, int32_t D, int splits) {
  const size_t n = (size_t)total_q * Hq * splits;
  return align_up(n * 2 * sizeof(float), 256) + align_up(n * D * sizeof(float), 256);
}
// Splits where decoding samples take the paired form: as many as two workgroups a compute unit hold; 0 where plan_splits_rows' form is ahead.
// Finding a workgroup's sample costs 0.4 us, and a piece wants keys: 500 where one workgroup a unit comes out even, 160 where it does not.
// Both launches, us, even splits and pairs (8 KV heads, all of one length and of half of it to all): 16 of 4388 keys 55.6 -> 52.7 and
// 49.4 -> 43.9, of 2500 36.1 -> 34.3 and 31.3 -> 29.0, one of 4388 and fifteen of 500 34.0 -> 25.0, 15 of 2000 31.1 -> 27.9 and 26.6 -> 23.4,
// 7 of 2000 21.4 -> 17.6 and 19.8 -> 16.8, 5 of 2000 17.4 -> 15.4; not taken: 16 of 1000 18.1 -> 18.5, 8 of 2000 18.0 -> 19.1, 5 of 1000 11.1 -> 11.9,
// 3 of 4388 16.5 -> 17.9.
int paired_splits(int32_t B, int32_t Hkv, int32_t Lcap) {
  const int64_t pairs = (int64_t)B * Hkv;
  if (B > 64 || pairs < 32 || pairs > 2 * kDecodeUnits) return 0;
  const int n = (int)(2 * kDecodeUnits / pairs);
  if (n * pairs < 400) return 0;                           // (too few places taken: 24 samples of 2000 43.3 -> 44.0)
  return Lcap >= n * (kDecodeUnits % pairs == 0 ? 500 : 160) ? n : 0;
}
// From how many keys of the longest sample on the pieces are dealt in pairs, in a launch that has the workgroups for it: fewer than the capacity's
// line above, where the choice is between these and half as many pieces in the same launch.
Pairing pairing_of(int64_t pairs, int n, int even) { return {n * (n == 1 || kDecodeUnits % pairs == 0 ? 300 : 50), std::min(even, n)}; }

}  // namespace

extern "C" size_t msa_attn_workspace_bytes(int32_t total_q, int32_t Hq, int32_t Hkv, int32_t D, int32_t max_kv) {
  if (total_q <= 0 || Hq <= 0 || Hkv <= 0 || D <= 0 || max_kv <= 0) return 0;
  // sized for whichever of the kernels has more partials
  const int by_tiles = plan_splits_tiles(total_q, 1, Hq / Hkv, Hkv, max_kv).n_split;
  return partials_bytes(total_q, Hq, D, std::max({rows_splits(total_q, Hkv, max_kv), paired_splits(total_q, Hkv, max_kv), by_tiles}));
}

extern "C" int msa_sparse_attn(const void* q, const int32_t* cu_q, const void* k, const void* v,
                               const int64_t* kv_off, const int32_t* kv_len, int32_t B, int32_t total_q,
                               int32_t max_sq, int32_t max_kv, int32_t Hq, int32_t Hkv, int32_t D, int32_t dtype,
                               float scale, int32_t causal, void* out, void* workspace, size_t workspace_bytes,
                               void* stream) {
  MSA_REQUIRE(q && k && v && kv_off && kv_len && out && workspace, "msa_sparse_attn: null pointer");
  MSA_REQUIRE(D == kHeadDim, "msa_sparse_attn: head dim %d unsupported (need %d)", D, kHeadDim);
  MSA_REQUIRE(B > 0 && total_q > 0 && max_sq > 0 && max_kv > 0, "msa_sparse_attn: bad sizes");
  MSA_REQUIRE(cu_q != nullptr || total_q == B, "msa_sparse_attn: cu_q is required when total_q != B");
  MSA_REQUIRE(Hkv > 0 && Hq % Hkv == 0 && Hq / Hkv <= kMaxG, "msa_sparse_attn: Hq=%d Hkv=%d unsupported", Hq, Hkv);
  MSA_REQUIRE(dtype == MSA_BF16 || dtype == MSA_F32, "msa_sparse_attn: bad dtype %d", dtype);
  MSA_REQUIRE(scale > 0.f, "msa_sparse_attn: scale must be positive");
  MSA_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15) == 0,
              "msa_sparse_attn: q, k, v and out must be 16-byte aligned");
  MSA_REQUIRE((int64_t)total_q * Hq < (int64_t)1 << 31 && total_q < 65536 * 32, "msa_sparse_attn: too many rows");
  const bool mfma = dtype == MSA_BF16 && max_sq >= 8;
  const SplitPlan tiles = plan_splits_tiles(total_q, B, Hq / Hkv, Hkv, max_kv);
  const bool by_tiles = mfma && partials_bytes(total_q, Hq, D, tiles.n_split) <= workspace_bytes;
  const SplitPlan plan = by_tiles ? tiles : mfma ? plan_splits(total_q, Hkv, max_kv) : plan_splits_rows(total_q, Hkv, max_kv, dtype == MSA_BF16 && takes_ring(total_q, Hkv, max_kv, Hq / Hkv));
  const int n_split = plan.n_split;
  MSA_REQUIRE(n_split <= 65535, "msa_sparse_attn: max_kv=%d too large", max_kv);
  const size_t need = partials_bytes(total_q, Hq, D, rows_splits(total_q, Hkv, max_kv));
  if (need > workspace_bytes) {
    msa_set_error("msa_sparse_attn: workspace of %zu bytes, need %zu", workspace_bytes, need);
    return MSA_ESIZE;
  }
  const size_t n = (size_t)total_q * Hq * n_split;
  float* part_ml = static_cast<float*>(workspace);
  float* part_acc = reinterpret_cast<float*>(static_cast<char*>(workspace) + align_up(n * 2 * sizeof(float), 256));
  hipStream_t st = as_stream(stream);
  if (mfma) {
    // bf16 query blocks: MFMA partial pass (K / V tiles through LDS, shared by a tile's rows) + the common combine; single rows
    // (decode) share nothing between them and take the split-KV forms of this file
    int rc = flash_attn_split_launch(q, cu_q, k, v, kv_off, kv_len, B, total_q, Hq, Hkv, scale, causal, plan, part_ml,
                                     part_acc, st);
    if (rc != MSA_OK) return rc;
    return launch_combine<bf16_t>(part_ml, part_acc, (int64_t)total_q * Hq, n_split, out, st);
  }
  if (dtype == MSA_BF16)
    return launch_attn_bf16(q, cu_q, k, v, kv_off, kv_len, B, total_q, max_kv, Hq, Hkv, scale, causal, plan, out, part_ml,
                            part_acc, st);
  return launch_attn<float>(q, cu_q, k, v, kv_off, kv_len, B, total_q, Hq, Hkv, scale, causal, plan, out, part_ml, part_acc, st,
                            spread_heads((int64_t)total_q * Hq * n_split, Hq / Hkv, n_split, max_kv));
}

extern "C" int msa_decode_attn_fused(const void* qkv, int64_t row_stride, const int64_t* positions, const void* q_norm_w,
                                     const void* k_norm_w, float eps, const float* rope_cos, const float* rope_sin,
                                     int32_t rope_rows, int32_t B, int32_t Hq, int32_t Hkv, int32_t D, void* kcache,
                                     void* vcache, int32_t Lcap, int32_t* kv_len, float scale, void* out,
                                     void* workspace, size_t workspace_bytes, void* stream) {
  MSA_REQUIRE(qkv && positions && q_norm_w && k_norm_w && rope_cos && rope_sin && kcache && vcache && kv_len && out &&
                  workspace, "msa_decode_attn_fused: null pointer");
  MSA_REQUIRE(D == kHeadDim, "msa_decode_attn_fused: head dim %d unsupported (need %d)", D, kHeadDim);
  MSA_REQUIRE(B > 0 && Hkv > 0 && Hkv <= 65535 && Hq % Hkv == 0 && (Hq / Hkv == 4 || Hq / Hkv == 8),
              "msa_decode_attn_fused: B=%d Hq=%d Hkv=%d (groups of 4 or 8 query heads)", B, Hq, Hkv);
  MSA_REQUIRE(row_stride >= (int64_t)(Hq + 2 * Hkv) * D && row_stride % 8 == 0, "msa_decode_attn_fused: bad row stride");
  MSA_REQUIRE((((uintptr_t)qkv | (uintptr_t)q_norm_w | (uintptr_t)k_norm_w | (uintptr_t)kcache | (uintptr_t)vcache) & 15) == 0,
              "msa_decode_attn_fused: pointers must be 16-byte aligned");
  MSA_REQUIRE(Lcap > 0 && rope_rows > 0 && eps > 0.f && scale > 0.f, "msa_decode_attn_fused: bad scalar argument");
  const int paired = paired_splits(B, Hkv, Lcap);
  const bool pairs = paired > 0 && partials_bytes(B, Hq, D, paired) <= workspace_bytes;
  const size_t need = partials_bytes(B, Hq, D, rows_splits(B, Hkv, Lcap));
  if (need > workspace_bytes) {
    msa_set_error("msa_decode_attn_fused: workspace of %zu bytes, need %zu", workspace_bytes, need);
    return MSA_ESIZE;
  }
  const int even = plan_splits_rows(B, Hkv, Lcap, true).n_split, n_split = pairs ? paired : even;
  const size_t n = (size_t)B * Hq * n_split;
  float* part_ml = static_cast<float*>(workspace);
  float* part_acc = reinterpret_cast<float*>(static_cast<char*>(workspace) + align_up(n * 2 * sizeof(float), 256));
  hipStream_t st = as_stream(stream);
  static std::atomic<int> lds_limit_raised[2] = {{0}, {0}};
  const auto kernel = pairs ? attn_decode_fused_kernel<true> : attn_decode_fused_kernel<false>;
  MSA_HIP(raise_dynamic_lds_limit(lds_limit_raised[pairs], reinterpret_cast<const void*>(kernel), kFusedLds));
  kernel<<<dim3((unsigned)B, (unsigned)Hkv, (unsigned)n_split), kRingWaves * 64, kFusedLds, st>>>(
      static_cast<const bf16_t*>(qkv), row_stride, Hq, Hkv, positions, static_cast<const bf16_t*>(q_norm_w),
      static_cast<const bf16_t*>(k_norm_w), eps, rope_cos, rope_sin, rope_rows, static_cast<bf16_t*>(kcache),
      static_cast<bf16_t*>(vcache), Lcap, kv_len, scale * 1.4426950408889634f, n_split, part_ml, part_acc,
      pairs ? pairing_of((int64_t)B * Hkv, n_split, even) : Pairing{});
  MSA_LAUNCH_CHECK();
  return launch_combine<bf16_t>(part_ml, part_acc, (int64_t)B * Hq, n_split, out, st, kv_len, Lcap, Hq);
}
