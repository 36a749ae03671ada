// Decode attention on a device-resident KV ring (gfx950): RoPE + append, and
// grouped-query attention with sink logits over a window of the ring.
//
// Replaces, for one decode token, apply_rope + KVCacheManager.append/get +
// the score / softmax / context steps of StreamedAttention.forward
// (streamed_attention.py:80-98, 120-141; kv_cache_manager.py:39-56).  The
// reference stacks the whole cache into fresh tensors every step and runs
// torch einsum/softmax; here the keys never move.
//
// Numerics follow the reference's cast points: RoPE rounds every bfloat16 op
// (a*cos, b*sin, difference/sum) and the rotated key and the value are
// stored in the cache's type (float16 by default, or bfloat16); scores are
// float32 q.k / sqrt(D) (the dot product accumulated in float64 and rounded
// once); the softmax over [scores, sink] is float32 with the maximum
// subtracted; probabilities are rounded to the cache's type before the value
// sum, which accumulates in float32 per split and float64 across splits, is
// rounded to the cache's type and then to bfloat16 (o_proj's input type).
//
// Kernels per step: scores with per-block maxima and sums (workgroup = one KV
// head x 64 to 256 keys, its whole query group), probabilities x values
// (workgroup = one KV head x 128 or 256 keys), and the sum of the splits; a
// window of at most 256 keys runs as one launch, scores to context, one
// workgroup per query head.  Measured for 64 / 8 heads x 64, float16 (cold
// rings): 128 keys 7.7 -> 6.0 us, 4,096 23.7 -> 16.5, 8,192 40.2 -> 20.5,
// 16,384 81.6 -> 27.6, 32,768 200 -> 42.7 against value workgroups per query
// head that each took their head's statistics over all its scores (quadratic
// in the context: 186 of the 200 us) and vector float64 dot products per
// query head (38 us -> 20).
#include <math.h>

#include <chrono>

#include "klc_common.h"

namespace klc {
namespace {

constexpr int kAttnThreads = 256;
constexpr int kProjThreads = 128;  // projection kernels: 64, 128 and 256 measured alike (2880 rows: 6.9, 6.7, 7.6 us)
constexpr int kPvKeys = 256;     // most keys of a value workgroup, and of a one-launch window
constexpr int kMaxHeadDim = 128;
constexpr int kMaxGroup = 16;    // query heads per KV head
constexpr int kMaxRow = 8 * 8 * kWave;  // longest projection input: 8 chunks of 16 bytes a lane
typedef double f64x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
__device__ __forceinline__ uint16_t to_bf(float f) { return (uint16_t)f32_to_bf16_rne(f); }
__device__ __forceinline__ float rbf(float f) { return bf(to_bf(f)); }
// the cache's element type: float16 (the reference's default "fp16") or bfloat16
__device__ __forceinline__ float kv_f(uint16_t b, bool f16) { return f16 ? __half2float(__ushort_as_half(b)) : bf(b); }
__device__ __forceinline__ uint16_t to_kv(float f, bool f16) {
  return f16 ? __half_as_ushort(__float2half_rn(f)) : to_bf(f);
}
__device__ __forceinline__ float rkv(float f, bool f16) { return kv_f(to_kv(f, f16), f16); }

// q [NH][D], k/v [NKV][D] -> q_out [NH][D]; k, v into ring slot `slot`.
__global__ __launch_bounds__(kAttnThreads) void rope_append_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    const uint16_t* __restrict__ cosv, const uint16_t* __restrict__ sinv, uint16_t* __restrict__ q_out,
    uint16_t* __restrict__ k_out, uint16_t* __restrict__ k_cache, uint16_t* __restrict__ v_cache, int64_t slot, int nh, int nkv, int d, bool f16) {
  const int half = d / 2;
  const int pairs = (nh + nkv) * half;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < pairs + nkv * d; i += gridDim.x * blockDim.x) {
    if (i < pairs) {
      const int row = i / half, j = i - row * half;
      const bool is_q = row < nh;
      const uint16_t* src = is_q ? q + (int64_t)row * d : k + (int64_t)(row - nh) * d;
      uint16_t* dst = is_q ? q_out + (int64_t)row * d : k_cache + (slot * nkv + (row - nh)) * d;
      const float a = bf(src[j]), b = bf(src[j + half]), c = bf(cosv[j]), s = bf(sinv[j]);
      const float lo = rbf(rbf(a * c) - rbf(b * s)), hi = rbf(rbf(b * c) + rbf(a * s));  // bfloat16 rotation
      dst[j] = is_q ? to_bf(lo) : to_kv(lo, f16);  // the key is stored in the cache's type
      dst[j + half] = is_q ? to_bf(hi) : to_kv(hi, f16);
      if (!is_q && k_out != nullptr) {  // the rotated key before storage, for diagnostics
        k_out[(int64_t)(row - nh) * d + j] = to_bf(lo);
        k_out[(int64_t)(row - nh) * d + j + half] = to_bf(hi);
      }
    } else {
      const int e = i - pairs;
      v_cache[slot * nkv * d + e] = f16 ? to_kv(bf(v[e]), true) : v[e];
    }
  }
}

// ---- one decode step's projections ------------------------------------------

// Dot products of two bfloat16 rows with the bfloat16 x [k], by one wave: lane
// l takes the 16-byte chunks l, l + 64, ...; all 3 J loads are issued by
// load(), so a caller can work under them.  A product of two bfloat16 values
// is exact in float64 and the sum is taken there, so what the caller rounds
// is the correctly rounded dot product (the float64 work rides under the
// weight stream).  Lanes past a row's end read zeros.  Every lane gets both
// sums.
template <int J>
struct TwoRows {
  u32x4_t xv[J], v0[J], v1[J];

  __device__ __forceinline__ void load(const uint16_t* w0, const uint16_t* w1, const uint16_t* x, int k) {
    const int lane = threadIdx.x % kWave;
    const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc((void*)x, (short)0, k * 2, kBufferWord3);
    const __amdgpu_buffer_rsrc_t b0 = __builtin_amdgcn_make_buffer_rsrc((void*)w0, (short)0, k * 2, kBufferWord3);
    const __amdgpu_buffer_rsrc_t b1 = __builtin_amdgcn_make_buffer_rsrc((void*)w1, (short)0, k * 2, kBufferWord3);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const uint32_t at = (uint32_t)(lane + kWave * j) * 16u;
      v0[j] = __builtin_amdgcn_raw_buffer_load_b128(b0, at, 0, kStreamPolicy);
      v1[j] = __builtin_amdgcn_raw_buffer_load_b128(b1, at, 0, kStreamPolicy);
      xv[j] = __builtin_amdgcn_raw_buffer_load_b128(xb, at, 0, 0);
    }
  }

  __device__ __forceinline__ void dot(double& sum0, double& sum1) const {
    double a0[2] = {0.0, 0.0}, a1[2] = {0.0, 0.0};
#pragma unroll
    for (int j = 0; j < J; ++j) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const double xl = (double)__uint_as_float(xv[j][i] << 16), xh = (double)__uint_as_float(xv[j][i] & 0xffff0000u);
        a0[0] = fma((double)__uint_as_float(v0[j][i] << 16), xl, a0[0]);
        a1[0] = fma((double)__uint_as_float(v1[j][i] << 16), xl, a1[0]);
        a0[1] = fma((double)__uint_as_float(v0[j][i] & 0xffff0000u), xh, a0[1]);
        a1[1] = fma((double)__uint_as_float(v1[j][i] & 0xffff0000u), xh, a1[1]);
      }
    }
    sum0 = a0[0] + a0[1];
    sum1 = a1[0] + a1[1];
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
      sum0 += __shfl_xor(sum0, off);
      sum1 += __shfl_xor(sum1, off);
    }
  }
};

// bias[row], 0 without a bias (an empty buffer), with no branch; loaded before
// the rows, so that nothing waits for it alone
__device__ __forceinline__ float bias_at(const uint16_t* bias, int row) {
  const __amdgpu_buffer_rsrc_t b = __builtin_amdgcn_make_buffer_rsrc((void*)bias, (short)0,
                                                                     bias != nullptr ? 2 * (row + 1) : 0, kBufferWord3);
  return bf((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(b, 2 * row, 0, 0));
}
__device__ __forceinline__ uint16_t biased_bf(double sum, float bias) { return to_bf((float)(sum + (double)bias)); }

struct QkvArgs {
  const uint16_t *x, *qw, *qb, *kw, *kb, *vw, *vb;
  const float* inv_freq;      // [d / 2]
  uint16_t *pre, *rot;        // [nh + nkv][d] queries then keys, before and after RoPE
  uint16_t *k_cache, *v_cache;
  int64_t slot;
  int hidden, nh, nkv, d;
  float position, rope_scale;
  bool f16;
};

// q, k and v projections of one token with RoPE and the append in the
// epilogue: a wave owns the two rows of one rotated pair (dims j and j +
// d / 2 of a head), or two value rows, so the rotation needs nothing from
// another wave and the step has no launch for it.  cos and sin are taken
// while the rows are on their way, with torch's rounding points (float32
// angle, float32 product with the scaling, bfloat16).  HBM bound: 29.5 MB for
// 5120 rows of 2880 in 8.5 us (10.4 with the biases read through a branch,
// which waited for every row in flight).
template <int J>
__global__ __launch_bounds__(kProjThreads) void attn_qkv_kernel(QkvArgs a) {
  const int half = a.d / 2, pairs = (a.nh + a.nkv) * half;
  const int p = blockIdx.x * (kProjThreads / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (p >= pairs + a.nkv * half) return;
  TwoRows<J> rows;
  double s0, s1;
  if (p >= pairs) {
    const int r0 = 2 * (p - pairs);
    const uint16_t* w = a.vw + (int64_t)r0 * a.hidden;
    const float b0 = bias_at(a.vb, r0), b1 = bias_at(a.vb, r0 + 1);
    rows.load(w, w + a.hidden, a.x, a.hidden);
    rows.dot(s0, s1);
    if (threadIdx.x % kWave == 0) {
      uint16_t* dst = a.v_cache + a.slot * a.nkv * a.d + r0;
      const uint16_t v0 = biased_bf(s0, b0), v1 = biased_bf(s1, b1);
      dst[0] = a.f16 ? to_kv(bf(v0), true) : v0;
      dst[1] = a.f16 ? to_kv(bf(v1), true) : v1;
    }
    return;
  }
  const int head = p / half, j = p - head * half;
  const bool is_q = head < a.nh;
  const int row = (is_q ? head : head - a.nh) * a.d + j;
  const uint16_t* w = (is_q ? a.qw : a.kw) + (int64_t)row * a.hidden;
  const uint16_t* b = is_q ? a.qb : a.kb;
  const float b0 = bias_at(b, row), b1 = bias_at(b, row + half), freq = a.inv_freq[j];
  rows.load(w, w + (int64_t)half * a.hidden, a.x, a.hidden);
  const float angle = __fmul_rn(freq, a.position);
  const float c = rbf(__fmul_rn(cosf(angle), a.rope_scale)), s = rbf(__fmul_rn(sinf(angle), a.rope_scale));
  rows.dot(s0, s1);
  if (threadIdx.x % kWave == 0) {
    const uint16_t pl = biased_bf(s0, b0), ph = biased_bf(s1, b1);
    const float x0 = bf(pl), x1 = bf(ph);
    const float lo = rbf(rbf(x0 * c) - rbf(x1 * s)), hi = rbf(rbf(x1 * c) + rbf(x0 * s));  // bfloat16 rotation
    const int at = head * a.d + j;
    a.pre[at] = pl;
    a.pre[at + half] = ph;
    a.rot[at] = to_bf(lo);
    a.rot[at + half] = to_bf(hi);
    if (!is_q) {
      uint16_t* dst = a.k_cache + a.slot * a.nkv * a.d + row;
      dst[0] = to_kv(lo, a.f16);
      dst[half] = to_kv(hi, a.f16);
    }
  }
}

// out[r] = bf16(x . w[r] + bias[r]) for a bfloat16 weight [rows][k]: two rows
// a wave.  HBM bound: 23.6 MB (2880 rows of 4096) in 6.7 us.
template <int J>
__global__ __launch_bounds__(kProjThreads) void attn_out_kernel(const uint16_t* __restrict__ w,
                                                                const uint16_t* __restrict__ bias,
                                                                const uint16_t* __restrict__ x,
                                                                uint16_t* __restrict__ out, int rows, int k) {
  const int r0 = 2 * (blockIdx.x * (kProjThreads / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave));
  if (r0 >= rows) return;
  const int r1 = min(r0 + 1, rows - 1);
  TwoRows<J> two;
  const float b0 = bias_at(bias, r0), b1 = bias_at(bias, r1);
  two.load(w + (int64_t)r0 * k, w + (int64_t)r1 * k, x, k);
  double s0, s1;
  two.dot(s0, s1);
  if (threadIdx.x % kWave == 0) {
    out[r0] = biased_bf(s0, b0);
    if (r1 > r0) out[r1] = biased_bf(s1, b1);
  }
}

// What the host reads back from a step: the norms of q and k before RoPE,
// after it and of the difference, the non-finite values after it, and a tag
// word written last, all in pinned host memory.
struct StepRecord {
  const uint16_t *pre, *rot;  // [nh + nkv][d]
  uint32_t* host;             // NULL: no record
  uint32_t tag;
};

// One workgroup: sums of squares in float64 and the record.  It runs beside
// the score workgroups of the same launch and must not outlast them: 16-byte
// loads, all in flight (2-byte ones made a 4,096-key score launch 10.2 us
// instead of 6.7).
__device__ __forceinline__ void write_record(const StepRecord& rec, int nh, int nkv, int d) {
  __shared__ double sums[kAttnThreads / kWave][6];
  __shared__ int bad[kAttnThreads / kWave][2];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  double t[6] = {};
  int n[2] = {0, 0};
  const int chunks = (nh + nkv) * d / 8, q_chunks = nh * d / 8;
  constexpr int kAhead = 3;
  for (int c0 = threadIdx.x; c0 < chunks; c0 += kAhead * kAttnThreads) {
    uint4 x[kAhead], y[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int c = min(c0 + i * kAttnThreads, chunks - 1);
      x[i] = reinterpret_cast<const uint4*>(rec.pre)[c];
      y[i] = reinterpret_cast<const uint4*>(rec.rot)[c];
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int c = c0 + i * kAttnThreads;
      if (c >= chunks) break;
      double pre = 0.0, post = 0.0, delta = 0.0;
      int count = 0;
      auto add = [&](uint32_t xa, uint32_t ya) {
        const float u = bf((uint16_t)xa), v = bf((uint16_t)ya), z = v - u;
        pre += (double)u * u;
        post += (double)v * v;
        delta += (double)z * z;
        count += !isfinite(v);
      };
      const uint32_t xs[4] = {x[i].x, x[i].y, x[i].z, x[i].w}, ys[4] = {y[i].x, y[i].y, y[i].z, y[i].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        add(xs[e] & 0xffffu, ys[e] & 0xffffu);
        add(xs[e] >> 16, ys[e] >> 16);
      }
      const bool is_q = c < q_chunks;
      t[0] += is_q ? pre : 0.0, t[1] += is_q ? 0.0 : pre;
      t[2] += is_q ? post : 0.0, t[3] += is_q ? 0.0 : post;
      t[4] += is_q ? delta : 0.0, t[5] += is_q ? 0.0 : delta;
      n[0] += is_q ? count : 0, n[1] += is_q ? 0 : count;
    }
  }
#pragma unroll
  for (int e = 0; e < 6; ++e)
    for (int off = kWave / 2; off > 0; off >>= 1) t[e] += __shfl_xor(t[e], off);
#pragma unroll
  for (int e = 0; e < 2; ++e)
    for (int off = kWave / 2; off > 0; off >>= 1) n[e] += __shfl_xor(n[e], off);
  if (lane == 0) {
    for (int e = 0; e < 6; ++e) sums[wave][e] = t[e];
    for (int e = 0; e < 2; ++e) bad[wave][e] = n[e];
  }
  __syncthreads();
  if (wave != 0) return;
  if (lane < 8) {
    uint32_t word;
    if (lane < 6) {
      double v = 0.0;
      for (int w = 0; w < kAttnThreads / kWave; ++w) v += sums[w][lane];
      word = __float_as_uint((float)sqrt(v));
    } else {
      int v = 0;
      for (int w = 0; w < kAttnThreads / kWave; ++w) v += bad[w][lane - 6];
      word = (uint32_t)v;
    }
    rec.host[lane] = word;
  }
  __threadfence_system();  // one wave wrote the record: its tag follows it
  if (lane == 0) __hip_atomic_store(rec.host + 8, rec.tag, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ring slot of key i of a span starting at slot `first`
__device__ __forceinline__ int64_t ring_slot(int64_t first, int64_t i, int64_t cap) {
  const int64_t s = first + i;
  return s >= cap ? s - cap : s;
}

// 8 elements of the cache type as float64 operands
template <bool kF16>
__device__ __forceinline__ double kv_d(const uint4& v, int i) {
  const uint32_t w = i < 2 ? v.x : i < 4 ? v.y : i < 6 ? v.z : v.w;
  return (double)kv_f((uint16_t)((i & 1) ? w >> 16 : w & 0xffffu), kF16);
}

// A window of at most 256 keys in one launch: workgroup = query head
// blockIdx.x (a KV head's group would halve the loads and leave the chip
// idle).  It is a latency chain, so everything it will read is requested at
// the start: a thread's key row (P threads share a row) and its value rows
// (thread (key slot, 8 dims)).  Scores are the same correctly rounded
// float64 dot products as attn_scores_kernel's; every wave takes the maximum
// and the sum over all of them itself, so the reductions need no exchange
// between waves.  Measured at 128 keys: 8.3 -> 6.1 us against statistics
// exchanged through LDS, value loads after them and slice sums through
// global memory.
template <int P, int kC, bool kF16>
__global__ __launch_bounds__(kAttnThreads) void attn_window_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_cache, const uint16_t* __restrict__ sinks,
    const uint16_t* __restrict__ v_cache, uint16_t* __restrict__ context, int64_t cap, int64_t first, int count,
    int nh, int nkv, int d, float sqrt_d, StepRecord rec) {
  if ((int)blockIdx.x == nh) {
    write_record(rec, nh, nkv, d);
    return;
  }
  constexpr int kDims = 64 * kC;             // head_dim <= kDims
  constexpr int kChunks = kDims / 8 / P;     // 16-byte chunks of a key row per thread
  __shared__ __align__(16) double qs[kDims];
  __shared__ __align__(16) float sc[kPvKeys];
  __shared__ float p[kPvKeys];
  __shared__ float red[kAttnThreads * 8];    // [slot][d]
  const int h = blockIdx.x, kvh = h / (nh / nkv);
  const int key = threadIdx.x / P, part = threadIdx.x % P;
  const uint16_t* krow = k_cache + (ring_slot(first, min(key, count - 1), cap) * nkv + kvh) * d;
  uint4 kr[kChunks];
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const int at = 8 * (P * c + part);
    kr[c] = make_uint4(0, 0, 0, 0);
    if (at < d) kr[c] = *reinterpret_cast<const uint4*>(krow + at);
  }
  const int dl = d / 8, slots = kAttnThreads / dl;
  const int dq = threadIdx.x % dl, slot = threadIdx.x / dl;
  constexpr int kAhead = 8;
  uint4 v[kAhead];
  auto vrow = [&](int i) {
    return *reinterpret_cast<const uint4*>(v_cache + (ring_slot(first, min(i, count - 1), cap) * nkv + kvh) * d + 8 * dq);
  };
#pragma unroll
  for (int j = 0; j < kAhead; ++j) {
    v[j] = make_uint4(0, 0, 0, 0);
    if (slot + j * slots < count) v[j] = vrow(slot + j * slots);
  }
  const float sink = sinks != nullptr ? bf(sinks[h]) : -INFINITY;
  for (int i = threadIdx.x; i < kDims; i += kAttnThreads) qs[i] = i < d ? (double)bf(q[(int64_t)h * d + i]) : 0.0;
  __syncthreads();
  {
    double acc[2] = {0.0, 0.0};
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      const double2* qc = reinterpret_cast<const double2*>(qs + 8 * (P * c + part));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const double2 qq = qc[e];
        acc[0] = fma(kv_d<kF16>(kr[c], 2 * e), qq.x, acc[0]);
        acc[1] = fma(kv_d<kF16>(kr[c], 2 * e + 1), qq.y, acc[1]);
      }
    }
    double dot = acc[0] + acc[1];
#pragma unroll
    for (int off = 1; off < P; off <<= 1) dot += __shfl_xor(dot, off);
    if (part == 0 && key < count) sc[key] = (float)dot / sqrt_d;
  }
  __syncthreads();
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  float s[4], m = sink;
  const float4 s4 = reinterpret_cast<const float4*>(sc)[lane];
  s[0] = s4.x, s[1] = s4.y, s[2] = s4.z, s[3] = s4.w;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (4 * lane + e < count) m = fmaxf(m, s[e]);
  for (int off = kWave / 2; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  double l = 0.0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    s[e] = expf(s[e] - m);
    if (4 * lane + e < count) l += (double)s[e];
  }
  for (int off = kWave / 2; off > 0; off >>= 1) l += __shfl_xor(l, off);
  if (sinks != nullptr) l += (double)expf(sink - m);
  const float lf = (float)l;
  if (lane / (kWave / 4) == wave) {  // each wave writes a quarter of the probabilities
#pragma unroll
    for (int e = 0; e < 4; ++e) p[4 * lane + e] = 4 * lane + e < count ? rkv(s[e] / lf, kF16) : 0.f;
  }
  __syncthreads();
  float a[8] = {};
  if (slot < slots) {
    for (int i0 = slot; i0 < count; i0 += kAhead * slots) {
      if (i0 != slot) {
#pragma unroll
        for (int j = 0; j < kAhead; ++j) v[j] = vrow(i0 + j * slots);
      }
#pragma unroll
      for (int j = 0; j < kAhead; ++j) {
        if (i0 + j * slots >= count) break;
        const float w = p[i0 + j * slots];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t x = e < 2 ? v[j].x : e < 4 ? v[j].y : e < 6 ? v[j].z : v[j].w;
          a[e] = fmaf(w, kv_f((uint16_t)((e & 1) ? x >> 16 : x & 0xffffu), kF16), a[e]);
        }
      }
    }
    float4* dst = reinterpret_cast<float4*>(red + slot * d + 8 * dq);
    dst[0] = make_float4(a[0], a[1], a[2], a[3]);
    dst[1] = make_float4(a[4], a[5], a[6], a[7]);
  }
  __syncthreads();
  if ((int)threadIdx.x < d) {
    float t = 0.f;
#pragma unroll 8
    for (int i = 0; i < min(slots, count); ++i) t += red[i * d + threadIdx.x];
    context[(int64_t)h * d + threadIdx.x] = to_bf(rkv(t, kF16));
  }
}

// Scores of one KV head's query group against 64 * T keys (blockIdx.y), and
// per head the block's maximum and sum of exp(score - maximum).
//
// A wave multiplies 16-key tiles with v_mfma_f64_16x16x4_f64: A = keys (lane
// l holds key row l % 16, dims 32 c + 8 (l / 16) + i), B = the group's
// queries (column l % 16, same dims), so every key element is converted to
// float64 once for all heads (a vector dot product per head converted it g
// times), and 16 lanes' loads cover 64 contiguous bytes of each key.  D lane l register i is
// row l / 16 + 4 i; tile row m holds key 4 (m % 4) + m / 4, so a lane ends up
// with 4 consecutive keys of head l % 16 and stores them as one float4.
// Groups of fewer than 16 heads leave MFMA columns idle.
template <int T, int kC, bool kF16>
__global__ __launch_bounds__(kAttnThreads) void attn_scores_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_cache, float* __restrict__ scores,
    float* __restrict__ stat_m, double* __restrict__ stat_l, int64_t cap, int64_t first, int count, int cs, int nblk,
    int nh, int nkv, int d, float sqrt_d, float inv_sqrt, StepRecord rec) {
  if ((int)blockIdx.y == nblk) {
    if (blockIdx.x == 0) write_record(rec, nh, nkv, d);
    return;
  }
  __shared__ __align__(16) uint16_t qs[kMaxGroup][kMaxHeadDim + 8];
  __shared__ float wm[kAttnThreads / kWave][kMaxGroup];
  __shared__ double wl[kAttnThreads / kWave][kMaxGroup];
  const int g = nh / nkv, kvh = blockIdx.x, blk = blockIdx.y;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int r = lane & 15, kq = lane >> 4;  // MFMA row / column, dim quarter
  const int key0 = (blk * (kAttnThreads / kWave) + wave) * 16 * T;
  // kC chunks of 32 dims (head_dim <= 32 kC): dims 32 c + 8 kq of the head exist: d is a multiple of 8
  uint4 kr[T][kC];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int key = min(key0 + 16 * t + 4 * (r & 3) + (r >> 2), count - 1);
    const uint16_t* row = k_cache + (ring_slot(first, key, cap) * nkv + kvh) * d + 8 * kq;
#pragma unroll
    for (int c = 0; c < kC; ++c)
      kr[t][c] = 32 * c + 8 * kq < d ? *reinterpret_cast<const uint4*>(row + 32 * c) : make_uint4(0, 0, 0, 0);
  }
  for (int i = threadIdx.x; i < g * d; i += kAttnThreads) qs[i / d][i % d] = q[(int64_t)kvh * g * d + i];
  __syncthreads();
  uint4 qr[kC];
#pragma unroll
  for (int c = 0; c < kC; ++c) {
    qr[c] = make_uint4(0, 0, 0, 0);
    if (32 * c + 8 * kq < d && r < g) qr[c] = *reinterpret_cast<const uint4*>(&qs[r][32 * c + 8 * kq]);
  }
  f64x4_t acc[T] = {};
#pragma unroll
  for (int c = 0; c < kC; ++c) {
    if (32 * c >= d) break;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const double qd = kv_d<false>(qr[c], i);
#pragma unroll
      for (int t = 0; t < T; ++t)
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(kv_d<kF16>(kr[t][c], i), qd, acc[t], 0, 0, 0);
    }
  }
  const int h = kvh * g + r;
  float s[T][4];
  float m = -INFINITY;
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int k4 = key0 + 16 * t + 4 * kq;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // a power of two divides exactly as its reciprocal multiplies
      s[t][i] = inv_sqrt != 0.f ? (float)acc[t][i] * inv_sqrt : (float)acc[t][i] / sqrt_d;
      if (k4 + i < count) m = fmaxf(m, s[t][i]);
    }
    if (r < g && k4 < count)  // rows are padded to 4 scores
      *reinterpret_cast<float4*>(scores + (int64_t)h * cs + k4) = make_float4(s[t][0], s[t][1], s[t][2], s[t][3]);
  }
  m = fmaxf(m, __shfl_xor(m, 16));
  m = fmaxf(m, __shfl_xor(m, 32));
  if (kq == 0) wm[wave][r] = m;
  __syncthreads();
  m = wm[0][r];
  for (int w = 1; w < kAttnThreads / kWave; ++w) m = fmaxf(m, wm[w][r]);
  // a block of -inf scores adds nothing (and NaN stays NaN)
  const float base = m == -INFINITY ? 0.f : m;
  double l = 0.0;
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (key0 + 16 * t + 4 * kq + i < count) l += (double)expf(s[t][i] - base);
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if (kq == 0) wl[wave][r] = l;
  __syncthreads();
  if ((int)threadIdx.x < g) {
    double sum = 0.0;
    for (int w = 0; w < kAttnThreads / kWave; ++w) sum += wl[w][r];
    const int64_t at = (int64_t)h * nblk + blk;
    stat_m[at] = m;
    stat_l[at] = sum;
  }
}

// partial[h][split][d] = sum over the split's keys of p * v for the heads of
// one KV head (blockIdx.x), p = exp(score - max) / sum rounded to the cache
// type.  Each value row is read once per 4 heads: thread (8 dims, block of 4
// heads, key slot).  The head's max and sum come from the score blocks'
// (a few KB instead of all its scores): 186 -> 18.8 us at 32,768 keys.
template <bool kF16>
__global__ __launch_bounds__(kAttnThreads) void attn_pv_kernel(
    const float* __restrict__ scores, const float* __restrict__ stat_m, const double* __restrict__ stat_l, int nblk,
    const uint16_t* __restrict__ sinks, const uint16_t* __restrict__ v_cache, float* __restrict__ partial, int64_t cap,
    int64_t first, int count, int cs, int ks_log2, int nh, int nkv, int d) {
  const int ks = 1 << ks_log2;
  // p [key][heads, 16-byte blocks, one spare to spread the banks], then, past
  // a barrier, the slots' sums [slot][head][d]
  constexpr int kRed = kAttnThreads * 32;
  __shared__ __align__(16) float lds[kRed];
  static_assert(kPvKeys * (kMaxGroup + 4) <= kRed, "p fits");
  __shared__ float head_m[kMaxGroup], head_l[kMaxGroup];
  float* const p = lds;
  float* const red = lds;
  const int g = nh / nkv, kvh = blockIdx.x, split = blockIdx.y;
  const int k0 = split * ks, nk = min(ks, count - k0);
  const int dl = d / 8, hb = (g + 3) / 4, slots = kAttnThreads / (dl * hb);
  const int dq = threadIdx.x % dl, hblk = threadIdx.x / dl % hb, slot = threadIdx.x / (dl * hb);
  const bool live = slot < slots;
  auto vrow = [&](int i) {
    return *reinterpret_cast<const uint4*>(v_cache + (ring_slot(first, k0 + i, cap) * nkv + kvh) * d + 8 * dq);
  };
  // the first value rows are on their way while the statistics are taken
  constexpr int kAhead = 8;
  uint4 v[kAhead];
#pragma unroll
  for (int j = 0; j < kAhead; ++j) v[j] = vrow(min(slot + j * slots, nk - 1));

  // and so are the scores
  constexpr int kHeldScores = kPvKeys * kMaxGroup / kAttnThreads;
  float sc[kHeldScores];
#pragma unroll
  for (int j = 0; j < kHeldScores; ++j) {
    const int i = threadIdx.x + j * kAttnThreads;
    const int hh = i >> ks_log2, key = i & (ks - 1);
    sc[j] = 0.f;
    if (hh < g) sc[j] = scores[(int64_t)(kvh * g + hh) * cs + k0 + min(key, nk - 1)];
  }
  // 16 to 64 lanes a head take its statistics, every head at once
  const int lanes = g > 8 ? 16 : g > 4 ? 32 : 64;
  {
    const int hh = threadIdx.x / lanes, ln = threadIdx.x % lanes;
    const int h = kvh * g + min(hh, g - 1);
    const float* sm = stat_m + (int64_t)h * nblk;
    const double* sl = stat_l + (int64_t)h * nblk;
    const float sink = sinks != nullptr ? bf(sinks[h]) : -INFINITY;
    constexpr int kHold = 4;
    float bm[kHold];
    double bl[kHold];
#pragma unroll
    for (int j = 0; j < kHold; ++j) {
      const int b = ln + j * lanes;
      bm[j] = b < nblk ? sm[b] : -INFINITY;
      bl[j] = b < nblk ? sl[b] : 0.0;
    }
    float m = sink;
#pragma unroll
    for (int j = 0; j < kHold; ++j) m = fmaxf(m, bm[j]);
    for (int b = ln + kHold * lanes; b < nblk; b += lanes) m = fmaxf(m, sm[b]);
    for (int off = lanes / 2; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    double l = 0.0;
#pragma unroll
    for (int j = 0; j < kHold; ++j)
      if (ln + j * lanes < nblk) l += bl[j] * (double)expf(bm[j] - m);
    for (int b = ln + kHold * lanes; b < nblk; b += lanes) l += sl[b] * (double)expf(sm[b] - m);
    for (int off = lanes / 2; off > 0; off >>= 1) l += __shfl_xor(l, off);
    if (sinks != nullptr) l += (double)expf(sink - m);
    if (ln == 0 && hh < g) head_m[hh] = m, head_l[hh] = (float)l;
  }
  const int stride = 4 * hb + 4;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kHeldScores; ++j) {
    const int i = threadIdx.x + j * kAttnThreads;
    const int hh = i >> ks_log2, key = i & (ks - 1);
    if (hh >= 4 * hb) break;
    float w = 0.f;
    if (hh < g && key < nk) w = rkv(expf(sc[j] - head_m[hh]) / head_l[hh], kF16);
    p[key * stride + hh] = w;
  }
  __syncthreads();
  float a[4][8] = {};
  if (live) {
    for (int i0 = slot; i0 < nk; i0 += kAhead * slots) {
      if (i0 != slot) {
#pragma unroll
        for (int j = 0; j < kAhead; ++j) v[j] = vrow(min(i0 + j * slots, nk - 1));
      }
#pragma unroll
      for (int j = 0; j < kAhead; ++j) {
        if (i0 + j * slots >= nk) break;
        const float4 w = *reinterpret_cast<const float4*>(p + (i0 + j * slots) * stride + 4 * hblk);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t x = e < 2 ? v[j].x : e < 4 ? v[j].y : e < 6 ? v[j].z : v[j].w;
          const float f = kv_f((uint16_t)((e & 1) ? x >> 16 : x & 0xffffu), kF16);
          a[0][e] = fmaf(w.x, f, a[0][e]);
          a[1][e] = fmaf(w.y, f, a[1][e]);
          a[2][e] = fmaf(w.z, f, a[2][e]);
          a[3][e] = fmaf(w.w, f, a[3][e]);
        }
      }
    }
  }
  __syncthreads();
  if (live) {
#pragma unroll
    for (int hh = 0; hh < 4; ++hh) {
      float4* dst = reinterpret_cast<float4*>(red + ((slot * hb + hblk) * 4 + hh) * d + 8 * dq);
      dst[0] = make_float4(a[hh][0], a[hh][1], a[hh][2], a[hh][3]);
      dst[1] = make_float4(a[hh][4], a[hh][5], a[hh][6], a[hh][7]);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < g * d; i += kAttnThreads) {
    float t = 0.f;
    for (int s = 0; s < slots; ++s) t += red[s * hb * 4 * d + i];
    partial[((int64_t)(kvh * g + i / d) * gridDim.y + split) * d + i % d] = t;
  }
}

// context[h][d] = bf16(sum over splits of partial[h][split][d]): one
// workgroup per head, thread (4 dims, group of splits), summed in float64.
__global__ __launch_bounds__(kAttnThreads) void attn_combine_kernel(const float* __restrict__ partial, int splits,
                                                                    int d, uint16_t* __restrict__ context, bool f16) {
  __shared__ double red[kAttnThreads * 4];
  const int h = blockIdx.x, quads = d / 4, groups = kAttnThreads / quads;
  const int dq = threadIdx.x % quads, grp = threadIdx.x / quads;
  const float* src = partial + (int64_t)h * splits * d + 4 * dq;
  if (grp < groups) {
    double t[4] = {0.0, 0.0, 0.0, 0.0};
    constexpr int kAhead = 8;
    for (int s0 = grp; s0 < splits; s0 += kAhead * groups) {
      float4 x[kAhead];
#pragma unroll
      for (int j = 0; j < kAhead; ++j)
        x[j] = *reinterpret_cast<const float4*>(src + (int64_t)min(s0 + j * groups, splits - 1) * d);
#pragma unroll
      for (int j = 0; j < kAhead; ++j)
        if (s0 + j * groups < splits) t[0] += x[j].x, t[1] += x[j].y, t[2] += x[j].z, t[3] += x[j].w;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) red[grp * d + 4 * dq + e] = t[e];
  }
  __syncthreads();
  if ((int)threadIdx.x < d) {
    double t = 0.0;
    for (int s = 0; s < groups; ++s) t += red[s * d + threadIdx.x];
    context[(int64_t)h * d + threadIdx.x] = to_bf(rkv((float)t, f16));  // the cache type's einsum result, then bfloat16
  }
}

// Scratch of klc_attn_decode past one window: scores [heads][count rounded
// up to 4], value partials [heads][splits][head_dim], then the score blocks'
// sums (float64) and maxima.
struct AttnPlan {
  int64_t cs, score_keys, nblk, split_keys, splits;
};
AttnPlan attn_plan(int64_t count) {
  AttnPlan a;
  a.cs = (count + 3) / 4 * 4;
  // 64 keys a score workgroup keep the chip busy on shorter contexts; larger
  // blocks leave fewer statistics for every value workgroup to read.  Core at
  // 12,000 keys with 64 / 128 / 256: 25.8 / 24.2 / 26.4 us, 16,384 30.6 /
  // 27.6 / 27.5, 32,768 48.6 / 42.7 / 42.9, 65,537 109 / 85.1 / 76.8, 131,072
  // 248 / 179 / 143, 262,144 719 / 480 / 350.
  a.score_keys = count <= 8192 ? 64 : count <= 65536 ? 128 : 256;
  a.nblk = (count + a.score_keys - 1) / a.score_keys;
  a.split_keys = count <= 8192 ? 128 : kPvKeys;  // 16,384 keys in splits of 128: 31.3 us against 27.6
  a.splits = (count + a.split_keys - 1) / a.split_keys;
  return a;
}

using ScoresKernel = void (*)(const uint16_t*, const uint16_t*, float*, float*, double*, int64_t, int64_t, int, int,
                              int, int, int, int, float, float, StepRecord);
template <int kC>
ScoresKernel pick_scores(int64_t keys, bool f16) {
  if (keys == 128) return f16 ? attn_scores_kernel<2, kC, true> : attn_scores_kernel<2, kC, false>;
  if (keys == 64) return f16 ? attn_scores_kernel<1, kC, true> : attn_scores_kernel<1, kC, false>;
  return f16 ? attn_scores_kernel<4, kC, true> : attn_scores_kernel<4, kC, false>;
}

using WindowKernel = void (*)(const uint16_t*, const uint16_t*, const uint16_t*, const uint16_t*, uint16_t*, int64_t,
                              int64_t, int, int, int, int, float, StepRecord);
// threads per key row: 256 threads over the window's keys
template <int kC>
WindowKernel pick_window(int n, bool f16) {
  if (n <= 64) return f16 ? attn_window_kernel<4, kC, true> : attn_window_kernel<4, kC, false>;
  if (n <= 128) return f16 ? attn_window_kernel<2, kC, true> : attn_window_kernel<2, kC, false>;
  return f16 ? attn_window_kernel<1, kC, true> : attn_window_kernel<1, kC, false>;
}

// Scores to context of one token (klc_attn_decode's kernels), with a step's
// record when rec.host is given.
int attn_core(const uint16_t* qb, const uint16_t* kb, const uint16_t* vb, const uint16_t* sk, int64_t cap,
              int64_t first, int n, int nh, int nkv, int d, bool f16, void* workspace, uint16_t* ctx,
              const StepRecord& rec, hipStream_t st) {
  const float sqrt_d = sqrtf((float)d);
  const unsigned extra = rec.host != nullptr ? 1 : 0;  // the record's workgroup (one per KV head in the score grid)
  if (n <= kPvKeys) {  // a window: one launch, one workgroup per query head
    auto run = d <= 64 ? pick_window<1>(n, f16) : pick_window<2>(n, f16);
    run<<<(unsigned)nh + extra, kAttnThreads, 0, st>>>(qb, kb, sk, vb, ctx, cap, first, n, nh, nkv, d, sqrt_d, rec);
    return check_launch("attn_window_kernel");
  }
  const AttnPlan a = attn_plan(n);
  float* scores = static_cast<float*>(workspace);
  float* partial = scores + (int64_t)nh * a.cs;
  double* stat_l = reinterpret_cast<double*>(partial + (int64_t)nh * a.splits * d);
  float* stat_m = reinterpret_cast<float*>(stat_l + (int64_t)nh * a.nblk);
  const dim3 sgrid((unsigned)nkv, (unsigned)a.nblk + extra), vgrid((unsigned)nkv, (unsigned)a.splits);
  auto run_scores = d <= 64 ? pick_scores<2>(a.score_keys, f16) : pick_scores<4>(a.score_keys, f16);
  run_scores<<<sgrid, kAttnThreads, 0, st>>>(qb, kb, scores, stat_m, stat_l, cap, first, n, (int)a.cs, (int)a.nblk,
                                             nh, nkv, d, sqrt_d, d == 16 || d == 64 ? 1.f / sqrt_d : 0.f, rec);
  int rc = check_launch("attn_scores_kernel");
  if (rc) return rc;
  auto run_pv = f16 ? attn_pv_kernel<true> : attn_pv_kernel<false>;
  run_pv<<<vgrid, kAttnThreads, 0, st>>>(scores, stat_m, stat_l, (int)a.nblk, sk, vb, partial, cap, first, n,
                                         (int)a.cs, a.split_keys == 128 ? 7 : 8, nh, nkv, d);
  if ((rc = check_launch("attn_pv_kernel"))) return rc;
  attn_combine_kernel<<<(unsigned)nh, kAttnThreads, 0, st>>>(partial, (int)a.splits, d, ctx, f16);
  return check_launch("attn_combine_kernel");
}

int64_t attn_bytes(int64_t n_heads, int64_t head_dim, int64_t count) {
  if (count <= kPvKeys) return 4 * n_heads * (count + head_dim);
  const AttnPlan a = attn_plan(count);
  return n_heads * (4 * a.cs + 12 * a.nblk + 4 * a.splits * head_dim);
}
// What a caller is told: the finest plan's bytes, which never shrink with the
// count, so a workspace made for a ring's capacity serves every shorter span
int64_t attn_bytes_up_to(int64_t n_heads, int64_t head_dim, int64_t count) {
  if (count <= kPvKeys) return 4 * n_heads * (count + head_dim);
  return n_heads * (4 * ((count + 3) / 4 * 4) + 12 * ((count + 63) / 64) + 4 * ((count + 127) / 128) * head_dim);
}

// Scratch of klc_attn_step before the core's: q and k before and after RoPE, the context
int64_t step_rows_bytes(int64_t nh, int64_t nkv, int64_t d) { return (2 * (2 * (nh + nkv) + nh) * d + 15) / 16 * 16; }

template <int J>
int launch_qkv(const QkvArgs& a, hipStream_t st) {
  const int waves = (a.nh + 2 * a.nkv) * (a.d / 2), per = kProjThreads / kWave;
  attn_qkv_kernel<J><<<(unsigned)((waves + per - 1) / per), kProjThreads, 0, st>>>(a);
  return check_launch("attn_qkv_kernel");
}

template <int J>
int launch_out(const uint16_t* w, const uint16_t* bias, const uint16_t* x, uint16_t* out, int rows, int k,
               hipStream_t st) {
  const int per = 2 * kProjThreads / kWave;
  attn_out_kernel<J><<<(unsigned)((rows + per - 1) / per), kProjThreads, 0, st>>>(w, bias, x, out, rows, k);
  return check_launch("attn_out_kernel");
}

}  // namespace
}  // namespace klc

using namespace klc;

extern "C" int klc_rope_append(const void* q, const void* k, const void* v, const void* cos_half,
                               const void* sin_half, void* q_out, void* k_out, void* k_cache, void* v_cache,
                               int64_t slot,
                               int64_t cap, int64_t n_heads, int64_t n_kv, int64_t head_dim, int kv_dtype,
                               void* stream) {
  KLC_REQUIRE(q && k && v && cos_half && sin_half && q_out && k_cache && v_cache, KLC_ERR_ARGUMENT,
              "klc_rope_append: null pointer");
  KLC_REQUIRE(n_heads > 0 && n_kv > 0 && head_dim > 0 && head_dim % 2 == 0 && head_dim <= kMaxHeadDim &&
                  n_heads % n_kv == 0 && n_heads <= 4096,
              KLC_ERR_SHAPE, "klc_rope_append: heads %lld / %lld, head_dim %lld", (long long)n_heads,
              (long long)n_kv, (long long)head_dim);
  KLC_REQUIRE(slot >= 0 && slot < cap, KLC_ERR_ARGUMENT, "klc_rope_append: slot %lld of %lld", (long long)slot,
              (long long)cap);
  KLC_REQUIRE(kv_dtype == KLC_DTYPE_BF16 || kv_dtype == KLC_DTYPE_F16, KLC_ERR_UNSUPPORTED,
              "klc_rope_append: kv_dtype %d (bfloat16 or float16)", kv_dtype);
  const int64_t items = (n_heads + n_kv) * (head_dim / 2) + n_kv * head_dim;  // one thread each
  rope_append_kernel<<<(unsigned)((items + kAttnThreads - 1) / kAttnThreads), kAttnThreads, 0, as_stream(stream)>>>(
      static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(k), static_cast<const uint16_t*>(v),
      static_cast<const uint16_t*>(cos_half), static_cast<const uint16_t*>(sin_half), static_cast<uint16_t*>(q_out),
      static_cast<uint16_t*>(k_out), static_cast<uint16_t*>(k_cache), static_cast<uint16_t*>(v_cache), slot, (int)n_heads, (int)n_kv,
      (int)head_dim, kv_dtype == KLC_DTYPE_F16);
  return check_launch("rope_append_kernel");
}

extern "C" int64_t klc_attn_workspace_bytes(int64_t n_heads, int64_t head_dim, int64_t count) {
  if (n_heads <= 0 || head_dim <= 0 || count <= 0)
    return set_error(KLC_ERR_ARGUMENT, "klc_attn_workspace_bytes: bad sizes");
  return attn_bytes_up_to(n_heads, head_dim, count);
}

extern "C" int klc_attn_decode(const void* q, const void* k_cache, const void* v_cache, const void* sinks,
                               int64_t cap, int64_t first, int64_t count, int64_t n_heads, int64_t n_kv,
                               int64_t head_dim, int kv_dtype, void* workspace, int64_t workspace_bytes,
                               void* context, void* stream) {
  KLC_REQUIRE(q && k_cache && v_cache && workspace && context, KLC_ERR_ARGUMENT, "klc_attn_decode: null pointer");
  KLC_REQUIRE(n_heads > 0 && n_kv > 0 && n_heads % n_kv == 0 && n_heads / n_kv <= kMaxGroup && head_dim >= 8 &&
                  head_dim % 8 == 0 && head_dim <= kMaxHeadDim,
              KLC_ERR_SHAPE, "klc_attn_decode: heads %lld / %lld (group <= %d), head_dim %lld (8..%d, multiple of 8)",
              (long long)n_heads, (long long)n_kv, kMaxGroup, (long long)head_dim, kMaxHeadDim);
  KLC_REQUIRE(cap > 0 && count > 0 && count <= cap && first >= 0 && first < cap && count <= (1 << 22) &&
                  n_heads * count < ((int64_t)1 << 31),
              KLC_ERR_ARGUMENT, "klc_attn_decode: %lld keys from slot %lld of a %lld-slot ring", (long long)count,
              (long long)first, (long long)cap);
  KLC_REQUIRE(((uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)workspace) % 16 == 0, KLC_ERR_ARGUMENT,
              "klc_attn_decode: caches and workspace must be 16-byte aligned");
  KLC_REQUIRE(kv_dtype == KLC_DTYPE_BF16 || kv_dtype == KLC_DTYPE_F16, KLC_ERR_UNSUPPORTED,
              "klc_attn_decode: kv_dtype %d (bfloat16 or float16)", kv_dtype);
  const bool f16 = kv_dtype == KLC_DTYPE_F16;
  const int64_t need = attn_bytes(n_heads, head_dim, count);
  KLC_REQUIRE(workspace_bytes >= need, KLC_ERR_ARGUMENT, "klc_attn_decode: workspace of %lld bytes, need %lld",
              (long long)workspace_bytes, (long long)need);
  return attn_core(static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(k_cache),
                   static_cast<const uint16_t*>(v_cache), static_cast<const uint16_t*>(sinks), cap, first, (int)count,
                   (int)n_heads, (int)n_kv, (int)head_dim, f16, workspace, static_cast<uint16_t*>(context),
                   StepRecord{}, as_stream(stream));
}

extern "C" int64_t klc_attn_step_workspace_bytes(int64_t n_heads, int64_t n_kv, int64_t head_dim, int64_t count) {
  if (n_heads <= 0 || n_kv <= 0 || head_dim <= 0 || count <= 0)
    return set_error(KLC_ERR_ARGUMENT, "klc_attn_step_workspace_bytes: bad sizes");
  return step_rows_bytes(n_heads, n_kv, head_dim) + attn_bytes_up_to(n_heads, head_dim, count);
}

extern "C" int klc_attn_step(const klc_attn_step_args* args, void* stream) {
  KLC_REQUIRE(args != nullptr, KLC_ERR_ARGUMENT, "klc_attn_step: null pointer");
  const klc_attn_step_args& a = *args;
  KLC_REQUIRE(a.hidden && a.q_weight && a.k_weight && a.v_weight && a.o_weight && a.inv_freq && a.k_cache &&
                  a.v_cache && a.workspace && a.out,
              KLC_ERR_ARGUMENT, "klc_attn_step: null pointer");
  const int64_t nh = a.n_heads, nkv = a.n_kv, d = a.head_dim, h = a.hidden_size;
  KLC_REQUIRE(nh > 0 && nkv > 0 && nh % nkv == 0 && nh / nkv <= kMaxGroup && d >= 8 && d % 8 == 0 &&
                  d <= kMaxHeadDim && nh * d <= kMaxRow && h > 0 && h % 8 == 0 && h <= kMaxRow && a.out_size > 0 &&
                  a.out_size < (1 << 30),
              KLC_ERR_SHAPE,
              "klc_attn_step: heads %lld / %lld (group <= %d) x %lld (8..%d, multiple of 8; at most %d in all), hidden "
              "%lld (a multiple of 8, at most %d), out %lld",
              (long long)nh, (long long)nkv, kMaxGroup, (long long)d, kMaxHeadDim, kMaxRow, (long long)h, kMaxRow,
              (long long)a.out_size);
  KLC_REQUIRE(a.cap > 0 && a.count > 0 && a.count <= a.cap && a.first >= 0 && a.first < a.cap &&
                  a.count <= (1 << 22) && nh * a.count < ((int64_t)1 << 31) && a.slot >= 0 && a.slot < a.cap,
              KLC_ERR_ARGUMENT, "klc_attn_step: slot %lld, %lld keys from slot %lld of a %lld-slot ring",
              (long long)a.slot, (long long)a.count, (long long)a.first, (long long)a.cap);
  KLC_REQUIRE(((uintptr_t)a.hidden | (uintptr_t)a.q_weight | (uintptr_t)a.k_weight | (uintptr_t)a.v_weight |
               (uintptr_t)a.o_weight | (uintptr_t)a.k_cache | (uintptr_t)a.v_cache | (uintptr_t)a.workspace) %
                      16 ==
                  0,
              KLC_ERR_ARGUMENT, "klc_attn_step: hidden, weights, caches and workspace must be 16-byte aligned");
  KLC_REQUIRE(a.kv_dtype == KLC_DTYPE_BF16 || a.kv_dtype == KLC_DTYPE_F16, KLC_ERR_UNSUPPORTED,
              "klc_attn_step: kv_dtype %lld (bfloat16 or float16)", (long long)a.kv_dtype);
  const int64_t need = step_rows_bytes(nh, nkv, d) + attn_bytes(nh, d, a.count);
  KLC_REQUIRE(a.workspace_bytes >= need, KLC_ERR_ARGUMENT, "klc_attn_step: workspace of %lld bytes, need %lld",
              (long long)a.workspace_bytes, (long long)need);
  StepRecord rec{};
  if (a.host_record != nullptr) {
    KLC_REQUIRE((uint32_t)a.tag != 0, KLC_ERR_ARGUMENT, "klc_attn_step: tag 0 (the caller clears the tag word to 0)");
    hipPointerAttribute_t attr;
    const hipError_t e = hipPointerGetAttributes(&attr, a.host_record);
    KLC_REQUIRE(e == hipSuccess && attr.devicePointer != nullptr, KLC_ERR_ARGUMENT,
                "klc_attn_step: host_record is not pinned host memory");
    rec.host = static_cast<uint32_t*>(attr.devicePointer);
    rec.tag = (uint32_t)a.tag;
  }
  hipStream_t st = as_stream(stream);
  uint16_t* pre = static_cast<uint16_t*>(a.workspace);
  uint16_t* rot = pre + (nh + nkv) * d;
  uint16_t* ctx = rot + (nh + nkv) * d;
  rec.pre = pre;
  rec.rot = rot;
  auto in = [](const void* p) { return static_cast<const uint16_t*>(p); };
  const bool f16 = a.kv_dtype == KLC_DTYPE_F16;
  const QkvArgs qkv{in(a.hidden), in(a.q_weight), in(a.q_bias), in(a.k_weight), in(a.k_bias), in(a.v_weight),
                    in(a.v_bias), static_cast<const float*>(a.inv_freq), pre, rot,
                    static_cast<uint16_t*>(a.k_cache), static_cast<uint16_t*>(a.v_cache), a.slot, (int)h, (int)nh,
                    (int)nkv, (int)d, (float)a.position, (float)a.rope_scale, f16};
  using QkvFn = int (*)(const QkvArgs&, hipStream_t);
  static constexpr QkvFn kQkv[] = {launch_qkv<1>, launch_qkv<2>, launch_qkv<3>, launch_qkv<4>,
                                   launch_qkv<5>, launch_qkv<6>, launch_qkv<7>, launch_qkv<8>};
  int rc = kQkv[(h / 8 + kWave - 1) / kWave - 1](qkv, st);
  if (rc) return rc;
  rc = attn_core(rot, in(a.k_cache), in(a.v_cache), in(a.sinks), a.cap, a.first, (int)a.count, (int)nh, (int)nkv,
                 (int)d, f16, static_cast<char*>(a.workspace) + step_rows_bytes(nh, nkv, d), ctx, rec, st);
  if (rc) return rc;
  using OutFn = int (*)(const uint16_t*, const uint16_t*, const uint16_t*, uint16_t*, int, int, hipStream_t);
  static constexpr OutFn kOut[] = {launch_out<1>, launch_out<2>, launch_out<3>, launch_out<4>,
                                   launch_out<5>, launch_out<6>, launch_out<7>, launch_out<8>};
  return kOut[(nh * d / 8 + kWave - 1) / kWave - 1](in(a.o_weight), in(a.o_bias), ctx, static_cast<uint16_t*>(a.out),
                                                    (int)a.out_size, (int)(nh * d), st);
}

extern "C" int klc_attn_step_wait(const void* host_record, int64_t tag, int64_t limit_us) {
  KLC_REQUIRE(host_record != nullptr && (uint32_t)tag != 0, KLC_ERR_ARGUMENT, "klc_attn_step_wait: no record or tag 0");
  const uint32_t* word = static_cast<const uint32_t*>(host_record) + 8;
  const auto begin = std::chrono::steady_clock::now();
  for (;;) {
    for (int i = 0; i < 256; ++i) {
      if (__atomic_load_n(word, __ATOMIC_ACQUIRE) == (uint32_t)tag) return 1;
      __builtin_ia32_pause();
    }
    if (std::chrono::steady_clock::now() - begin > std::chrono::microseconds(limit_us)) return 0;
  }
}
