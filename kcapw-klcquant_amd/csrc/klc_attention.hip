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
// head x 64 or 256 keys, its whole query group), probabilities x values
// (workgroup = one KV head x 128 or 256 keys), and the sum of the splits; a
// window of at most 256 keys runs as one launch, scores to context, one
// workgroup per query head.  Measured for 64 / 8 heads x 64, float16 (cold
// rings): 4,096 keys 23.7 -> 17.6 us, 8,192 40.2 -> 21.2, 16,384 81.6 ->
// 29.8, 32,768 200 -> 43.2 against value workgroups per query head that each
// took their head's statistics over all its scores (quadratic in the
// context: 186 of the 200 us) and vector float64 dot products per query head
// (38 us -> 20).
#include <math.h>

#include "klc_common.h"

namespace klc {
namespace {

constexpr int kAttnThreads = 256;
constexpr int kPvKeys = 256;     // most keys of a value workgroup, and of a one-launch window
constexpr int kMaxHeadDim = 128;
constexpr int kMaxGroup = 16;    // query heads per KV head
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

// Query head h's m = max(scores, sink) and l = sum exp(x - m) over [scores,
// sink], l summed in float64 and rounded once; each reduction is a wave
// shuffle tree plus one exchange of the 4 waves' values.  Every thread of
// the workgroup calls it and gets both.
__device__ __forceinline__ void head_stats(const float* __restrict__ s, int count, const uint16_t* __restrict__ sinks,
                                           int h, float& m_out, float& l_out) {
  __shared__ float wm[kAttnThreads / kWave];
  __shared__ double wl[kAttnThreads / kWave];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  // both passes issue 8 loads before using them (a thread's scores are
  // otherwise a chain of dependent L2 round trips); the sum keeps the
  // thread's order i, i + 256, ...
  constexpr int kAhead = 8;
  float m = sinks != nullptr ? bf(sinks[h]) : -INFINITY;
  int i = threadIdx.x;
  for (; i + (kAhead - 1) * kAttnThreads < count; i += kAhead * kAttnThreads) {
    float x[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) x[j] = s[i + j * kAttnThreads];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) m = fmaxf(m, x[j]);
  }
  for (; i < count; i += kAttnThreads) m = fmaxf(m, s[i]);
  for (int off = kWave / 2; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  if (lane == 0) wm[wave] = m;
  __syncthreads();
  m = wm[0];
  for (int w = 1; w < kAttnThreads / kWave; ++w) m = fmaxf(m, wm[w]);
  double l = 0.0;
  i = threadIdx.x;
  for (; i + (kAhead - 1) * kAttnThreads < count; i += kAhead * kAttnThreads) {
    float x[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) x[j] = s[i + j * kAttnThreads];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) l += (double)expf(x[j] - m);
  }
  for (; i < count; i += kAttnThreads) l += (double)expf(s[i] - m);
  if (threadIdx.x == 0 && sinks != nullptr) l += (double)expf(bf(sinks[h]) - m);
  for (int off = kWave / 2; off > 0; off >>= 1) l += __shfl_xor(l, off);
  if (lane == 0) wl[wave] = l;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < kAttnThreads / kWave; ++w) t += wl[w];
  m_out = m;
  l_out = (float)t;
}

// The value half of a window workgroup: the context of query head
// h = blockIdx.x whose `count` <= 256 scores s_head (LDS) holds; p rounded to
// the cache type, the slices' float32 sums in `partial` [h][d].
__device__ __forceinline__ void pv_body(const float* __restrict__ s_head, const uint16_t* __restrict__ sinks,
                                        const uint16_t* __restrict__ v_cache, float* __restrict__ partial,
                                        uint16_t* __restrict__ context, int64_t cap, int64_t first, int count, int nh,
                                        int nkv, int d, bool f16) {
  __shared__ float p[kPvKeys];
  __shared__ float acc_s[kAttnThreads / 32][kMaxHeadDim];
  const int h = blockIdx.x, g = nh / nkv, kvh = h / g;
  const int nk = count;
  float m, l;
  head_stats(s_head, count, sinks, h, m, l);
  for (int i = threadIdx.x; i < nk; i += kAttnThreads) p[i] = rkv(expf(s_head[i] - m) / l, f16);
  __syncthreads();
  // thread (slice, four dims): slices of keys; each thread issues the 8-byte
  // loads of four keys before their multiply-adds, so L2 round trips overlap
  const int quads = d / 4, slices = kAttnThreads / quads;
  const int dq = threadIdx.x % quads, sl = threadIdx.x / quads;
  float a[4] = {0.f, 0.f, 0.f, 0.f};
  auto vrow = [&](int i) {
    return *reinterpret_cast<const uint2*>(v_cache + (((first + i) % cap) * nkv + kvh) * d + 4 * dq);
  };
  auto add = [&](float pi, uint2 w) {
    a[0] = fmaf(pi, kv_f((uint16_t)(w.x & 0xffffu), f16), a[0]);
    a[1] = fmaf(pi, kv_f((uint16_t)(w.x >> 16), f16), a[1]);
    a[2] = fmaf(pi, kv_f((uint16_t)(w.y & 0xffffu), f16), a[2]);
    a[3] = fmaf(pi, kv_f((uint16_t)(w.y >> 16), f16), a[3]);
  };
  if (sl < slices) {
    int i = sl;
    for (; i + 3 * slices < nk; i += 4 * slices) {
      const uint2 w0 = vrow(i), w1 = vrow(i + slices), w2 = vrow(i + 2 * slices), w3 = vrow(i + 3 * slices);
      add(p[i], w0);
      add(p[i + slices], w1);
      add(p[i + 2 * slices], w2);
      add(p[i + 3 * slices], w3);
    }
    for (; i < nk; i += slices) add(p[i], vrow(i));
  }
  // sum the slices, kAttnThreads / 32 of them at a time through LDS
  for (int base = 0; base < slices; base += kAttnThreads / 32) {
    if (sl >= base && sl < base + kAttnThreads / 32) {
#pragma unroll
      for (int e = 0; e < 4; ++e) acc_s[sl - base][4 * dq + e] = a[e];
    }
    __syncthreads();
    if ((int)threadIdx.x < d) {
      float t = 0.f;
      for (int s2 = 0; s2 < min(kAttnThreads / 32, slices - base); ++s2) t += acc_s[s2][threadIdx.x];
      float* out = partial + (int64_t)h * d + threadIdx.x;
      *out = base == 0 ? t : *out + t;
    }
    __syncthreads();
  }
  if ((int)threadIdx.x < d)
    context[(int64_t)h * d + threadIdx.x] = to_bf(rkv(partial[(int64_t)h * d + threadIdx.x], f16));
}

// A window of at most 256 keys in one launch: workgroup = query head
// blockIdx.x.  Its scores (the same float64 dot products as
// attn_scores_kernel, one key per thread) go to LDS, then the value body
// takes the max, the sum and the context.
__global__ __launch_bounds__(kAttnThreads) void attn_window_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_cache, const uint16_t* __restrict__ sinks,
    const uint16_t* __restrict__ v_cache, float* __restrict__ partial, uint16_t* __restrict__ context, int64_t cap,
    int64_t first, int count, int nh, int nkv, int d, float sqrt_d, bool f16) {
  __shared__ float qs[kMaxHeadDim];
  __shared__ float sc[kPvKeys];
  const int h = blockIdx.x, kvh = h / (nh / nkv);
  const int key = threadIdx.x;
  const bool live = key < count;
  uint4 kr[kMaxHeadDim / 8] = {};
  const uint16_t* krow = k_cache + (((first + (live ? key : 0)) % cap) * nkv + kvh) * d;
#pragma unroll
  for (int c = 0; c < kMaxHeadDim / 8; ++c)
    if (live && c * 8 < d) kr[c] = *reinterpret_cast<const uint4*>(krow + c * 8);
  for (int i = threadIdx.x; i < d; i += blockDim.x) qs[i] = bf(q[(int64_t)h * d + i]);
  __syncthreads();
  if (live) {
    double acc = 0.0;
#pragma unroll
    for (int c = 0; c < kMaxHeadDim / 8; ++c) {
      if (c * 8 >= d) break;
      const uint32_t wd[4] = {kr[c].x, kr[c].y, kr[c].z, kr[c].w};
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        acc = fma((double)kv_f((uint16_t)(wd[t] & 0xffffu), f16), (double)qs[8 * c + 2 * t], acc);
        acc = fma((double)kv_f((uint16_t)(wd[t] >> 16), f16), (double)qs[8 * c + 2 * t + 1], acc);
      }
    }
    sc[key] = (float)acc / sqrt_d;
  }
  __syncthreads();
  pv_body(sc, sinks, v_cache, partial, context, cap, first, count, nh, nkv, d, f16);
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
template <int T, bool kF16>
__global__ __launch_bounds__(kAttnThreads) void attn_scores_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_cache, float* __restrict__ scores,
    float* __restrict__ stat_m, double* __restrict__ stat_l, int64_t cap, int64_t first, int count, int cs, int nh,
    int nkv, int d, float sqrt_d) {
  __shared__ __align__(16) uint16_t qs[kMaxGroup][kMaxHeadDim + 8];
  __shared__ float wm[kAttnThreads / kWave][kMaxGroup];
  __shared__ double wl[kAttnThreads / kWave][kMaxGroup];
  const int g = nh / nkv, kvh = blockIdx.x, blk = blockIdx.y;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int r = lane & 15, kq = lane >> 4;  // MFMA row / column, dim quarter
  const int key0 = (blk * (kAttnThreads / kWave) + wave) * 16 * T;
  constexpr int kC = kMaxHeadDim / 32;
  // dims 32 c + 8 kq of the head exist: d is a multiple of 8
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
      s[t][i] = (float)acc[t][i] / sqrt_d;
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
    const int64_t at = (int64_t)h * gridDim.y + blk;
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

  // 16 to 256 lanes a head take its statistics, every head at once
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
#pragma unroll 4
  for (int i = threadIdx.x; i < ks * 4 * hb; i += kAttnThreads) {
    const int hh = i >> ks_log2, key = i & (ks - 1);
    float w = 0.f;
    if (hh < g && key < nk)
      w = rkv(expf(scores[(int64_t)(kvh * g + hh) * cs + k0 + key] - head_m[hh]) / head_l[hh], kF16);
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
  // 64 keys a workgroup keep the chip busy on shorter contexts; past 8,192
  // keys 256 (fewer block statistics for every value workgroup to read)
  a.score_keys = count <= 8192 ? 64 : 256;
  a.nblk = (count + a.score_keys - 1) / a.score_keys;
  a.split_keys = count <= 8192 ? 128 : kPvKeys;
  a.splits = (count + a.split_keys - 1) / a.split_keys;
  return a;
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
  if (count <= kPvKeys) return 4 * n_heads * (count + head_dim);
  const AttnPlan a = attn_plan(count);
  return n_heads * (4 * a.cs + 12 * a.nblk + 4 * a.splits * head_dim);
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
  const int64_t need = klc_attn_workspace_bytes(n_heads, head_dim, count);
  KLC_REQUIRE(workspace_bytes >= need, KLC_ERR_ARGUMENT, "klc_attn_decode: workspace of %lld bytes, need %lld",
              (long long)workspace_bytes, (long long)need);
  hipStream_t st = as_stream(stream);
  const uint16_t* qb = static_cast<const uint16_t*>(q);
  const uint16_t* kb = static_cast<const uint16_t*>(k_cache);
  const uint16_t* vb = static_cast<const uint16_t*>(v_cache);
  const uint16_t* sk = static_cast<const uint16_t*>(sinks);
  uint16_t* ctx = static_cast<uint16_t*>(context);
  const float sqrt_d = sqrtf((float)head_dim);
  const int n = (int)count, nh = (int)n_heads, nkv = (int)n_kv, d = (int)head_dim;
  if (count <= kPvKeys) {  // a window: one launch, one workgroup per query head
    static_assert(kPvKeys == kAttnThreads, "one key per thread");
    attn_window_kernel<<<(unsigned)n_heads, kAttnThreads, 0, st>>>(
        qb, kb, sk, vb, static_cast<float*>(workspace), ctx, cap, first, n, nh, nkv, d, sqrt_d, f16);
    return check_launch("attn_window_kernel");
  }
  const AttnPlan a = attn_plan(count);
  float* scores = static_cast<float*>(workspace);
  float* partial = scores + n_heads * a.cs;
  double* stat_l = reinterpret_cast<double*>(partial + n_heads * a.splits * head_dim);
  float* stat_m = reinterpret_cast<float*>(stat_l + n_heads * a.nblk);
  const dim3 sgrid((unsigned)n_kv, (unsigned)a.nblk), vgrid((unsigned)n_kv, (unsigned)a.splits);
  auto run_scores = a.score_keys == 64 ? (f16 ? attn_scores_kernel<1, true> : attn_scores_kernel<1, false>)
                                       : (f16 ? attn_scores_kernel<4, true> : attn_scores_kernel<4, false>);
  run_scores<<<sgrid, kAttnThreads, 0, st>>>(qb, kb, scores, stat_m, stat_l, cap, first, n, (int)a.cs, nh, nkv, d,
                                             sqrt_d);
  int rc = check_launch("attn_scores_kernel");
  if (rc) return rc;
  auto run_pv = f16 ? attn_pv_kernel<true> : attn_pv_kernel<false>;
  run_pv<<<vgrid, kAttnThreads, 0, st>>>(scores, stat_m, stat_l, (int)a.nblk, sk, vb, partial, cap, first, n,
                                         (int)a.cs, a.split_keys == 128 ? 7 : 8, nh, nkv, d);
  if ((rc = check_launch("attn_pv_kernel"))) return rc;
  attn_combine_kernel<<<(unsigned)n_heads, kAttnThreads, 0, st>>>(partial, (int)a.splits, d, ctx, f16);
  return check_launch("attn_combine_kernel");
}
