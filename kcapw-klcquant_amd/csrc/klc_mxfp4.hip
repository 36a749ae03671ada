// MXFP4 -> dense dequant and checkpoint -> row-tile repack (gfx950).
//
// Dequant is HBM bound (1 byte of codes + 1/32 byte of scale in, 2 or 4 bytes
// out per value), and the transposed [in, out] output sets its pace: each
// output row is one input column of the checkpoint, so workgroups write runs
// of every output row they touch, of a length that follows the call's size,
// and there are enough of them for the chip however few matrices it has.
// Measured (new inputs and outputs every call) against one workgroup per 64
// output columns and all groups (and 768 columns x 4 groups for bfloat16 of
// 64-row multiples): 1 x 5760 x 90 groups to float16 25.4 -> 10.1 us, 16 x
// 2880 x 90 74 -> 64, 24 x 2880 x 90 116 -> 90, 57 x 4160 x 20 71.4 -> 73.1
// (58.3 -> 58.4 with a reused output), 57 x 4160 x 24 86.3 -> 86.1, 128 x 2880
// x 90 535 -> 458 (5.9 TB/s), to bfloat16 508 -> 458; 100 x 2880 x 90 to
// float32 1,412 -> 716 (5.2 TB/s, a copy's rate), 32 x 2881 x 90 to bfloat16
// 468 -> 176 (odd rows: one unaligned 16-byte store instead of eight 2-byte
// ones); packed, 1 x 5760 x 90 26.4 -> 9.3, 57 x 4160 x 20 70 -> 73.  Values
// come from gfx950's scaled E2M1 conversions
// (v_cvt_scalef32_pk_{bf16,f16,f32}_fp4), exact for every scale byte below
// 255; the MX NaN scale 255 takes an integer path (mxfp4_f32_bits) that
// reproduces the reference's +-inf / NaN.
#include <algorithm>
#include <type_traits>

#include "klc_common.h"

namespace klc {
namespace {

// Converts one exact float32 bit pattern to the output dtype's bits.
template <int kDtype>
__device__ __forceinline__ uint32_t to_out_bits(uint32_t f32bits) {
  if constexpr (kDtype == KLC_DTYPE_BF16) {
    return f32bits >> 16;  // every finite MXFP4 value is exact in bfloat16
  } else if constexpr (kDtype == KLC_DTYPE_F16) {
    return (uint32_t)__half_as_ushort(__float2half_rn(__uint_as_float(f32bits)));
  } else {
    return f32bits;
  }
}

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

// Elements 2q, 2q + 1 of the 8 codes in `word` times `scale`, as two 16-bit
// values packed low-first (bfloat16 or float16 per kDtype).
template <int kDtype>
__device__ __forceinline__ void cvt_word(uint32_t word, float scale, uint32_t (&pr)[4]) {
  if constexpr (kDtype == KLC_DTYPE_F16) {
    pr[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, scale, 0));
    pr[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, scale, 1));
    pr[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, scale, 2));
    pr[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, scale, 3));
  } else {
    pr[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, scale, 0));
    pr[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, scale, 1));
    pr[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, scale, 2));
    pr[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, scale, 3));
  }
}

// 2^(e - 127) of a scale byte below 255, exact (e = 0: the float32 subnormal)
__device__ __forceinline__ float scale_f32(uint32_t e) { return __uint_as_float(e == 0u ? 0x00400000u : (e << 23)); }

// One 16-byte piece of an output row: whole lines are streamed past the L2;
// at an odd row length the piece has element alignment only (one unaligned
// store) and shares its lines with its neighbours, so those stay in the L2.
template <bool kAligned>
__device__ __forceinline__ void store_piece(void* dst, u32x4_t v) {
  if constexpr (kAligned) {
    __builtin_nontemporal_store(v, static_cast<u32x4_t*>(dst));
  } else {
    typedef u32x4_t loose_t __attribute__((aligned(2)));
    *static_cast<loose_t*>(dst) = v;
  }
}

// MXFP4 -> dense [in, out]: workgroup (matrix, column block, part of the
// groups) stages up to kGroups groups' code chunks and scale bytes of up to
// kCols checkpoint rows (= output columns) in LDS, word-major (word w of row
// r at sw[w * kCols + r]), and writes its 32 x groups output rows at its
// columns.  In the checkpoint layout a row's chunks of the part are
// contiguous, and consecutive parts, which share a 128-byte line of each row,
// run in pairs side by side on one XCD (workgroups go to the XCDs
// round-robin), so that line is fetched once; in the packed layout a group's
// chunks of 64 rows are contiguous.  The pairs run on over matrices: pairs
// within a matrix leave half a pair idle at an odd number of parts (at 3
// parts, all on every other XCD: 60 x 512 x 77 groups to bfloat16 41.9 us
// against 38.4; 200,000 matrices of 1 x 1 1,860 against 953).  A task is 8 output rows (a band: one word of one group's
// chunks) x 16 bytes of output columns; the threads take consecutive tasks,
// so a task's 8 stores are, across the workgroup, runs of consecutive 16-byte
// pieces of output rows.  The scaled conversion (exact for every scale byte
// below 255) gives pairs of input elements of one row; v_perm_b32 pairs them
// up as pairs of columns.  Scale byte 255 (the MX NaN scale) is rare: those
// tasks are written again with the exact integer path (mxfp4_f32_bits) after
// the main loop, by the thread that wrote them (program order), so the main
// loop has no branch for it.

// Column block cb of nb over rows: nearly equal widths, multiples of 64 columns but for the last
__host__ __device__ inline int dq_col0(int rows, int nb, int cb) {
  const int col = (int)((int64_t)((rows + 63) / 64) * cb / nb) * 64;
  return col < rows ? col : rows;
}

template <int kDtype, bool kPacked, bool kAligned, int kThreads, int kCols, int kGroups>
__global__ __launch_bounds__(kThreads) void dequant_kernel(const uint8_t* __restrict__ blocks,
                                                           const uint8_t* __restrict__ scales, uint8_t* __restrict__ out,
                                                           int n_mat, int rows, int groups, int nb,
                                                           int64_t packed_stride) {
  constexpr int kElem = kDtype == KLC_DTYPE_F32 ? 4 : 2;
  constexpr int kPiece = 16 / kElem;                     // output columns of a 16-byte piece
  constexpr int kRounds = kCols * kGroups / kThreads;  // 16-byte loads per thread
  static_assert(kCols * kGroups % kThreads == 0, "whole load rounds");
  __shared__ __align__(16) uint32_t sw[4 * kGroups * kCols];
  __shared__ __align__(16) uint8_t ss[kGroups * kCols];
  // workgroup -> item (matrix, column block, part), numbered with the parts
  // innermost; items 2 i and 2 i + 1 are 8 workgroups apart in a window of 16
  const int parts = (groups + kGroups - 1) / kGroups;
  const int b = blockIdx.x;
  const int item = (b >> 4) * 16 + (b & 7) * 2 + ((b >> 3) & 1);
  if (item >= n_mat * nb * parts) return;
  const int mcb = item / parts;  // (matrix, column block)
  const int part = item - mcb * parts;
  const int m = mcb / nb;
  const int cb = mcb - m * nb;
  const int col0 = dq_col0(rows, nb, cb);
  const int ncols = dq_col0(rows, nb, cb + 1) - col0;
  // parts of nearly equal size (17 groups in parts of 8, 8 and 1 leave a third of the workgroups idle);
  // 4-group parts stay whole 64-byte runs
  const int g0 = kGroups > 4 ? (int)((int64_t)groups * part / parts) : part * kGroups;
  const int ng = (kGroups > 4 ? (int)((int64_t)groups * (part + 1) / parts) : min(groups, g0 + kGroups)) - g0;
  const int tid = threadIdx.x;
  // Load i of this thread is chunk c of row r; rows and groups past the end
  // read the last one again (the line is there already), so no load is
  // guarded.  Every load first, then the LDS writes.
  auto where = [&](int i, int& r, int& c) {
    const int idx = tid + i * kThreads;
    if constexpr (kPacked) {  // a wave reads one group's 64-row tile
      r = (idx & 63) + idx / (64 * kGroups) * 64;
      c = (idx >> 6) % kGroups;
    } else {
      r = idx / kGroups;
      c = idx % kGroups;
    }
  };
  u32x4_t v[kRounds];
  uint32_t e[kRounds];
#pragma unroll
  for (int i = 0; i < kRounds; ++i) {
    int r, c;
    where(i, r, c);
    r = col0 + min(r, ncols - 1);
    c = g0 + min(c, ng - 1);
    if constexpr (kPacked) {
      const uint8_t* mat = blocks + (int64_t)m * packed_stride;
      v[i] = *reinterpret_cast<const u32x4_t*>(mat + ((int64_t)(r / kTileRows) * groups + c) * 1024 + (r % kTileRows) * 16);
      e[i] = mat[packed_scale_offset(rows, groups, r, c)];
    } else {
      const int64_t chunk = ((int64_t)m * rows + r) * groups + c;
      v[i] = *reinterpret_cast<const u32x4_t*>(blocks + chunk * 16);
      e[i] = scales[chunk];
    }
  }
#pragma unroll
  for (int i = 0; i < kRounds; ++i) {
    int r, c;
    where(i, r, c);
    if (r < ncols) {
#pragma unroll
      for (int w = 0; w < 4; ++w) sw[(4 * c + w) * kCols + r] = v[i][w];
      ss[c * kCols + r] = (uint8_t)e[i];
    }
  }
  __syncthreads();

  const int ppr = (ncols + kPiece - 1) / kPiece;  // pieces per output run
  const int ntask = 4 * ng * ppr;
  const int64_t row_bytes = (int64_t)rows * kElem;
  uint8_t* obase = out + ((int64_t)m * groups + g0) * 32 * row_bytes + (int64_t)col0 * kElem;
  bool nan_scale = false;
  for (int t = tid; t < ntask; t += kThreads) {
    const int band = t / ppr;  // group band / 4, word band % 4
    const int pc = t - band * ppr;
    const uint32_t* wrow = sw + band * kCols + pc * kPiece;
    const uint8_t* srow = ss + (band >> 2) * kCols + pc * kPiece;
    uint8_t* o = obase + (int64_t)(8 * band) * row_bytes + pc * 16;
    u32x4_t row[8];
    if constexpr (kElem == 4) {
      const u32x4_t wa = *reinterpret_cast<const u32x4_t*>(wrow);
      const uint32_t sc4 = *reinterpret_cast<const uint32_t*>(srow);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t eb = (sc4 >> (8 * j)) & 0xffu;
        nan_scale |= eb == 255u;
        const float scale = scale_f32(eb);
        const f32x2_t p0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(wa[j], scale, 0);
        const f32x2_t p1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(wa[j], scale, 1);
        const f32x2_t p2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(wa[j], scale, 2);
        const f32x2_t p3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(wa[j], scale, 3);
        row[0][j] = __float_as_uint(p0.x), row[1][j] = __float_as_uint(p0.y);
        row[2][j] = __float_as_uint(p1.x), row[3][j] = __float_as_uint(p1.y);
        row[4][j] = __float_as_uint(p2.x), row[5][j] = __float_as_uint(p2.y);
        row[6][j] = __float_as_uint(p3.x), row[7][j] = __float_as_uint(p3.y);
      }
    } else {
      const u32x4_t wa = *reinterpret_cast<const u32x4_t*>(wrow);
      const u32x4_t wb = *reinterpret_cast<const u32x4_t*>(wrow + 4);
      const uint2 sc8 = *reinterpret_cast<const uint2*>(srow);
      const uint32_t word[8] = {wa[0], wa[1], wa[2], wa[3], wb[0], wb[1], wb[2], wb[3]};
      uint32_t pr[8][4];  // pr[j][q]: elements 2q, 2q + 1 of the band for column j
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t eb = ((j < 4 ? sc8.x : sc8.y) >> (8 * (j & 3))) & 0xffu;
        nan_scale |= eb == 255u;
        cvt_word<kDtype>(word[j], scale_f32(eb), pr[j]);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {  // output row i: half i % 2 of every column's pair i / 2, columns paired low-first
        const int q = i >> 1;
        const uint32_t sel = (i & 1) ? 0x07060302u : 0x05040100u;
        row[i] = u32x4_t{__builtin_amdgcn_perm(pr[1][q], pr[0][q], sel), __builtin_amdgcn_perm(pr[3][q], pr[2][q], sel),
                         __builtin_amdgcn_perm(pr[5][q], pr[4][q], sel), __builtin_amdgcn_perm(pr[7][q], pr[6][q], sel)};
      }
    }
    if (kAligned || (pc + 1) * kPiece <= ncols) {
#pragma unroll
      for (int i = 0; i < 8; ++i) store_piece<kAligned>(o + i * row_bytes, row[i]);
    } else {  // the last columns of an odd row length
#pragma unroll
      for (int j = 0; j < kPiece - 1; ++j) {
        if (pc * kPiece + j >= ncols) break;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if constexpr (kElem == 4)
            reinterpret_cast<uint32_t*>(o + i * row_bytes)[j] = row[i][j];
          else
            reinterpret_cast<uint16_t*>(o + i * row_bytes)[j] = (uint16_t)(row[i][j >> 1] >> (16 * (j & 1)));
        }
      }
    }
  }
  if (!__syncthreads_or(nan_scale)) return;
  // tasks with a scale byte 255, again with the integer path, by the same threads (same addresses,
  // program order: these stores land after the first ones)
  for (int t = tid; t < ntask; t += kThreads) {
    const int band = t / ppr;
    const int pc = t - band * ppr;
    uint8_t* o = obase + (int64_t)(8 * band) * row_bytes + pc * 16;
    for (int j = 0; j < min(kPiece, ncols - pc * kPiece); ++j) {
      const uint32_t eb = ss[(band >> 2) * kCols + pc * kPiece + j];
      if (eb != 255u) continue;
      const uint32_t word = sw[band * kCols + pc * kPiece + j];
      for (int i = 0; i < 8; ++i) {
        const uint32_t bits = to_out_bits<kDtype>(mxfp4_f32_bits((word >> (4 * i)) & 0xfu, eb));
        if constexpr (kElem == 4)
          reinterpret_cast<uint32_t*>(o + i * row_bytes)[j] = bits;
        else
          reinterpret_cast<uint16_t*>(o + i * row_bytes)[j] = (uint16_t)bits;
      }
    }
  }
}

// Checkpoint layout -> row-tile layout: one thread per (matrix, tile, group,
// row in tile) 16-byte chunk, writes coalesced; runs once per load.  The
// block and scale regions of matrix m start at out_blocks / out_scales +
// m * mat_stride, so a run of whole tiles can be packed into the middle of a
// larger matrix.
__global__ __launch_bounds__(256) void pack_blocks_kernel(const uint8_t* __restrict__ blocks,
                                                          uint8_t* __restrict__ out_blocks, int64_t n_mat, int rows,
                                                          int groups, int64_t mat_stride) {
  const int tiles = rows / kTileRows;
  const int64_t total = n_mat * tiles * groups * kTileRows;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int rr = (int)(idx % kTileRows);
    int64_t rest = idx / kTileRows;
    const int g = (int)(rest % groups);
    rest /= groups;
    const int tile = (int)(rest % tiles);
    const int64_t m = rest / tiles;
    const int r = tile * kTileRows + rr;
    const uint4 v = *reinterpret_cast<const uint4*>(blocks + ((m * rows + r) * groups + g) * 16);
    *reinterpret_cast<uint4*>(out_blocks + m * mat_stride + ((int64_t)tile * groups + g) * 1024 + rr * 16) = v;
  }
}

// Scale records: one thread per (matrix, row, quarter, step) byte, padding zero.
__global__ __launch_bounds__(256) void pack_scales_kernel(const uint8_t* __restrict__ scales,
                                                          uint8_t* __restrict__ out_scales, int64_t n_mat, int rows,
                                                          int groups, int64_t mat_stride) {
  // one thread per packed scale byte, in packed order: (matrix, tile, pair,
  // row in tile, quarter, byte); padding bytes (steps past the last group) are 0
  const int rec = (int)packed_scale_record(groups);
  const int64_t total = n_mat * rows * 4 * rec;
  const int64_t per_mat = (int64_t)rows * 4 * rec;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t m = idx / per_mat;
    int64_t rest = idx - m * per_mat;
    const int b = (int)(rest & 7);
    rest >>= 3;
    const int q = (int)(rest & 3);
    rest >>= 2;
    const int rr = (int)(rest % kTileRows);
    rest /= kTileRows;
    const int p = (int)(rest % (rec / 8));
    const int tile = (int)(rest / (rec / 8));
    const int r = tile * kTileRows + rr;
    const int g = 4 * (8 * p + b) + q;
    const uint8_t e = g < groups ? scales[(m * rows + r) * groups + g] : (uint8_t)0;
    out_scales[m * mat_stride + packed_scale_word(groups, r, p, q) + b] = e;
  }
}

// Packs one run of whole tiles read straight from pinned host memory (the
// GPU reads it over PCIe, so every read is 16 bytes per lane in source order:
// a wavefront reads 1 KiB of contiguous host memory).  Three grid-stride
// passes: block chunks (four loads in flight per thread before the four
// scattered 16-byte stores), scale bytes read 16 at a time and scattered
// (a row's 32 consecutive groups land in 32 contiguous bytes), and the zero
// bytes that pad each row's scale record.  rows * groups < 2^30.
__global__ __launch_bounds__(256) void pack_host_kernel(const uint8_t* __restrict__ blocks,
                                                        const uint8_t* __restrict__ scales,
                                                        uint8_t* __restrict__ out_blocks,
                                                        uint8_t* __restrict__ out_scales, int rows, int groups) {
  const int n = rows * groups;  // block chunks = scale bytes
  const int stride = (int)(gridDim.x * blockDim.x);
  const int tid = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const uint4* src = reinterpret_cast<const uint4*>(blocks);
  uint4* dst = reinterpret_cast<uint4*>(out_blocks);
  for (int base = tid; base < n; base += 4 * stride) {
    uint4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (base + k * stride < n) v[k] = src[base + k * stride];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = base + k * stride;
      if (i < n) {
        const int r = i / groups, g = i - r * groups;
        dst[((r / kTileRows) * groups + g) * kTileRows + (r % kTileRows)] = v[k];
      }
    }
  }
  const uint4* ssrc = reinterpret_cast<const uint4*>(scales);
  for (int j = tid; j < n / 16; j += stride) {
    const uint4 v = ssrc[j];
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    int r = (16 * j) / groups, g = 16 * j - r * groups;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int step = g >> 2;
      out_scales[packed_scale_word(groups, r, step >> 3, g & 3) + (step & 7)] = (uint8_t)(w[k >> 2] >> (8 * (k & 3)));
      if (++g == groups) {
        g = 0;
        ++r;
      }
    }
  }
  const int pad = 4 * (int)packed_scale_record(groups) - groups;
  for (int k = tid; k < rows * pad; k += stride) {
    const int r = k / pad, g = groups + (k - r * pad);
    const int step = g >> 2;
    out_scales[packed_scale_word(groups, r, step >> 3, g & 3) + (step & 7)] = 0;
  }
}

}  // namespace

int launch_pack_from_host(const uint8_t* blocks, const uint8_t* scales, uint8_t* out_blocks, uint8_t* out_scales,
                          int rows, int groups, hipStream_t st) {
  if (rows == 0) return KLC_OK;
  KLC_REQUIRE(rows % kTileRows == 0 && (int64_t)rows * groups < (int64_t)1 << 30 &&
                  (int64_t)rows * 4 * packed_scale_record(groups) < (int64_t)1 << 31,
              KLC_ERR_UNSUPPORTED, "pack_host_kernel: %d rows x %d groups in one run", rows, groups);
  // PCIe reads: a few hundred wavefronts with four 1 KiB reads each keep
  // enough bytes in flight; more workgroups only add contention (a plain
  // host-to-device copy kernel measured 51.7 GB/s at 64 workgroups, 40 at 512)
  const int64_t want = ((int64_t)rows * groups + 1023) / 1024;
  pack_host_kernel<<<(unsigned)std::min<int64_t>(128, std::max<int64_t>(1, want)), 256, 0, st>>>(
      blocks, scales, out_blocks, out_scales, rows, groups);
  return check_launch("pack_host_kernel");
}

int launch_pack(const uint8_t* blocks, const uint8_t* scales, uint8_t* out_blocks, uint8_t* out_scales, int64_t n_mat,
                int rows, int groups, int64_t mat_stride, hipStream_t st) {
  if (n_mat == 0 || rows == 0) return KLC_OK;
  const int64_t chunks = n_mat * rows * groups;
  const unsigned grid_b = (unsigned)((chunks + 255) / 256 < 65536 ? (chunks + 255) / 256 : 65536);
  pack_blocks_kernel<<<grid_b, 256, 0, st>>>(blocks, out_blocks, n_mat, rows, groups, mat_stride);
  const int rc = check_launch("pack_blocks_kernel");
  if (rc) return rc;
  const int64_t bytes = n_mat * rows * 4 * packed_scale_record(groups);
  const unsigned grid_s = (unsigned)((bytes + 255) / 256 < 65536 ? (bytes + 255) / 256 : 65536);
  pack_scales_kernel<<<grid_s, 256, 0, st>>>(scales, out_scales, n_mat, rows, groups, mat_stride);
  return check_launch("pack_scales_kernel");
}

namespace {

// One launch: workgroups of kThreads over nb column blocks of at most kCols
// columns and parts of at most kGroups groups.
template <int kDtype, bool kPacked, bool kAligned, int kThreads, int kCols, int kGroups>
int launch_dequant_shape(const uint8_t* blocks, const uint8_t* scales, uint8_t* out, int64_t n_mat, int64_t rows,
                         int64_t groups, int64_t packed_stride, hipStream_t stream) {
  const int64_t parts = (groups + kGroups - 1) / kGroups;
  // narrower blocks (down to 128 columns) until there are 768 workgroups
  const int64_t least = (rows + kCols - 1) / kCols, most = std::max(least, rows / 128);
  const int64_t nb = std::clamp((768 + n_mat * parts - 1) / (n_mat * parts), least, most);
  const int64_t grid = (n_mat * nb * parts + 15) / 16 * 16;
  KLC_REQUIRE(grid <= 0x7fffffff, KLC_ERR_UNSUPPORTED, "dequant: too many matrices (%lld)", (long long)n_mat);
  dequant_kernel<kDtype, kPacked, kAligned, kThreads, kCols, kGroups><<<(unsigned)grid, kThreads, 0, stream>>>(
      blocks, scales, out, (int)n_mat, (int)rows, (int)groups, (int)nb, packed_stride);
  return check_launch("dequant_kernel");
}

// The workgroup shape, columns x groups.  What decides is how much of a call's
// input and output the 256 MB memory-side cache holds from call to call, so
// each figure is given for new inputs and a reused output (as an allocator
// gives it) / for new inputs and outputs, us.  16-bit outputs of aligned rows:
// 64 x 16 up to 400 MB (whole 256-byte pieces of each row), 128 x 8 on 512
// threads up to 1 GB, then 128 x 4.
//   matrices x rows x groups   64 x 16        128 x 8        128 x 4
//     8 x 2880 x 90 (168 MB)   29.1 / 33.4    29.7 / 32.6    31.6 / 33.0
//    57 x 4160 x 17 (327 MB)   51.1 / 62.3    55.3 / 56.7    60.7 / 60.8
//   100 x 2048 x 26 (431 MB)   71.7 / 81.5    71.0 / 75.1    75.9 / 75.2
//    24 x 2880 x 90 (504 MB)   92.6 / 97.5    86.5 / 90.1    88.9 / 89.9
//    38 x 3840 x 56 (662 MB)    130 / 128      126 / 124      123 / 122
//    48 x 2880 x 90 (1.0 GB)    198 / 194      177 / 177      174 / 176
//    64 x 2880 x 90 (1.3 GB)    265 / 264      237 / 238      230 / 235
//   128 x 2880 x 90 (2.7 GB)    531 / 529      482 / 481      455 / 455
// 256 x 4 is never more than 8 % from the best with new outputs, but 20 % at
// 57 x 4160 x 17 with a reused one (61.2).  float32 (its runs are twice as
// long): 384 x 4.  Odd row lengths want long runs, since each run's ends share
// lines with its neighbours': 1024 x 4 once that gives 1200 workgroups (384 x
// 4 / 1024 x 4: 93 x 3709 x 65 474 / 444, 48 x 1601 x 83 147 / 136, 25 x 2278
// x 67, 1,275 workgroups, 85.5 / 81.9; 28 x 3627 x 19 to float32, 560, alike),
// but not where its columns stand empty (1000 x 101 x 30 78 / 86; 500 x 201 x
// 33 to float32 106 / 93; 200,000 x 1 x 1 332 / 953).
template <int kDtype, bool kPacked>
int launch_dequant_as(const uint8_t* blocks, const uint8_t* scales, uint8_t* out, int64_t n_mat, int64_t rows,
                      int64_t groups, int64_t packed_stride, hipStream_t stream) {
  if constexpr (!kPacked) {  // packed matrices have whole 64-row tiles
    if (rows % (kDtype == KLC_DTYPE_F32 ? 4 : 8) != 0) {
      if (rows >= 192 && n_mat * ((groups + 3) / 4) * ((rows + 1023) / 1024) >= 1200)
        return launch_dequant_shape<kDtype, false, false, 512, 1024, 4>(blocks, scales, out, n_mat, rows, groups, 0,
                                                                        stream);
      return launch_dequant_shape<kDtype, false, false, 256, 384, 4>(blocks, scales, out, n_mat, rows, groups, 0,
                                                                     stream);
    }
  }
  if constexpr (kDtype == KLC_DTYPE_F32) {
    return launch_dequant_shape<kDtype, kPacked, true, 256, 384, 4>(blocks, scales, out, n_mat, rows, groups,
                                                                    packed_stride, stream);
  } else {
    const int64_t bytes = n_mat * rows * groups * (17 + 64);
    if (bytes >= (int64_t)1 << 30)
      return launch_dequant_shape<kDtype, kPacked, true, 256, 128, 4>(blocks, scales, out, n_mat, rows, groups,
                                                                      packed_stride, stream);
    if (bytes >= (int64_t)400 << 20)
      return launch_dequant_shape<kDtype, kPacked, true, 512, 128, 8>(blocks, scales, out, n_mat, rows, groups,
                                                                      packed_stride, stream);
    return launch_dequant_shape<kDtype, kPacked, true, 256, 64, 16>(blocks, scales, out, n_mat, rows, groups,
                                                                    packed_stride, stream);
  }
}

template <bool kPacked>
int launch_dequant(const void* blocks, const void* scales, void* out, int64_t n_mat, int64_t rows, int64_t groups,
                   int dtype, int64_t packed_stride, hipStream_t stream) {
  const auto* b = static_cast<const uint8_t*>(blocks);
  const auto* s = static_cast<const uint8_t*>(scales);
  auto* o = static_cast<uint8_t*>(out);
  switch (dtype) {
    case KLC_DTYPE_BF16:
      return launch_dequant_as<KLC_DTYPE_BF16, kPacked>(b, s, o, n_mat, rows, groups, packed_stride, stream);
    case KLC_DTYPE_F16:
      return launch_dequant_as<KLC_DTYPE_F16, kPacked>(b, s, o, n_mat, rows, groups, packed_stride, stream);
    case KLC_DTYPE_F32:
      return launch_dequant_as<KLC_DTYPE_F32, kPacked>(b, s, o, n_mat, rows, groups, packed_stride, stream);
    default:
      return set_error(KLC_ERR_ARGUMENT, "dequant: unknown dtype %d", dtype);
  }
}

}  // namespace
}  // namespace klc

using namespace klc;

extern "C" int klc_mxfp4_dequant(const void* blocks, const void* scales, void* out, int64_t n_mat, int64_t out_dim,
                                 int64_t groups, int out_dtype, void* stream) {
  KLC_REQUIRE(blocks && scales && out, KLC_ERR_ARGUMENT, "klc_mxfp4_dequant: null pointer");
  KLC_REQUIRE(n_mat >= 0 && out_dim > 0 && groups > 0, KLC_ERR_ARGUMENT,
              "klc_mxfp4_dequant: bad sizes n_mat=%lld out_dim=%lld groups=%lld", (long long)n_mat,
              (long long)out_dim, (long long)groups);
  KLC_REQUIRE(out_dim < (1 << 30) && groups < (1 << 24), KLC_ERR_UNSUPPORTED, "klc_mxfp4_dequant: matrix too large");
  if (n_mat == 0) return KLC_OK;
  return launch_dequant<false>(blocks, scales, out, n_mat, out_dim, groups, out_dtype, 0, as_stream(stream));
}

extern "C" int64_t klc_mxfp4_packed_bytes(int64_t out_dim, int64_t groups) {
  if (out_dim <= 0 || groups <= 0)
    return set_error(KLC_ERR_ARGUMENT, "klc_mxfp4_packed_bytes: bad sizes out_dim=%lld groups=%lld",
                     (long long)out_dim, (long long)groups);
  if (out_dim % kTileRows)
    return set_error(KLC_ERR_SHAPE, "klc_mxfp4_packed_bytes: out_dim=%lld is not a multiple of %d",
                     (long long)out_dim, kTileRows);
  return packed_matrix_bytes(out_dim, groups);
}

extern "C" int klc_mxfp4_pack(const void* blocks, const void* scales, void* packed, int64_t n_mat, int64_t out_dim,
                              int64_t groups, void* stream) {
  KLC_REQUIRE(blocks && scales && packed, KLC_ERR_ARGUMENT, "klc_mxfp4_pack: null pointer");
  const int64_t stride = klc_mxfp4_packed_bytes(out_dim, groups);
  if (stride < 0) return (int)stride;
  KLC_REQUIRE(n_mat >= 0, KLC_ERR_ARGUMENT, "klc_mxfp4_pack: n_mat=%lld", (long long)n_mat);
  KLC_REQUIRE(out_dim < (1 << 30) && groups < (1 << 24), KLC_ERR_UNSUPPORTED, "klc_mxfp4_pack: matrix too large");
  uint8_t* out = static_cast<uint8_t*>(packed);
  return launch_pack(static_cast<const uint8_t*>(blocks), static_cast<const uint8_t*>(scales), out,
                     out + packed_block_bytes(out_dim, groups), n_mat, (int)out_dim, (int)groups, stride,
                     as_stream(stream));
}

extern "C" int klc_mxfp4_dequant_packed(const void* packed, void* out, int64_t n_mat, int64_t out_dim,
                                        int64_t groups, int out_dtype, void* stream) {
  KLC_REQUIRE(packed && out, KLC_ERR_ARGUMENT, "klc_mxfp4_dequant_packed: null pointer");
  const int64_t stride = klc_mxfp4_packed_bytes(out_dim, groups);
  if (stride < 0) return (int)stride;
  KLC_REQUIRE(n_mat >= 0, KLC_ERR_ARGUMENT, "klc_mxfp4_dequant_packed: n_mat=%lld", (long long)n_mat);
  KLC_REQUIRE(out_dim < (1 << 30) && groups < (1 << 24), KLC_ERR_UNSUPPORTED,
              "klc_mxfp4_dequant_packed: matrix too large");
  if (n_mat == 0) return KLC_OK;
  return launch_dequant<true>(packed, packed, out, n_mat, out_dim, groups, out_dtype, stride, as_stream(stream));
}
