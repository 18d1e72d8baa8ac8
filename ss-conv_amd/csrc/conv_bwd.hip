// Filter gradient of the sparse convolution:
//   dW[k][ci][co] = sum over the pairs (i, o) of offset k of feat[i][ci] * dout[o][co]
// (reference: src/conv/indice_conv.h:344-426, the torch::mm_out(filterGradSub, ...)
// of every offset).  The input gradient needs no kernel of its own: it is the forward
// convolution of dout with the pairs swapped and the filters transposed.
//
// Per offset this is a tall-skinny product [Cin x P_k] * [P_k x Cout].  A workgroup owns one
// offset, one 64 x 64 tile of (ci, co) and one contiguous range of the offset's pairs.  Which
// pair sits in which k slot of a matrix instruction does not matter for the sum, and neither
// does which channel a lane stands for, as long as the result is stored accordingly: lane l of
// channel block j stands for channel 4l + j, so one 16-byte read of a row hands a lane its
// operands for all four channel blocks.  Every wave keeps the whole 64 x 64 tile (16
// independent accumulators) over a quarter of the pairs; the four waves' tiles are added in
// wave order at the end, and the ranges of pairs by a second kernel in ascending order: the
// result does not depend on timing, no atomics.
//
// conv_bwd_filter_parts_kernel takes output rows of four channels or more and matrices with
// 31-bit offsets; conv_bwd_filter_kernel takes the rest: it gathers 64 pairs at a time into LDS,
// rows as they lie in memory, and multiplies with float instructions.
#include "ssc_common.h"

#include <algorithm>
#include <type_traits>

namespace ssc {

typedef float float4v __attribute__((ext_vector_type(4)));

constexpr int kBwChunk = 64;    // pairs per LDS stage
constexpr int kBwStride = 68;   // floats per channel row in LDS (64 pairs + 4)
constexpr int kBwTile = 64;     // channels per tile side

// Rows of float or half-precision elements; the products and sums are fp32 either way
// (half rows are widened when they are staged in LDS).
typedef int int2v __attribute__((ext_vector_type(2)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4v widen4(const float4v &v) { return v; }
__device__ __forceinline__ float4v widen4(const int2v &v) {
  return __builtin_convertvector(__builtin_bit_cast(half4v, v), float4v);
}
__device__ __forceinline__ float4v load4(const float *p) {
  return *reinterpret_cast<const float4v *>(p);
}
__device__ __forceinline__ float4v load4(const _Float16 *p) {
  return widen4(*reinterpret_cast<const int2v *>(p));
}
// four channels at byte offset `off` of a buffer, as loaded
__device__ __forceinline__ float4v buf_quad(__amdgpu_buffer_rsrc_t r, unsigned off, const float *) {
  return __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}
__device__ __forceinline__ int2v buf_quad(__amdgpu_buffer_rsrc_t r, unsigned off,
                                          const _Float16 *) {
  return __builtin_bit_cast(int2v, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}

// one channel, as loaded, and an element of a quad or of one channel as a float
__device__ __forceinline__ float buf_one(__amdgpu_buffer_rsrc_t r, unsigned off, const float *) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}
__device__ __forceinline__ _Float16 buf_one(__amdgpu_buffer_rsrc_t r, unsigned off,
                                            const _Float16 *) {
  return __builtin_bit_cast(_Float16, __builtin_amdgcn_raw_buffer_load_b16(r, (int)off, 0, 0));
}
__device__ __forceinline__ float element(const float4v &v, int c) { return v[c]; }
__device__ __forceinline__ float element(const int2v &v, int c) { return widen4(v)[c]; }
__device__ __forceinline__ float element(float v, int) { return v; }
__device__ __forceinline__ float element(_Float16 v, int) { return (float)v; }

// Four channels of row `row`, zero outside the matrix.
template <typename IO>
__device__ __forceinline__ float4v load_quad(const IO *__restrict__ m, int64_t row, int ch,
                                             int width) {
  float4v v = {0.f, 0.f, 0.f, 0.f};
  if (row < 0) return v;
  const IO *p = m + row * width + ch;
  if ((width & 3) == 0) {
    if (ch < width) v = load4(p);
  } else {
    if (ch + 0 < width) v.x = (float)p[0];
    if (ch + 1 < width) v.y = (float)p[1];
    if (ch + 2 < width) v.z = (float)p[2];
    if (ch + 3 < width) v.w = (float)p[3];
  }
  return v;
}

// grid: x = range of pairs, y = offset k, z = tile (ci tile major).  256 threads, four
// workgroups per CU (one wave of each per SIMD: 128 registers a wave).
// BUF: rows are multiples of four channels and both matrices are below 4 GiB, so the gathers
// are range-checked buffer loads at 32-bit byte offsets (a row beyond the range's pairs
// gets an offset outside the buffer and reads zeros): no 64-bit address arithmetic and
// no branches around the loads.
template <typename IO, bool BUF>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4)))
    conv_bwd_filter_kernel(const IO *__restrict__ feats, int cin, unsigned feat_bytes,
                           const IO *__restrict__ dout, int cout, unsigned dout_bytes,
                           const int32_t *__restrict__ pairs, int64_t pair_stride,
                           const int32_t *__restrict__ pair_num, int plane_in, int n_split,
                           int n_co_tiles, float *__restrict__ partial) {
  __shared__ __align__(16) float ft[kBwChunk * kBwStride];  // features, [pair][ci]
  __shared__ __align__(16) float dt[kBwChunk * kBwStride];  // output gradient, [pair][co]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int s = blockIdx.x, k = blockIdx.y, K = gridDim.y;
  const int ci0 = (blockIdx.z / n_co_tiles) * kBwTile;
  const int co0 = (blockIdx.z % n_co_tiles) * kBwTile;
  const int n = pair_num[k];
  // ranges are multiples of the chunk, so that every workgroup starts on a chunk boundary
  int len = (n + n_split - 1) / n_split;
  len = (len + kBwChunk - 1) / kBwChunk * kBwChunk;
  const int p_begin = min(s * len, n), p_end = min(p_begin + len, n);
  const int32_t *rows_in = pairs + ((int64_t)k * 2 + plane_in) * pair_stride;
  const int32_t *rows_out = pairs + ((int64_t)k * 2 + (1 - plane_in)) * pair_stride;

  // staging: 16 threads per gathered row (256 contiguous bytes), pairs (tid >> 4) + 16j
  const int sp = tid >> 4, sq = (tid & 15) * 4;
  constexpr unsigned kEB = sizeof(IO);
  // rows in flight: as loaded from a buffer, or widened already by the pointer path
  typedef std::conditional_t<BUF, decltype(buf_quad(__amdgpu_buffer_rsrc_t(), 0u, (const IO *)nullptr)),
                             float4v> Held;
  Held rf[4], rd[4];
  const __amdgpu_buffer_rsrc_t rs_f =
      __builtin_amdgcn_make_buffer_rsrc((void *)feats, 0, (int)feat_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_d =
      __builtin_amdgcn_make_buffer_rsrc((void *)dout, 0, (int)dout_bytes, 0x00020000);
  // a quad of channels beyond the matrix width reads zeros as well
  const unsigned col_f = ci0 + sq < cin ? (unsigned)(ci0 + sq) * kEB : 0xFFFFF000u;
  const unsigned col_d = co0 + sq < cout ? (unsigned)(co0 + sq) * kEB : 0xFFFFF000u;
  // row numbers of the chunk after the one being fetched: the gathers never wait for
  // their own index loads
  int idx_i[4], idx_o[4];
  auto fetch_idx = [&](int p0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int p = p0 + sp + 16 * j;
      idx_i[j] = p < p_end ? rows_in[p] : -1;
      idx_o[j] = p < p_end ? rows_out[p] : -1;
    }
  };
  auto fetch = [&](int p0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int p = p0 + sp + 16 * j;
      if constexpr (BUF) {
        const unsigned ri = idx_i[j] >= 0 ? (unsigned)idx_i[j] * ((unsigned)cin * kEB) : 0xFFFFF000u;
        const unsigned ro = idx_o[j] >= 0 ? (unsigned)idx_o[j] * ((unsigned)cout * kEB) : 0xFFFFF000u;
        // saturating: an offset that is already outside stays outside
        const unsigned of = ri > 0xFFFFF000u - col_f ? 0xFFFFF000u : ri + col_f;
        const unsigned od = ro > 0xFFFFF000u - col_d ? 0xFFFFF000u : ro + col_d;
        rf[j] = buf_quad(rs_f, of, feats);
        rd[j] = buf_quad(rs_d, od, dout);
      } else {
        (void)p;
        rf[j] = load_quad(feats, idx_i[j], ci0 + sq, cin);
        rd[j] = load_quad(dout, idx_o[j], co0 + sq, cout);
      }
    }
    fetch_idx(p0 + kBwChunk);
  };
  auto stage = [&]() {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      *reinterpret_cast<float4v *>(ft + (sp + 16 * j) * kBwStride + sq) = widen4(rf[j]);
      *reinterpret_cast<float4v *>(dt + (sp + 16 * j) * kBwStride + sq) = widen4(rd[j]);
    }
  };

  // acc[jm][jn]: D[ci0 + 4*(4g + r) + jm][co0 + 4*l16 + jn] in component r
  float4v acc[4][4];
#pragma unroll
  for (int jm = 0; jm < 4; ++jm)
#pragma unroll
    for (int jn = 0; jn < 4; ++jn) acc[jm][jn] = float4v{0.f, 0.f, 0.f, 0.f};
  // k slot g of this wave's MFMA step tt is pair 4 * (wave + 4 * tt) + g of the chunk
  const float *a_row = ft + (4 * wave + g) * kBwStride + 4 * l16;
  const float *b_row = dt + (4 * wave + g) * kBwStride + 4 * l16;

  if (p_begin < p_end) {
    fetch_idx(p_begin);
    fetch(p_begin);
  }
  for (int p0 = p_begin; p0 < p_end; p0 += kBwChunk) {
    stage();
    __syncthreads();
    if (p0 + kBwChunk < p_end) fetch(p0 + kBwChunk);  // in flight during the MFMAs
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      const float4v a = *reinterpret_cast<const float4v *>(a_row + tt * 16 * kBwStride);
      const float4v b = *reinterpret_cast<const float4v *>(b_row + tt * 16 * kBwStride);
#pragma unroll
      for (int jm = 0; jm < 4; ++jm)
#pragma unroll
        for (int jn = 0; jn < 4; ++jn)
          acc[jm][jn] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[jm], b[jn], acc[jm][jn], 0, 0, 0);
    }
    __syncthreads();
  }
  // Add the four waves' tiles in wave order through LDS (tile[ci][co], 64 x 64 floats in
  // the staging memory), then write the tile out.
  float *tile = ft;
  static_assert(2 * kBwChunk * kBwStride >= kBwTile * kBwTile, "the tile fits the staging memory");
  for (int w = 0; w < 4; ++w) {
    if (wave == w) {
#pragma unroll
      for (int jm = 0; jm < 4; ++jm)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          // the four column blocks of a lane are four neighbouring columns
          float4v *t = reinterpret_cast<float4v *>(tile + (4 * (4 * g + r) + jm) * kBwTile + 4 * l16);
          const float4v v = {acc[jm][0][r], acc[jm][1][r], acc[jm][2][r], acc[jm][3][r]};
          *t = w == 0 ? v : *t + v;
        }
    }
    __syncthreads();
  }
  float *dst = partial + ((int64_t)s * K + k) * cin * cout;
  for (int e = tid; e < kBwTile * kBwTile; e += 256) {
    const int ci = ci0 + e / kBwTile, co = co0 + e % kBwTile;
    if (ci < cin && co < cout) dst[(int64_t)ci * cout + co] = tile[e];
  }
}

// The same tile of the same sums on the bfloat16 matrix instructions, sixteen times the rate of
// the float ones: every element is cut into bfloat16 parts that add up to it (three for a
// float, two for a half), and of the products of parts those are taken that a float sum still
// sees -- six of nine for floats, the ones left out are below 2^-24 of the product; all four
// for halves.
//
// No LDS in the loop: a wave takes 32 pairs at a time, lane (l16, g) reads four channels
// (4 l16 .. + 3) of the rows of pairs 8 g .. 8 g + 7, and as the parts of two neighbouring
// pairs' elements are packed into a word, the words of a channel are the operand of one
// matrix step as it is wanted (eight pairs to a lane): the transposition costs nothing.
//
// What bounds it, 64 -> 128 channels, 1.54M pairs, floats: matrix instructions (96 of 16
// cycles a wave and step) keep the matrix cores busy for a third of the time, 350 vector
// instructions (7 for every two elements that are cut) and the gathers take about as long
// each, and with the two waves a SIMD that 252 registers leave the three overlap in part only
// (a wave waits for rows in 37 % of its time).  Finer interleaving of loads and matrix
// instructions gained nothing, rows that all lie in L1 a tenth.  Measured, both kernels with
// their reduction, on pairs drawn at random, conv_bwd_filter_kernel -> this one:
//                                   float            half
//    64 -> 128, 1.54M pairs    272 -> 175 us    270 -> 118 us
//   128 -> 128, 0.78M pairs    260 -> 163       272 -> 121
//    64 -> 64,  137k pairs      31 -> 21         32 -> 18
//    32 -> 32,  44k pairs       19 -> 13         20 -> 11
//    64 -> 152, stride 2, 52k   31 -> 21         31 -> 18
//    64 -> 128, 5^3, 480k       89 -> 56         94 -> 45
//    30 -> 31,  205k            46 -> 20         54 -> 18
//    64 -> 64,  10k             17 -> 11         18 -> 10
//    32 -> 32,  stride 2, 5.5k  13 -> 9.3        14 -> 8.7
// Rows need not be whole quads: a row's last quad is its last four channels.
//
// JM = 4 is that tile.  JM = 1 is for up to 16 input channels: a tile of 16 x 64 with one input
// channel to a lane, a quarter of the matrix instructions and of the features' cutting, and
// four waves a SIMD.  It is bound by the gathers of the output gradient and the wait for them.
//     3 -> 64,  415k pairs       65 -> 22 us      75 -> 20 us
//    16 -> 64,  415k             56 -> 21 (39 with JM = 4)   56 -> 18 (33)
//    14 -> 46,  205k             48 -> 13         54 -> 12
// Error of the gradient against 64 bits, relative, of the first six rows above, floats:
// 5.1e-7 -> 2.9e-7, 5.1e-7 -> 2.2e-7, 2.1e-7 -> 1.2e-7, 1.9e-7 -> 0.9e-7, 1.5e-7 -> 0.9e-7,
// 2.8e-7 -> 1.2e-7.
//
// What the parts cannot do is worked out with float instructions instead: a workgroup that meets
// one of the following takes its range again (lane (l16, g)'s row 8 g + j is k slot g of step j).
//  - Infinities, NaN, and floats that round to an infinity as bfloat16: a sum that is not finite.
//  - Elements with bits below 2^-133, the last of a bfloat16: parts that do not add up.  What is
//    left of an element for its third part is a bfloat16 then and only then if the lower half of
//    its word is zero (conversion, dot product and matrix instruction keep subnormals), so one
//    OR of two elements' words shows it.  Elements of 2^-110 and above, and zero, always pass.
//  - Sums that are not zero and below 2^-95: six products of parts, each rounded at 2^-150, where
//    the float instruction rounds one; of 2^26 pairs (a wave's most) they are off by 2^-121.4,
//    which is 2^-26 of 2^-95.  A sum of zero has no product above the smallest subnormal, or its
//    products cancel as they are.
// Where every workgroup does so, 64 -> 128 channels take 360 us instead of 174 (260 in
// conv_bwd_filter_kernel), 64 -> 64 with 137k pairs 38 instead of 21 (31), 16 -> 64 35 instead of
// 21 (55).
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef int int4v __attribute__((ext_vector_type(4)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
constexpr int kBwStep = 32;                      // pairs of a wave's step
constexpr unsigned kBwOutside = 0x7FFFF000u;     // byte offset beyond either matrix
constexpr unsigned kBwColOutside = 0x80000000u;  // (added to any row's offset: outside as well)

template <typename IO, int JM>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(JM == 4 ? 2 : 4)))
    conv_bwd_filter_parts_kernel(const IO *__restrict__ feats, int n_in, int cin,
                                 const IO *__restrict__ dout, int n_out, int cout,
                                 const int32_t *__restrict__ pairs, int64_t pair_stride,
                                 const int32_t *__restrict__ pair_num, int plane_in, int n_split,
                                 int n_co_tiles, int K, int n_tiles, float *__restrict__ partial) {
  constexpr int P = sizeof(IO) == 4 ? 3 : 2;
  constexpr unsigned kEB = sizeof(IO);
  constexpr int kRows = 16 * JM;  // rows (ci) of the tile
  typedef decltype(buf_quad(__amdgpu_buffer_rsrc_t(), 0u, (const IO *)nullptr)) Quad;
  typedef std::conditional_t<JM == 4, Quad, IO> FeatQuad;
  __shared__ __align__(16) float tile[4 * kRows * kBwTile];
  __shared__ int odd_s;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  // Consecutive workgroups land on different XCDs, one L2 each.  The pairs of an offset ascend
  // in their output row, so the offsets' ranges of one number touch the same rows of the
  // output gradient: the ranges, each with all offsets and tiles, go to the XCDs in runs.
  const int total = gridDim.x, xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int item = xcd * (total >> 3) + min(xcd, total & 7) + slot;
  const int s = item / (K * n_tiles), kt = item - s * (K * n_tiles);
  const int k = kt / n_tiles, t_co = kt % n_tiles;
  const int ci0 = (t_co / n_co_tiles) * kRows;
  const int co0 = (t_co % n_co_tiles) * kBwTile;
  const int n = pair_num[k];
  int len = (n + n_split - 1) / n_split;
  len = (len + 4 * kBwStep - 1) / (4 * kBwStep) * (4 * kBwStep);
  const int p_begin = min(s * len, n), p_end = min(p_begin + len, n);
  const int32_t *rows_in = pairs + ((int64_t)k * 2 + plane_in) * pair_stride;
  const int32_t *rows_out = pairs + ((int64_t)k * 2 + (1 - plane_in)) * pair_stride;
  const unsigned row_f = (unsigned)cin * kEB, row_d = (unsigned)cout * kEB;
  // (pairs behind the range read as 0)
  const __amdgpu_buffer_rsrc_t rs_i =
      __builtin_amdgcn_make_buffer_rsrc((void *)rows_in, 0, p_end * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_o =
      __builtin_amdgcn_make_buffer_rsrc((void *)rows_out, 0, p_end * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_f =
      __builtin_amdgcn_make_buffer_rsrc((void *)feats, 0, (int)(n_in * row_f), 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_d =
      __builtin_amdgcn_make_buffer_rsrc((void *)dout, 0, (int)(n_out * row_d), 0x00020000);
  // The last quad of a row that ends within it is the row's last four channels: its first ones
  // are worked out twice, and stored by the quad that begins with them (or before them), which
  // may be another workgroup's.
  const auto quad = [](int c, int width) { return min(c, width - 4); };
  const int ci = JM == 4 ? ci0 + 4 * l16 : ci0 + l16, co = co0 + 4 * l16;
  const unsigned col_f =
      ci < cin ? (unsigned)(JM == 4 ? quad(ci, cin) : ci) * kEB : kBwColOutside;
  const unsigned col_d = co < cout ? (unsigned)quad(co, cout) * kEB : kBwColOutside;
  if (tid == 0) odd_s = 0;

  // acc[jm][jn]: D[ci0 + JM*(4g + r) + jm][co0 + 4*l16 + jn] in component r
  float4v acc[JM][4];
  int idx_f[8], idx_d[8];
  FeatQuad qf[8];
  Quad qd[8];
  auto load_idx = [&](const __amdgpu_buffer_rsrc_t &rs, int p0, int (&idx)[8])
      __attribute__((always_inline)) {
    if (p0 + kBwStep > p_end) {  // (a word at a time: those behind the range read as 0)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        idx[j] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs, (p0 + 8 * g + j) * 4, 0, 0);
      return;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int4v v = __builtin_bit_cast(
          int4v, __builtin_amdgcn_raw_buffer_load_b128(rs, (p0 + 8 * g + 4 * h) * 4, 0, 0));
#pragma unroll
      for (int j = 0; j < 4; ++j) idx[4 * h + j] = v[j];
    }
  };
  // Byte offsets of a step's rows.  Row `rows` is behind the matrix' end and reads as zeros, for
  // pairs behind the range and row numbers below 0.
  auto offsets = [&](int p0, int rows, int (&idx)[8], unsigned row, unsigned col,
                     unsigned (&off)[8]) __attribute__((always_inline)) {
    if (p0 + kBwStep > p_end)
#pragma unroll
      for (int j = 0; j < 8; ++j) idx[j] = p0 + 8 * g + j < p_end ? idx[j] : rows;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      off[j] = __umul24(min((unsigned)idx[j], (unsigned)rows), row) + col;
  };
  // A step's rows, and after them the row numbers of the wave's next step: a wait for those
  // is not a wait for loads of rows that are younger.
  auto load_f = [&](int p0) __attribute__((always_inline)) {
    unsigned off[8];
    offsets(p0, n_in, idx_f, row_f, col_f, off);
    load_idx(rs_i, p0 + 4 * kBwStep, idx_f);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if constexpr (JM == 4)
        qf[j] = buf_quad(rs_f, off[j], feats);
      else
        qf[j] = buf_one(rs_f, off[j], feats);
    }
  };
  auto load_d = [&](int p0) __attribute__((always_inline)) {
    unsigned off[8];
    offsets(p0, n_out, idx_d, row_d, col_d, off);
    load_idx(rs_o, p0 + 4 * kBwStep, idx_d);
#pragma unroll
    for (int j = 0; j < 8; ++j) qd[j] = buf_quad(rs_d, off[j], dout);
  };
  // the waves take the range's steps in turn
  const int p_wave = p_begin + wave * kBwStep;
  auto run = [&](auto multiply) __attribute__((always_inline)) {
#pragma unroll
    for (int jm = 0; jm < JM; ++jm)
#pragma unroll
      for (int jn = 0; jn < 4; ++jn) acc[jm][jn] = float4v{0.f, 0.f, 0.f, 0.f};
    if (p_wave < p_end) {
      load_idx(rs_i, p_wave, idx_f);
      load_idx(rs_o, p_wave, idx_d);
      load_f(p_wave);
      load_d(p_wave);
    }
    for (int p0 = p_wave; p0 < p_end; p0 += 4 * kBwStep) multiply(p0);
  };
  // (the pairs (-1, 0) and (0, -1) in registers: as literals they would be packed into one
  // half of the operand, which the instruction reads twice)
  uint32_t minus0 = 0x0000BF80u, minus1 = 0xBF800000u;
  asm volatile("" : "+s"(minus0), "+s"(minus1));
  const bf16x2 m0 = __builtin_bit_cast(bf16x2, minus0), m1 = __builtin_bit_cast(bf16x2, minus1);
  uint32_t rest = 0;  // the words of which the third parts are made
  // The operand of channel block c, part by part.  `hold` has the chain of ORs end with the block:
  // left to the compiler, the features' holds all of them at once (53 registers spilled), and
  // held at every element it waits for the dot products (184 us for 64 -> 128 channels instead
  // of 174; 171 with the maximum that misses elements below 2^-134).
  auto cut = [&](const auto (&q)[8], int c, int4v (&part)[P], bool hold)
      __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float u = element(q[2 * j], c), v = element(q[2 * j + 1], c);
#pragma unroll
      for (int p = 0; p < P; ++p) {
        if (p == 2) {
          rest |= __builtin_bit_cast(uint32_t, u) | __builtin_bit_cast(uint32_t, v);
          if (hold && j == 3) asm volatile("" : "+v"(rest));
        }
        const bf16x2 b = __builtin_convertvector(float2v{u, v}, bf16x2);
        part[p][j] = __builtin_bit_cast(int, b);
        if (p + 1 < P) {
          u = __builtin_amdgcn_fdot2_f32_bf16(b, m0, u, false);
          v = __builtin_amdgcn_fdot2_f32_bf16(b, m1, v, false);
        }
      }
    }
  };
  run([&](int p0) __attribute__((always_inline)) {
    int4v pf[JM][P];
#pragma unroll
    for (int c = 0; c < JM; ++c) cut(qf, c, pf[c], true);
    load_f(p0 + 4 * kBwStep);  // (in flight during the multiplications)
    // (a channel block of the gradient is cut among the multiplications of the one before; the
    // barriers keep the compiler from cutting them all at once, for which there are no registers)
    int4v pds[2][P];
    cut(qd, 0, pds[0], false);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int jn = 0; jn < 4; ++jn) {
      const int4v (&pd)[P] = pds[jn & 1];
      if (jn < 3) cut(qd, jn + 1, pds[(jn + 1) & 1], false);
      if (jn == 2) {
        __builtin_amdgcn_sched_barrier(0);
        load_d(p0 + 4 * kBwStep);
      }
      // A step's products are summed by themselves, the smallest first (of floats only those
      // of parts a + b <= 2), and added to the sum of the steps before: one rounding at its
      // size a step, not one an instruction.
      float4v t[JM];
#pragma unroll
      for (int jm = 0; jm < JM; ++jm) t[jm] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int a = P - 1; a >= 0; --a)
#pragma unroll
        for (int b = P - 1; b >= 0; --b) {
          if (a + b > 2) continue;
#pragma unroll
          for (int jm = 0; jm < JM; ++jm)
            t[jm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, pf[jm][a]),
                                                            __builtin_bit_cast(bf16x8, pd[b]), t[jm],
                                                            0, 0, 0);
        }
#pragma unroll
      for (int jm = 0; jm < JM; ++jm) acc[jm][jn] += t[jm];
      __builtin_amdgcn_sched_barrier(0);
    }
  });
  __syncthreads();  // (odd_s is cleared)
  {
    // (bits << 1) - 1 takes the sign away and zero to the top; 0 times what is not finite is NaN
    uint32_t least = 0xFFFFFFFFu;
    float nan = 0.f;
#pragma unroll
    for (int jm = 0; jm < JM; ++jm)
#pragma unroll
      for (int jn = 0; jn < 4; ++jn)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = acc[jm][jn][r];
          least = min(least, (__builtin_bit_cast(uint32_t, v) << 1) - 1u);
          nan = __builtin_fmaf(v, 0.f, nan);
        }
    const bool odd = nan != 0.f || (rest & 0xFFFFu) != 0 || least < ((127u - 95u) << 24) - 1u;
    if (odd) odd_s = 1;
  }
  __syncthreads();
  if (odd_s != 0) {
    run([&](int p0) __attribute__((always_inline)) {
      float xf[8][JM], xd[8][4];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
#pragma unroll
        for (int c = 0; c < JM; ++c) xf[j][c] = element(qf[j], c);
#pragma unroll
        for (int c = 0; c < 4; ++c) xd[j][c] = element(qd[j], c);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int jm = 0; jm < JM; ++jm)
#pragma unroll
          for (int jn = 0; jn < 4; ++jn)
            acc[jm][jn] =
                __builtin_amdgcn_mfma_f32_16x16x4f32(xf[j][jm], xd[j][jn], acc[jm][jn], 0, 0, 0);
      load_f(p0 + 4 * kBwStep);
      load_d(p0 + 4 * kBwStep);
    });
  }
  // The four waves' tiles in wave order, then the tile out.
#pragma unroll
  for (int jm = 0; jm < JM; ++jm)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *reinterpret_cast<float4v *>(tile + (wave * kRows + JM * (4 * g + r) + jm) * kBwTile + 4 * l16) =
          float4v{acc[jm][0][r], acc[jm][1][r], acc[jm][2][r], acc[jm][3][r]};
  __syncthreads();
  float *dst = partial + ((int64_t)s * K + k) * cin * cout;
#pragma unroll
  for (int i = 0; i < JM; ++i) {
    const int row = JM == 4 ? 4 * (4 * wave + i) + g : 4 * wave + g;
    const float4v *t = reinterpret_cast<const float4v *>(tile + row * kBwTile + 4 * l16);
    constexpr int kQ = kRows * kBwTile / 4;
    const float4v v = ((t[0] + t[kQ]) + t[2 * kQ]) + t[3 * kQ];
    const int c0 = JM == 4 ? ci0 + 4 * (4 * wave + i) : ci0 + row;
    const int c = JM == 4 ? quad(c0, cin) + g : c0;
    if (c0 >= cin || co >= cout || c < c0) continue;  // (c < c0: a row of the quad before)
    float *const to = dst + (int64_t)c * cout + quad(co, cout);
    const int skip = co - quad(co, cout);  // columns of the quad before
    if (skip == 0)
      *reinterpret_cast<float4u *>(to) = v;
    else
#pragma unroll
      for (int j = 1; j < 4; ++j)
        if (j >= skip) to[j] = v[j];
  }
}

// out[e] = partial[0][e] + partial[1][e] + ... in that order; out may have any strides.
template <typename IO>
__global__ void __launch_bounds__(256)
    conv_bwd_reduce_kernel(const float *__restrict__ partial, int n_split, int K, int cin, int cout,
                           IO *__restrict__ out, int64_t os_k, int64_t os_ci, int64_t os_co) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per = (int64_t)K * cin * cout;
  if (e >= per) return;
  float v = partial[e];
  for (int s = 1; s < n_split; s += 8) {  // (eight loads in flight, also at the end)
    float w[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = partial[(int64_t)min(s + i, n_split - 1) * per + e];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (s + i < n_split) v += w[i];
  }
  int co, ci, k;
  if (per <= 0xFFFFFFFFll) {
    const unsigned r = (unsigned)e / (unsigned)cout;
    co = (int)((unsigned)e - r * cout);
    k = (int)(r / (unsigned)cin);
    ci = (int)(r - (unsigned)k * cin);
  } else {
    const int64_t r = e / cout;
    co = (int)(e % cout);
    ci = (int)(r % cin);
    k = (int)(r / cin);
  }
  out[k * os_k + ci * os_ci + co * os_co] = (IO)v;
}

static int bwd_split(int K, int c_in, int c_out, int64_t pair_stride) {
  // four workgroups a CU (256 CUs) when the tiles alone are fewer, but ranges of at least 8 chunks
  const int64_t tiles = ceil_div(c_in, kBwTile) * ceil_div(c_out, kBwTile) * K;
  int64_t s = 1024 / tiles;
  const int64_t max_s = ceil_div(pair_stride > 0 ? pair_stride : 1, 8 * kBwChunk);
  if (s > max_s) s = max_s;
  if (s < 1) s = 1;
  return (int)s;
}

// Ranges of conv_bwd_filter_parts_kernel, at most bwd_split's: as many workgroups as the chip
// holds at once (two a CU), twice as many where their ranges are still 2048 pairs long (they
// end less unevenly: 128 -> 128 channels, 29k pairs an offset, 206 us with 4 ranges, 200 with
// 9), and one to about 384 pairs of the longest possible offset, as a range costs a tile written
// and read (385 pairs make two ranges; shorter offsets have shorter ones): 64 -> 152 with
// 1.9k pairs an offset 36 us with 12 ranges, 25 with 6; 64 -> 128 at 5^3 and 3.8k 84 us with 4
// and 75 with 2; 32 -> 32 with 1.6k 18.9 us with 4 and 21.1 with 2.
// An offset has no more pairs than either side has rows.
static int bwd_parts_split(int K, int c_in, int c_out, int64_t pair_stride, int64_t n_in,
                           int64_t n_out) {
  const int64_t tiles = ceil_div(c_in, kBwTile) * ceil_div(c_out, kBwTile) * K;
  const int64_t longest = std::min(pair_stride, std::min(n_in, n_out));
  const int64_t once = std::max<int64_t>(1, (512 + tiles / 2) / tiles);
  int64_t s = std::min(std::max(longest / 2048, once), 2 * once);
  s = std::min(s, ceil_div(longest, 384));
  return (int)std::min<int64_t>(s, bwd_split(K, c_in, c_out, pair_stride));
}

}  // namespace ssc

using namespace ssc;

extern "C" {

size_t ssc_conv_bwd_filter_workspace_bytes(int32_t kernel_volume, int32_t c_in, int32_t c_out,
                                           int64_t pair_stride) {
  if (kernel_volume < 1 || c_in < 1 || c_out < 1 || pair_stride < 0) return 0;
  const int s = bwd_split(kernel_volume, c_in, c_out, pair_stride);
  return align_up((size_t)s * kernel_volume * c_in * c_out * sizeof(float));
}

}  // extern "C"

template <typename IO>
static int conv_bwd_filter(const IO *features, int64_t n_in, int32_t c_in, const IO *out_grad,
                           int64_t n_out, int32_t c_out, const int32_t *pairs,
                           int64_t pair_stride, const int32_t *pair_num, int32_t kernel_volume,
                           int32_t inverse, IO *filters_grad, int64_t gs_k, int64_t gs_ci,
                           int64_t gs_co, void *workspace, size_t workspace_bytes,
                           ssc_stream_t stream) {
  const int K = kernel_volume;
  SSC_CHECK(K >= 1 && K <= SSC_MAX_KERNEL_VOLUME, SSC_ERUNTIME, "kernel volume %d out of range", K);
  SSC_CHECK(c_in >= 1 && c_out >= 1, SSC_EINVAL, "channel counts must be positive");
  SSC_CHECK(n_in >= 0 && n_out >= 0 && pair_stride >= 0, SSC_EINVAL, "negative size");
  SSC_CHECK(filters_grad != nullptr, SSC_EINVAL, "filters_grad is NULL");
  hipStream_t s = (hipStream_t)stream;
  const int64_t per = (int64_t)K * c_in * c_out;
  if (pair_stride == 0 || n_in == 0 || n_out == 0) {
    // no pairs: the gradient is zero (the reduce kernel of one zeroed range writes it)
    SSC_CHECK(workspace != nullptr && workspace_bytes >= (size_t)per * sizeof(float),
              SSC_EWORKSPACE, "conv backward workspace too small");
    int rc = fill_f32(static_cast<float *>(workspace), per, 0.f, s);
    if (rc != SSC_OK) return rc;
    hipLaunchKernelGGL(conv_bwd_reduce_kernel<IO>, dim3((unsigned)ceil_div(per, 256)), dim3(256), 0, s,
                       static_cast<const float *>(workspace), 1, K, c_in, c_out, filters_grad, gs_k,
                       gs_ci, gs_co);
    SSC_LAUNCH_CHECK("conv_bwd_reduce");
    return SSC_OK;
  }
  SSC_CHECK(features && out_grad && pairs && pair_num && workspace, SSC_EINVAL,
            "NULL pointer argument");
  const size_t need = ssc_conv_bwd_filter_workspace_bytes(K, c_in, c_out, pair_stride);
  SSC_CHECK(workspace_bytes >= need, SSC_EWORKSPACE,
            "conv backward workspace too small: %zu < %zu", workspace_bytes, need);
  const int n_ci_tiles = (int)ceil_div(c_in, kBwTile), n_co_tiles = (int)ceil_div(c_out, kBwTile);
  SSC_CHECK((int64_t)n_ci_tiles * n_co_tiles <= 65535, SSC_ERUNTIME, "too many channel tiles");
  float *partial = static_cast<float *>(workspace);
  // features are gathered through the plane the forward pass gathered them through
  const int plane_in = inverse ? 1 : 0;
  const uint64_t feat_bytes = (uint64_t)n_in * c_in * sizeof(IO);
  const uint64_t dout_bytes = (uint64_t)n_out * c_out * sizeof(IO);
  // the largest byte offset must stay below the marker that stands for "outside"
  const bool buf = (c_in & 3) == 0 && (c_out & 3) == 0 && feat_bytes <= 0xFFFFF000u &&
                   dout_bytes <= 0xFFFFF000u;
  // (row numbers and row sizes of 24 bits, offsets of 31: the index arithmetic of the kernel;
  // within it that kernel is the faster one at every size measured, from 1.4 to 4.4 times)
  const bool parts = c_out >= 4 && feat_bytes <= kBwOutside &&
                     dout_bytes <= kBwOutside && n_in < (1 << 24) && n_out < (1 << 24) &&
                     (uint64_t)c_in * sizeof(IO) < (1u << 24) && (uint64_t)c_out * sizeof(IO) < (1u << 24) &&
                     pair_stride < (1 << 28);
  const int n_split = parts ? bwd_parts_split(K, c_in, c_out, pair_stride, n_in, n_out)
                            : bwd_split(K, c_in, c_out, pair_stride);
  const dim3 grid((unsigned)n_split, (unsigned)K, (unsigned)(n_ci_tiles * n_co_tiles));
  if (parts) {
    // up to 16 channels: a tile of 16 rows, one to a lane, that takes a quarter of the instructions
    const int n_tiles = (c_in <= 16 ? 1 : n_ci_tiles) * n_co_tiles;
    hipLaunchKernelGGL((c_in <= 16 ? conv_bwd_filter_parts_kernel<IO, 1>
                                   : conv_bwd_filter_parts_kernel<IO, 4>),
                       dim3((unsigned)(n_split * K * n_tiles)), dim3(256), 0, s, features, (int)n_in,
                       c_in, out_grad, (int)n_out, c_out, pairs, pair_stride, pair_num, plane_in,
                       n_split, n_co_tiles, K, n_tiles, partial);
  } else if (buf)
    hipLaunchKernelGGL((conv_bwd_filter_kernel<IO, true>), grid, dim3(256), 0, s, features, c_in,
                       (unsigned)feat_bytes, out_grad, c_out, (unsigned)dout_bytes, pairs,
                       pair_stride, pair_num, plane_in, n_split, n_co_tiles, partial);
  else
    hipLaunchKernelGGL((conv_bwd_filter_kernel<IO, false>), grid, dim3(256), 0, s, features, c_in, 0u,
                       out_grad, c_out, 0u, pairs, pair_stride, pair_num, plane_in, n_split,
                       n_co_tiles, partial);
  SSC_LAUNCH_CHECK("conv_bwd_filter");
  hipLaunchKernelGGL(conv_bwd_reduce_kernel<IO>, dim3((unsigned)ceil_div(per, 256)), dim3(256), 0, s,
                     partial, n_split, K, c_in, c_out, filters_grad, gs_k, gs_ci, gs_co);
  SSC_LAUNCH_CHECK("conv_bwd_reduce");
  return SSC_OK;
}

extern "C" {

int ssc_conv_bwd_filter_f32(const float *features, int64_t n_in, int32_t c_in,
                            const float *out_grad, int64_t n_out, int32_t c_out,
                            const int32_t *pairs, int64_t pair_stride, const int32_t *pair_num,
                            int32_t kernel_volume, int32_t inverse, float *filters_grad,
                            int64_t gs_k, int64_t gs_ci, int64_t gs_co, void *workspace,
                            size_t workspace_bytes, ssc_stream_t stream) {
  return conv_bwd_filter<float>(features, n_in, c_in, out_grad, n_out, c_out, pairs, pair_stride,
                                pair_num, kernel_volume, inverse, filters_grad, gs_k, gs_ci, gs_co,
                                workspace, workspace_bytes, stream);
}

int ssc_conv_bwd_filter_f16(const void *features, int64_t n_in, int32_t c_in,
                            const void *out_grad, int64_t n_out, int32_t c_out,
                            const int32_t *pairs, int64_t pair_stride, const int32_t *pair_num,
                            int32_t kernel_volume, int32_t inverse, void *filters_grad,
                            int64_t gs_k, int64_t gs_ci, int64_t gs_co, void *workspace,
                            size_t workspace_bytes, ssc_stream_t stream) {
  return conv_bwd_filter<_Float16>(
      static_cast<const _Float16 *>(features), n_in, c_in, static_cast<const _Float16 *>(out_grad),
      n_out, c_out, pairs, pair_stride, pair_num, kernel_volume, inverse,
      static_cast<_Float16 *>(filters_grad), gs_k, gs_ci, gs_co, workspace, workspace_bytes, stream);
}
}
