// The convolution kernel (conv_fwd_kernel), what a launch of it needs to know of a plan,
// and the launch itself.  Ten translation units instantiate it: conv.hip the plain form
// (float and half rows), conv_epi.hip the one with the epilogue, conv_tail.hip and
// conv_tail_epi.hip the one-column-group form without and with it, conv_five.hip and
// conv_five_epi.hip the five-group form, conv_wide.hip and conv_wide_epi.hip the plain
// kernel over plans of the five-group form, conv_parts.hip and conv_parts_epi.hip the
// bfloat16-parts form -- compiled side by side, the parts of the instances take a third of
// the time.
#pragma once
#include "conv_pack.h"
#include "ssc_common.h"

#include <type_traits>

namespace ssc {

typedef float float4v __attribute__((ext_vector_type(4)));
typedef int int4v __attribute__((ext_vector_type(4)));

constexpr int kKC = 64;       // input channels per chunk = 16 MFMA steps of 4
constexpr int kStage = 64;    // pairs staged per barrier = 4 row blocks of 16
constexpr int kAStride = 64;  // floats per staged row (its 16-byte pieces permuted: staged_piece)
constexpr int kMinTile = 64;

// ---- the convolution --------------------------------------------------------------------
// Persistent kernel: one workgroup per CU walks a contiguous, work-balanced range
// of tiles.  A workgroup owns T output rows x 16*NCW output columns at a time; the
// fp32 accumulators of that tile live in LDS.
//   waves 0..NCW-1    consumers: wave w owns 16 columns of the workgroup's column
//                     range.  It multiplies the staged input rows of a stage with the
//                     weight fragments of its columns and adds the products to the
//                     accumulators.
//   waves NCW..NCW+3  producers: gather the input rows of the coming stages from
//                     global memory (several stages ahead, in registers) and stage
//                     them in LDS.
// NCW = 4 (64 columns) is what the host code launches.  NCW = 8 (128 columns, two
// consumers per SIMD, tiles half as tall) computes the same result; on the 64 -> 128
// channel benchmark layer it is 6 % slower, because the shorter tiles pack the row
// blocks less densely and the weight-fragment traffic per tile row doubles.
// A stage = one group of the schedule (4 row blocks = 64 pair slots, any mix of
// offsets) x one 64-channel chunk of Cin.  One barrier per stage hands the buffer
// filled with stage s+1 to the consumers and the buffer of stage s back to the
// producers.  After a tile's last stage all waves write the tile out and clear
// the accumulators.
//
// fp32 MFMAs and ordinary vector-ALU instructions do not overlap on a SIMD, no
// matter which wave issues them (measured: every VALU instruction next to a
// stream of v_mfma_f32_16x16x4_f32 costs about five cycles of matrix time), while
// scalar, LDS and memory instructions of another wave are free.  So the loops
// below keep vector arithmetic out of the steady state: the schedule already
// holds byte offsets, addresses are (scalar offset + constant lane offset) of
// buffer loads, per-stage bookkeeping is scalar loads and scalar arithmetic, and
// the producers do not touch the VALU except for one add per gathered row chunk.
// Buffer loads are range-checked by the hardware and return zero outside their
// buffer: padding slots carry an offset beyond the features and gather zeros,
// and the prefetches that run past the end of a workgroup's schedule are harmless.
//
// MFMA orientation: D[16 channels x 16 pairs] = W^T[16 x 4] * F^T[4 x 16], so a
// lane ends up with 4 consecutive output channels of one pair and adds them to
// the LDS accumulator row of that pair with one 16-byte read-modify-write.  A
// column group belongs to exactly one wave, which walks the schedule in order,
// so every output element sees its offsets added in ascending k: reproducible,
// no atomics.
//
// Dynamic LDS: acc[T+1][16*NCW+4] | abuf[2][64][64]
constexpr int kRowsAhead = 4;  // stages whose gathered rows are in flight in registers
constexpr int kIdxAhead = 2;   // further stages whose gather offsets are in flight
constexpr unsigned kGatherPad = 0xFFFFF000u;  // byte offset that gathers zeros (beyond any feature buffer)
constexpr int kRsrcFlags = 0x00020000;        // raw buffer of 32-bit data

__device__ __forceinline__ float4v buf_load4(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
typedef int int3v __attribute__((ext_vector_type(3)));
__device__ __forceinline__ int3v buf_load3(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(int3v, __builtin_amdgcn_raw_buffer_load_b96(r, voff, soff, 0));
}
__device__ __forceinline__ int buf_load1(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return (int)__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
}

// Element type of the features, the filters and the output.  float: fp32 rows in LDS,
// v_mfma_f32_16x16x4_f32.  _Float16: half rows in LDS, v_mfma_f32_16x16x32_f16; the
// accumulators are fp32 either way and are rounded once, when a finished tile is written.
typedef int int2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float3v __attribute__((ext_vector_type(3)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
template <typename IO> struct Io;
template <> struct Io<float> {
  static constexpr int kBytes = 4;
  static constexpr int kRowBytes = kAStride * 4;  // a staged row of 64 channels in LDS
  static constexpr int kFragBytes = 4096;         // packed filters of (offset, column block, chunk)
  typedef float4v Raw;  // four channels as they are loaded
  static __device__ __forceinline__ Raw zero() { return Raw{0.f, 0.f, 0.f, 0.f}; }
  static __device__ __forceinline__ Raw gather(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return buf_load4(r, voff, soff);
  }
  static __device__ __forceinline__ Raw load(const float *p) {
    return *reinterpret_cast<const float4v *>(p);
  }
  // the first n (possibly <= 0 or > 4) of four channels, zeros for the rest
  static __device__ __forceinline__ Raw load_first(const float *p, int n) {
    Raw v = zero();
    if (n > 0) v.x = p[0];
    if (n > 1) v.y = p[1];
    if (n > 2) v.z = p[2];
    if (n > 3) v.w = p[3];
    return v;
  }
  static __device__ __forceinline__ void store_stream(float *p, const float4v &v) {
    __builtin_nontemporal_store(v, reinterpret_cast<float4v *>(p));
  }
};
template <> struct Io<_Float16> {
  static constexpr int kBytes = 2;
  static constexpr int kRowBytes = 128;
  static constexpr int kFragBytes = 2048;
  typedef int2v Raw;
  static __device__ __forceinline__ Raw zero() { return Raw{0, 0}; }
  static __device__ __forceinline__ Raw gather(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(int2v, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
  }
  static __device__ __forceinline__ Raw load(const _Float16 *p) {
    return *reinterpret_cast<const int2v *>(p);
  }
  static __device__ __forceinline__ Raw load_first(const _Float16 *p, int n) {
    half4v v = {(_Float16)0.f, (_Float16)0.f, (_Float16)0.f, (_Float16)0.f};
    if (n > 0) v.x = p[0];
    if (n > 1) v.y = p[1];
    if (n > 2) v.z = p[2];
    if (n > 3) v.w = p[3];
    return __builtin_bit_cast(int2v, v);
  }
  static __device__ __forceinline__ void store_stream(_Float16 *p, const float4v &v) {
    const half4v h = __builtin_convertvector(v, half4v);  // round to nearest even
    __builtin_nontemporal_store(__builtin_bit_cast(int2v, h), reinterpret_cast<int2v *>(p));
  }
};

// Where 16-byte piece `piece` of a staged row (16 of a float one, 8 of a half one) lies in it, row:
// its number in its row block.  A read of one piece by the 16 rows of a block, and by four lane
// groups of four neighbouring pieces, then meets no bank twice: 4.1 cycles a KiB where rows with
// 16 bytes of padding take 8.4 (the float form 64 -> 128 channels, 1.54M pairs: 289 -> 281 us).
template <bool HALF> __device__ __forceinline__ int staged_piece(int piece, int row) {
  return (HALF ? piece ^ (row >> 1) : piece ^ row) * 16;
}

// Position of a stage in the schedule: group index and channel chunk.  Advanced
// with scalar arithmetic only.
struct StagePos {
  int g, cc;
  __device__ __forceinline__ void advance(int nch) {
    ++cc;
    if (cc == nch) {
      cc = 0;
      ++g;
    }
  }
};

// GATHER selects how the producers read the input rows:
//   1  Cin is a multiple of 64 and the features are smaller than 4 GiB: the schedule
//      holds byte offsets of the gather rows and the gather is a range-checked
//      buffer load;
//   2  the same with Cin a multiple of 4 only: in the last channel chunk the lanes
//      beyond Cin gather from the padding offset, i.e. zeros;
//   0  anything else: the schedule holds row numbers and the gather uses 64-bit
//      addresses with per-channel masks.
//
// The waves-per-SIMD attribute states the occupancy the workgroup size gives anyway
// (one workgroup per CU), so that the compiler uses the whole register budget.
// NS: MFMA steps (of 4 input channels) per chunk, 16 for chunks of 64 channels.  A layer
// whose input channels do not fill whole chunks of 64 is cut into ceil(Cin / 64) chunks of
// equal width 4 NS instead (200 channels: 4 chunks of 52, 13 steps each, where chunks of 64
// would run 64 steps for 50 steps' worth of channels): MFMA steps, fragment loads, gathers
// and staged-row reads beyond NS are left out.  Half precision always runs whole chunks.
// What conv_fwd_kernel applies to a finished tile instead of storing its sums: per column c
// of the accumulators z = (x - shift[c]) * scale[c] + add[c], then by mode[c]
//   0  y = z                                          2  y = z * act_gate(z_g + pre[g]),
//   1  y = act_scalar(z + pre[c])                        g = gate[c], a column of the same
//   3  nothing is stored (gates, padding)                workgroup's column range
// stored at column dest[c] of rows of c_dest columns.  The gates of a block of 64 columns
// are one run of at most 16 columns (gate_run): act_gate is evaluated once per gate and
// row, not once per gated column.  mode == nullptr: plain store.
struct ConvEpilogue {
  const float *shift, *scale, *add, *pre;  // [cout]
  const int32_t *mode, *gate, *dest;       // [cout]
  const int32_t *gate_run;                 // [2 * blocks of 64 columns]: first gate, gates
  int act_s, act_g, c_dest;
};

// ---- bfloat16 parts ---------------------------------------------------------------------
// An element of a float matrix, times 2^16, as three bfloat16 parts that add up to it: the element
// rounded, what is left rounded, and the rest (the last bit of a float is 2^-149, that of a bfloat16
// 2^-133).  The matrix cores multiply bfloat16 sixteen times as fast as floats; of the nine products
// of parts six are taken (the ones left out are below 2^-24 of the product).
// What the parts cannot do (PartsCheck::odd) and what then happens: see the parts form below.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
struct PartsCheck {
  float nan;       // NaN once a sum was not finite (0 times it is NaN)
  uint32_t least;  // smallest magnitude of a sum that is not zero: (bits << 1) - 1
  __device__ __forceinline__ void sum(float v) {
    least = min(least, (__builtin_bit_cast(uint32_t, v) << 1) - 1u);
    nan = __builtin_fmaf(v, 0.f, nan);
  }
  __device__ __forceinline__ bool odd() const {
    return nan != 0.f || least < ((127u - 94u) << 24) - 1u;
  }
};
// Elements' parts, each two of them packed into a word.  (What a part leaves by the dot
// product of a bfloat16 pair: it holds the matrix cores up for its time, which shift, mask and
// subtraction do not -- 48 matrix instructions of a wave beside 112 others of another one: 812
// cycles alone, 1392 with dot products, 900 with subtractions -- but those are twice as many, and
// the kernel is 2 % slower with them.)
struct PartsCut {
  bf16x2 m0, m1;  // (-1, 0) and (0, -1)
  __device__ __forceinline__ PartsCut() {
    // (in registers: as literals they would be packed into one half of the operand, which the
    // instruction reads twice)
    uint32_t minus0 = 0x0000BF80u, minus1 = 0xBF800000u;
    asm volatile("" : "+s"(minus0), "+s"(minus1));
    m0 = __builtin_bit_cast(bf16x2, minus0);
    m1 = __builtin_bit_cast(bf16x2, minus1);
  }
  // (step by step over all of them: a pair's own steps each wait for the one before, and one pair
  // after the other makes the kernel 7-9 % slower; scheduling barriers behind the conversions as well
  // as behind the dot products 1 %, none at all 1.5 %)
  template <int N>
  __device__ __forceinline__ void all(const float4v (&v)[N], int2v (&p)[N][3]) const {
    float4v u[N];
    bf16x2 part[N][2];
#pragma unroll
    for (int j = 0; j < N; ++j) u[j] = v[j] * kPartsScale;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
      for (int j = 0; j < N; ++j) {
        part[j][0] = __builtin_convertvector(float2v{u[j].x, u[j].y}, bf16x2);
        part[j][1] = __builtin_convertvector(float2v{u[j].z, u[j].w}, bf16x2);
        p[j][i] = int2v{__builtin_bit_cast(int, part[j][0]), __builtin_bit_cast(int, part[j][1])};
      }
      if (i == 2) break;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        u[j].x = __builtin_amdgcn_fdot2_f32_bf16(part[j][0], m0, u[j].x, false);
        u[j].y = __builtin_amdgcn_fdot2_f32_bf16(part[j][0], m1, u[j].y, false);
        u[j].z = __builtin_amdgcn_fdot2_f32_bf16(part[j][1], m0, u[j].z, false);
        u[j].w = __builtin_amdgcn_fdot2_f32_bf16(part[j][1], m1, u[j].w, false);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
};
// Staged rows in LDS: two stages of 2 blk pairs x 32 channels x 3 parts (blk: pairs to a block).
inline size_t parts_staged_bytes(int blk) { return 2 * (size_t)(2 * blk) * 192 + 16; }
// Position in the schedule of the parts form: group and chunk of 64 channels.  The last group
// repeats: what is fetched ahead of a workgroup's end is its last group again.
struct PartsPos {
  int g, cc;
  __device__ __forceinline__ void advance(int gs, int nch, int g_last) {  // gs: groups to a stage
    ++cc;
    if (cc == nch) {
      cc = 0;
      g = g < g_last ? g + gs : g_last;
    }
  }
};

// FORM: 0 the kernel as described above; 1 the one-column-group form; 2 the five-group form
// (see the consumers); 3 the plain kernel on a plan of the five-group form, whose accumulator
// rows are 16 columns wider (the launches of such a plan that have no fifth group); 4 and 5 the
// bfloat16-parts form, over blocks of 32 and of 64 pairs.
template <typename IO, int GATHER, int NCW, int NS, bool EPI, int FORM>
__global__ void __launch_bounds__((NCW + 4) * 64)
    __attribute__((amdgpu_waves_per_eu((NCW + 4) / 4, (NCW + 4) / 4)))
    conv_fwd_kernel(const IO *__restrict__ features, int cin, unsigned feat_bytes,
                    const void *__restrict__ packed, unsigned packed_bytes,
                    const int32_t *__restrict__ sched_in, const int32_t *__restrict__ sched_out,
                    const int32_t *__restrict__ grp_meta, unsigned sched_bytes, unsigned meta_bytes,
                    const int32_t *__restrict__ wg_grp,
                    int nch, int ncb, IO *__restrict__ out, int cout, int T, int cols_per_xcd,
                    int col_base, int xcol, ConvEpilogue epi) {
  constexpr bool TAIL = FORM == 1, FIVE = FORM == 2, WIDE = FORM == 3,
                 PARTS = FORM == 4 || FORM == 5;
  constexpr int kCN = 16 * NCW;   // output columns per workgroup
  constexpr int kEB = Io<IO>::kBytes;
  constexpr bool kHalf = kEB == 2;
  constexpr int kRowB = Io<IO>::kRowBytes;    // bytes of a staged row
  constexpr int kFragB = Io<IO>::kFragBytes;  // bytes of a packed filter fragment
  static_assert(NS >= 1 && NS <= 16 && (!kHalf || NS == 16), "steps per chunk");
  static_assert(GATHER != 1 || NS == 16, "the unchecked gather reads whole chunks of 64");
  constexpr int kChunk = kHalf ? kKC : 4 * NS;  // input channels per chunk
  constexpr int kQFull = NS / 4, kQRem = NS % 4;  // whole quarters, steps of the partial one
  typedef typename Io<IO>::Raw Raw;
  // accumulator row stride in floats (the five-group form: 16 more columns)
  constexpr int kAS = kCN + (FIVE || WIDE ? 16 : 0) + 4;
  constexpr int NT = (NCW + 4) * 64;
  // threads that write a tile out (the parts form over blocks of 64 with the epilogue: the
  // consumers only.  With all waves 50 registers of the producers were spilled, 512 -> 608 channels
  // 5.3 ms instead of 4.4; that was before rows were scaled, whose cut takes fewer of them, and has
  // not been measured since)
  constexpr bool kProducersFlush = !(EPI && FORM == 5);
  constexpr int NTF = kProducersFlush ? NT : NCW * 64;
  constexpr int NP = 256;  // producer threads
  constexpr int NE = kStage * 16 / NP;
  extern __shared__ __align__(16) float lds[];
  float *acc = lds;
  float *abuf = acc + (size_t)(T + 1) * kAS;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool producer = wave >= NCW;
  // Consecutive workgroup ids land on different XCDs (8 of them, one L2 each): give
  // every XCD a contiguous run of tile ranges so neighbouring tiles, which gather
  // the same input rows, share an L2.  Which column blocks an XCD works on depends on the
  // size of the packed filters.  Small ones (they stay in every L2): all column blocks of
  // a run of ranges, so that the gathered rows are shared as well.  Large ones (an L2
  // holds a fraction of them, and a workgroup walks all of its column block's fragments
  // once per tile): one column block per XCD (cols_per_xcd: XCDs per column block), so that
  // the 32 workgroups of an XCD ask for the same fragments at about the same time and
  // one fetch serves them all.
  int chunk = blockIdx.x, cblk = blockIdx.y;
  {
    const int nwg = gridDim.x;
    if (cols_per_xcd > 0) {
      const int lin = blockIdx.y * nwg + blockIdx.x;  // dispatch order: XCD = lin % 8
      const int xcd = lin & 7, slot = lin >> 3;
      const int ncol = gridDim.y;  // divides 8
      cblk = xcd % ncol;
      chunk = (xcd / ncol) * ((nwg * ncol) >> 3) + slot;
    } else if ((nwg & 7) == 0) {
      chunk = (chunk & 7) * (nwg >> 3) + (chunk >> 3);
    } else if (cols_per_xcd < 0) {
      // any other grid: the (range, column block) items, numbered range by range (-1) or
      // column block by column block (-2), are dealt to the XCDs in contiguous runs; XCD x
      // has the workgroups x, x + 8, ...
      const int ncol = gridDim.y, total = nwg * ncol;
      const int lin = blockIdx.y * nwg + blockIdx.x;
      const int xcd = lin & 7, slot = lin >> 3;
      const int item = xcd * (total >> 3) + min(xcd, total & 7) + slot;
      if (cols_per_xcd == -1) {
        chunk = item / ncol;
        cblk = item - chunk * ncol;
      } else {  // filters larger than an L2: column block by column block (an XCD sees few)
        cblk = item / nwg;
        chunk = item - cblk * nwg;
      }
    }
  }
  const int g_begin = wg_grp[2 * chunk], g_end = wg_grp[2 * chunk + 1];  // this workgroup's groups
  const int nstages = (g_end - g_begin) * nch;  // stages of this workgroup
  const int col0 = col_base + cblk * kCN;
  static_assert(FORM == 0 || (NCW == 4 && !kHalf), "the other forms are built for float");
  static_assert(!PARTS || (NS == 16 && GATHER != 0), "the parts form: whole chunks, buffer loads");
  PartsCheck check = {0.f, 0xFFFFFFFFu};  // (the parts form: what its sums showed)
  float unscale = PARTS ? 1.f / (kPartsScale * kPartsScale) : 1.f;  // of the accumulators

  {
    float4v z = {0.f, 0.f, 0.f, 0.f};
    float4v *a4 = reinterpret_cast<float4v *>(acc);
    for (int i = tid; i < (T + 1) * kAS / 4; i += NT) a4[i] = z;
  }

  // Tile `tl` is complete: write its rows, clear the accumulators.
  // (slot0 = accumulator slot of the tile's first row; slots wrap around at T)
  // Epilogue constants of this thread, loaded once: when a tile is written out a thread
  // keeps its 4 columns (c_t) and walks down the rows; lane l of a row's 16 lanes also
  // owns gate l of the workgroup's column block.
  //   z = x * ca + cb (cb includes the bias in front of a scalar activation);
  //   mg = mode | LDS column of the gate << 4;  dest = output column
  //   gate l: activated value = act_gate(x * gca + gcb), LDS column gcl (-1: none)
  // LDS columns count from the first column of the block (a fifth group's from its own).
  // (EpiConsts: ca, cb, mg, dest per column of the thread; gca, gcb, gcl of its gate)
  struct EpiConsts {
    float ca[4], cb[4], gca, gcb;
    int mg[4], dest[4], gcl;
    bool any, vec;
  };
  // bcol0: first output column of the block of 64 the columns belong to; ncols: how many of
  // the block's columns the workgroup has (64, or the 16 of a fifth group)
  auto epi_consts = [&](int bcol0, int ncols, int tid) -> EpiConsts {
    EpiConsts e;
    e.gca = 0.f;
    e.gcb = 0.f;
    e.gcl = -1;
    const int c_t = (tid % (kCN / 4)) * 4, col = bcol0 + c_t;
    const bool col_ok = col < cout && c_t < ncols;
    static_assert(!EPI || kCN == 64, "the epilogue's gate runs are per block of 64 columns");
    const int eblk = bcol0 / kCN;  // block of 64 columns the workgroup's columns start
    const int gfirst = epi.gate_run[2 * eblk], gcount = min(epi.gate_run[2 * eblk + 1], 16);
    const bool run_ok = gfirst >= bcol0 && gfirst + gcount <= min(bcol0 + ncols, cout);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = col_ok ? col + i : 0;
      int mode = col_ok ? epi.mode[c] : 3;
      e.dest[i] = epi.dest[c];
      const int g = epi.gate[c];
      // tables that point outside the output row or outside the block's run of gates
      // switch the column off
      if (e.dest[i] < 0 || e.dest[i] >= epi.c_dest || mode < 0 || mode > 2 ||
          (mode == 2 && (!run_ok || g < gfirst || g >= gfirst + gcount)))
        mode = 3;
      e.mg[i] = mode | ((mode == 2 ? g - bcol0 : col_ok ? c_t + i : 0) << 4);
      e.ca[i] = epi.scale[c];
      e.cb[i] = epi.add[c] - epi.shift[c] * e.ca[i] + (mode == 1 ? epi.pre[c] : 0.f);
    }
    e.any = (e.mg[0] & 15) != 3 || (e.mg[1] & 15) != 3 || (e.mg[2] & 15) != 3 || (e.mg[3] & 15) != 3;
    e.vec = (e.mg[0] & 15) != 3 && (e.mg[1] & 15) != 3 && (e.mg[2] & 15) != 3 &&
            (e.mg[3] & 15) != 3 && e.dest[1] == e.dest[0] + 1 && e.dest[2] == e.dest[0] + 2 &&
            e.dest[3] == e.dest[0] + 3 && ((e.dest[0] | epi.c_dest) & 3) == 0;
    const int gi = (tid % (kCN / 4));
    if (run_ok && gi < gcount) {
      const int g = gfirst + gi;
      e.gcl = g - bcol0;
      e.gca = epi.scale[g];
      e.gcb = epi.add[g] - epi.shift[g] * e.gca + epi.pre[g];
    }
    return e;
  };
  // of the workgroup's block of 64 columns; of a fifth group
  // (the parts form has no registers to keep them in: it loads them as a tile is written out)
  EpiConsts ec = {}, ecx = {};
  if constexpr (EPI && !PARTS) {
    ec = epi_consts(col0, kCN, tid);
    if constexpr (FIVE) ecx = epi_consts(xcol, 16, tid);
  }
  const int e_c_dest = epi.c_dest, e_act_s = epi.act_s, e_act_g = epi.act_g;
  auto flush_tile = [&](int row0, int rows, int slot0) __attribute__((always_inline)) {
    if (!kProducersFlush && producer) return;
    int tid = threadIdx.x;
    // (the parts form: or what follows from it alone is worked out ahead of the loop, kept in
    // scratch memory, and its loads stand between those of the rows)
    if constexpr (PARTS) asm volatile("" : "+v"(tid));
    if constexpr (FIVE && !EPI) {
      // the fifth column group (accumulator columns kCN .. kCN + 15): four threads a row
      if (xcol >= 0) {
        const float4v z = {0.f, 0.f, 0.f, 0.f};
        const int c4 = (tid & 3) * 4;
        for (int r = tid >> 2; r < rows; r += NTF / 4) {
          int sl = slot0 + r;
          if (sl >= T) sl -= T;
          float4v *ap = reinterpret_cast<float4v *>(acc + sl * kAS + kCN + c4);
          const float4v v = *ap;
          *ap = z;
          IO *gp = out + (int64_t)(row0 + r) * cout + xcol + c4;
          if ((cout & 3) == 0) {
            if (xcol + c4 < cout) Io<IO>::store_stream(gp, v);
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (xcol + c4 + i < cout) __builtin_nontemporal_store((IO)v[i], gp + i);
          }
        }
      }
    }
    if constexpr (TAIL) {
      // The four consumer waves each hold a partial sum of the one column group, in the
      // 16 columns a wave owns: add them up in the first 16, clear the others, and write
      // the tile out as any other.
      const float4v z = {0.f, 0.f, 0.f, 0.f};
      for (int r = tid >> 2; r < rows; r += NTF / 4) {
        int sl = slot0 + r;
        if (sl >= T) sl -= T;
        float4v *ap = reinterpret_cast<float4v *>(acc + sl * kAS + (tid & 3) * 4);
        const float4v v = (ap[0] + ap[4]) + (ap[8] + ap[12]);
        ap[0] = v;
        ap[4] = z;
        ap[8] = z;
        ap[12] = z;
      }
      __syncthreads();
    }
    if constexpr (EPI) {
      // Batch norm constants and gate applied on the way out (cout % 4 == 0).  Threads,
      // columns and rows as in the plain store below.  The 16 lanes of a row sit in one wave
      // and a wave's LDS operations execute in order: first the row's gates are replaced by
      // their activated values (lane l: gate l), then every lane reads its sums and the
      // gates of its columns, then the wave clears the row.
      // FAST: scalar activation none or relu, gate activation none or sigmoid -- a few instructions
      // per element and no branch (a taken branch costs a wave more than the arithmetic of
      // a whole row); the other activations go through act_fn.
      // (e: the constants; XG: the pass over a fifth group, whose 16 columns begin at
      // accumulator column kCN and belong to the first four of a row's 16 threads)
      auto rows_out = [&](auto fast_tag, auto x_tag, const EpiConsts &e) __attribute__((always_inline)) {
        constexpr bool FAST = decltype(fast_tag)::value;
        constexpr bool XG = decltype(x_tag)::value;
        constexpr int U = 2;
        constexpr int RS = NTF / (kCN / 4);
        const int r_t = tid / (kCN / 4), c_t = (tid % (kCN / 4)) * 4;
        const bool own = !XG || c_t < 16;  // the thread has columns
        constexpr int kCol0 = XG ? kCN : 0;
        const float4v z = {0.f, 0.f, 0.f, 0.f};
        // FAST: max(t, lo) is the scalar activation where there is one, t elsewhere
        float lo[4];
        bool gated[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          lo[i] = ((e.mg[i] & 15) == 1 && e_act_s == SSC_ACT_RELU) ? 0.f : -INFINITY;
          gated[i] = (e.mg[i] & 15) == 2;
        }
        auto gate_act = [&](float x) -> float {
          const float u = x * e.gca + e.gcb;
          if constexpr (FAST)
            return e_act_g == SSC_ACT_SIGMOID ? __builtin_amdgcn_rcpf(1.f + __expf(-u)) : u;
          else
            return act_fn(e_act_g, u);
        };
        IO *gp = out + (int64_t)(row0 + r_t) * e_c_dest;
        const int64_t gstep = (int64_t)RS * e_c_dest;
        for (int r = r_t; r < rows; r += U * RS) {
          const bool two = r + RS < rows;
          int sl0 = slot0 + r, sl1 = slot0 + r + RS;
          if (sl0 >= T) sl0 -= T;
          if (sl1 >= T) sl1 -= T;
          float *a0 = acc + sl0 * kAS + kCol0, *a1 = acc + sl1 * kAS + kCol0;
          if (e.gcl >= 0) {
            const float x0 = a0[e.gcl], x1 = two ? a1[e.gcl] : 0.f;
            if constexpr (PARTS) {
              check.sum(x0);
              check.sum(x1);
            }
            a0[e.gcl] = gate_act(PARTS ? x0 * unscale : x0);
            if (two) a1[e.gcl] = gate_act(PARTS ? x1 * unscale : x1);
          }
          __builtin_amdgcn_sched_barrier(0);
          float4v v0 = own ? *reinterpret_cast<float4v *>(a0 + c_t) : z, v1 = z, g1 = z;
          float4v g0 = {a0[e.mg[0] >> 4], a0[e.mg[1] >> 4], a0[e.mg[2] >> 4], a0[e.mg[3] >> 4]};
          if (two) {
            if (own) v1 = *reinterpret_cast<float4v *>(a1 + c_t);
            g1 = float4v{a1[e.mg[0] >> 4], a1[e.mg[1] >> 4], a1[e.mg[2] >> 4], a1[e.mg[3] >> 4]};
          }
          if constexpr (PARTS) {
            // (a gate's column holds its activated value by now: its sum was looked at above)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const bool stored = (e.mg[i] & 15) != 3;
              check.sum(stored ? v0[i] : 0.f);
              check.sum(stored ? v1[i] : 0.f);
              v0[i] *= unscale;
              v1[i] *= unscale;
            }
          }
          __builtin_amdgcn_sched_barrier(0);  // the clears stay behind every read above
          if (own) *reinterpret_cast<float4v *>(a0 + c_t) = z;
          if (two && own) *reinterpret_cast<float4v *>(a1 + c_t) = z;
          if (e.any) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
              if (u == 1 && !two) break;
              const float4v v = u == 0 ? v0 : v1, gv = u == 0 ? g0 : g1;
              float4v y;
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const float t = v[i] * e.ca[i] + e.cb[i];
                if constexpr (FAST) {
                  y[i] = fmaxf(t, lo[i]) * (gated[i] ? gv[i] : 1.f);
                } else {  // every form, then select: no divergent branches
                  const float ts = act_fn(e_act_s, t);
                  const int m = e.mg[i] & 15;
                  y[i] = m == 1 ? ts : m == 2 ? t * gv[i] : t;
                }
              }
              IO *p = gp + u * gstep;
              if (e.vec) {
                Io<IO>::store_stream(p + e.dest[0], y);
              } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                  if ((e.mg[i] & 15) != 3) __builtin_nontemporal_store((IO)y[i], p + e.dest[i]);
              }
            }
          }
          gp += U * gstep;
        }
      };
      if constexpr (PARTS) ec = epi_consts(col0, kCN, tid);
      const bool fast = (e_act_s == SSC_ACT_NONE || e_act_s == SSC_ACT_RELU) &&
                        (e_act_g == SSC_ACT_NONE || e_act_g == SSC_ACT_SIGMOID);
      if constexpr (FIVE) {
        if (xcol >= 0) {
          if (fast)
            rows_out(std::true_type(), std::true_type(), ecx);
          else
            rows_out(std::false_type(), std::true_type(), ecx);
        }
      }
      if (fast)
        rows_out(std::true_type(), std::false_type(), ec);
      else
        rows_out(std::false_type(), std::false_type(), ec);
      return;
    }
    if ((cout & 3) == 0) {
      // A thread keeps its 4 columns and walks down the rows, NTF / (kCN / 4) rows per
      // step: addresses advance by constants, so a step is little more than its LDS
      // read, LDS clear and store, and four reads are in flight before the first store
      // (one at a time, every step would pay the full LDS latency while the matrix
      // cores idle).
      const float4v z = {0.f, 0.f, 0.f, 0.f};
      constexpr int U = 4;
      constexpr int RS = NTF / (kCN / 4);  // rows per step
      const int r_t = tid / (kCN / 4), c_t = (tid % (kCN / 4)) * 4;
      const bool col_ok = col0 + c_t < cout;
      IO *gp = out + (int64_t)(row0 + r_t) * cout + col0 + c_t;
      const int64_t gstep = (int64_t)RS * cout;
      for (int r = r_t; r < rows; r += U * RS) {
        float4v v[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (r + u * RS < rows) {
            int sl = slot0 + r + u * RS;
            if (sl >= T) sl -= T;
            float4v *ap = reinterpret_cast<float4v *>(acc + sl * kAS + c_t);
            v[u] = *ap;
            *ap = z;
            if constexpr (PARTS) {
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                check.sum(v[u][i]);
                v[u][i] *= unscale;
              }
            }
          }
#pragma unroll
        for (int u = 0; u < U; ++u)
          // streaming store: the output is not read again by this kernel and must not
          // push the weights and the gathered rows out of L2
          if (r + u * RS < rows && col_ok)
            Io<IO>::store_stream(gp + u * gstep, v[u]);
        gp += U * gstep;
      }
    } else {
      for (int e = tid; e < rows * kCN; e += NTF) {
        int r = e / kCN, c = e % kCN;
        int sl = slot0 + r;
        if (sl >= T) sl -= T;
        if constexpr (PARTS) check.sum(acc[sl * kAS + c]);
        if (col0 + c < cout)
          __builtin_nontemporal_store((IO)(PARTS ? acc[sl * kAS + c] * unscale : acc[sl * kAS + c]),
                                      out + (int64_t)(row0 + r) * cout + col0 + c);
        acc[sl * kAS + c] = 0.f;
      }
    }
  };
  // The tile of stage `pos` (first row, rows) ends with it when the group is the
  // tile's last one and the chunk is the last chunk.  Scalar loads: the address is
  // uniform.
  auto tile_end = [&](const StagePos &pos, int &row0, int &rows, int &slot0) -> bool {
    const int32_t *m = grp_meta + (int64_t)pos.g * 8;
    row0 = m[4];
    slot0 = m[6];
    const int r = m[5];
    rows = r < 0 ? -r : r;
    return r > 0 && pos.cc == nch - 1;
  };

  // ---------------------------------------------------------------- the bfloat16-parts form
  // The plan's blocks are kBP = 16 NB pairs of one offset (NB row blocks, 2 or 4).  A stage is two
  // blocks x 32 input channels, one matrix step of v_mfma_f32_16x16x32_bf16; two stages are a
  // chunk.  Consumer wave (r, c) multiplies block r with the 32 columns c of the workgroup's
  // 64: a weight fragment serves 16 NB rows, a staged row 32 columns.  Producers cut the gathered
  // rows into parts on their way into LDS, the filters come in parts (conv_pack.h).
  // A stage's barrier stands before its last row block: by then the consumers hold that in
  // registers and the next stage is in LDS; its first row block is read during the last one's
  // products.
  // The products of a chunk are summed by themselves and then added to those of the chunks
  // before (one rounding at the sum's size a chunk, not twelve); a group's stay in registers.
  // Waves (0, c) and (1, c) have the same columns and may have the same output rows: (0, c) adds
  // its products of a group to the accumulators during the first stage of the next group and
  // (1, c) during the second, or one after the other when the tile ends: every sum in the
  // order of the schedule.
  //
  // What the parts cannot do is worked out again with float instructions: a workgroup that has
  // met one of the following walks its groups a second time (see the end of the form).
  //  - Infinities, NaN, elements of 2^111 and sums of 2^95 or more (an infinity among the scaled
  //    parts): a sum not finite.
  //  - Sums that are not zero and below 2^-126 (scaled: 2^-94): six products of parts, each rounded
  //    at 2^-150.
  // (Without the scale elements with bits below 2^-133 and sums below 2^-95 went that way too, and
  // one such element sent a workgroup through its range a second time: 128 -> 64 channels, every row,
  // 756 us with a single one and 936 with one in every workgroup, where the float form takes 283.)
  //
  // What bounds it (128 -> 64 channels, 216 stages of 48 matrix instructions a wave, 185 us): a
  // stage is 788 cycles of matrix instructions and takes about 1800; LDS (48 reads of a KiB at 4-8
  // cycles, 48 writes of 512 bytes at 8) and the vector memory path (40 KiB at 64 bytes a cycle)
  // are busy 600-700 cycles each, the producers' cutting 450-500, which share the SIMDs with the
  // products; none of them alone sets the pace.  Blocks of 64 halve the fragment loads of a product
  // and the barriers, and pad more; four row blocks leave registers for two stages of fragments.
  // Error against 64 bits, float form -> parts (times stand at parts_block, conv.hip):
  //   128 -> 64   2.0e-7 -> 1.5e-7      512 -> 608   2.6e-7 -> 1.6e-7
  //   128 -> 304  1.8e-7 -> 1.3e-7      608 -> 512   3.3e-7 -> 1.8e-7
  //   256 -> 608  2.1e-7 -> 1.4e-7      304 -> 128   1.7e-7 -> 1.2e-7
  // With the sums of all chunks in one chain the error of the wide ones is 2.7e-7 to 4.1e-7.
  if constexpr (PARTS) {
    constexpr int NB = FORM == 5 ? 4 : 2;
    constexpr int GS = NB / 2;                  // groups of the schedule to a stage
    constexpr int kStageB = 2 * NB * 3 * 1024;  // bytes of a staged stage
    const int g_last = g_end - GS;
    const int n_ck = (g_end - g_begin) / GS * nch;  // chunks of this workgroup
    char *const abytes = reinterpret_cast<char *>(abuf);
    int *const odd_s = reinterpret_cast<int *>(abytes + 2 * kStageB);
    const __amdgpu_buffer_rsrc_t rs_feat =
        __builtin_amdgcn_make_buffer_rsrc((void *)features, 0, (int)feat_bytes, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t rs_w =
        __builtin_amdgcn_make_buffer_rsrc((void *)packed, 0, (int)packed_bytes, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t rs_in =
        __builtin_amdgcn_make_buffer_rsrc((void *)sched_in, 0, (int)sched_bytes, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t rs_out =
        __builtin_amdgcn_make_buffer_rsrc((void *)sched_out, 0, (int)sched_bytes, kRsrcFlags);
    if (n_ck == 0) return;  // (the whole workgroup)
    if (tid == 0) odd_s[0] = 0;
    // A staged row block is, part by part, a KiB in the order of the consumers' lanes: lane
    // (l16, g) has the 16 bytes at 256 g + 16 (l16 ^ swizzle(g)), which neither their reads
    // nor the producers' writes meet banks twice with (reads 4-7 cycles a KiB, where rows of
    // 192 + 16 bytes take 8; writes 8 cycles for 512 bytes either way).
    auto swizzle = [](int g) -> int { return (0x84C0 >> (4 * g)) & 15; };  // 0, 12, 4, 8
    if (producer) {
      const PartsCut cut;
      const int pt = tid - NCW * 64;
      const int row = pt >> 3;   // this thread's pairs: row, row + 32, ...
      const int piece = pt & 7;  // its four channels of a stage
      const bool beyond[2] = {(nch - 1) * 64 + piece * 4 >= cin, (nch - 1) * 64 + 32 + piece * 4 >= cin};
      // lane group g of an operand has channels 4 g .. + 3 and 16 + 4 g .. + 3 of a stage, as
      // in the packed filters
      char *const st_base = abytes + (row >> 4) * 3072 + (piece & 3) * 256 +
                            (((row & 15) ^ swizzle(piece & 3)) * 16) + (piece >> 2) * 8;
      // rows[s % RD]: the rows of stage s, RD stages (RC chunks) in flight; idx[c % 4]: the
      // gather offsets of chunk c, four chunks further (loads return in order: a wait for
      // offsets is one for the rows that were asked for before them)
      constexpr int RD = 16 / NB, RC = RD / 2;
      int idx[4][NB];
      float4v rows[RD][NB];
      auto load_idx = [&](const PartsPos &pos, int (&ix)[NB]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NB; ++j) ix[j] = buf_load1(rs_in, row * 4 + j * 128, pos.g * 256);
      };
      auto load_rows = [&](const PartsPos &pos, int ks, const int (&ix)[NB], float4v (&v)[NB])
          __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          int off = ix[j];
          if constexpr (GATHER == 2) off = (pos.cc == nch - 1 && beyond[ks]) ? (int)kGatherPad : off;
          v[j] = buf_load4(rs_feat, off + piece * 16, pos.cc * 256 + ks * 128);
        }
      };
      auto store_rows = [&](int buf, const float4v (&v)[NB]) __attribute__((always_inline)) {
        int2v p[NB][3];
        cut.all(v, p);
        char *dst = st_base + buf * kStageB;
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int i = 0; i < 3; ++i)
            *reinterpret_cast<int2v *>(dst + j * 2 * 3072 + i * 1024) = p[j][i];
      };
      PartsPos p_rows = {g_begin, 0}, p_idx = {g_begin, 0}, p_cur = {g_begin, 0};
      {
        // stage 0 goes to LDS, the rows of stages 1 .. RD stay in flight, and the offsets of
        // chunks RC .. RC + 3; loads in the order in which the loop waits for them
        int ix[RC][NB];
#pragma unroll
        for (int c = 0; c < RC; ++c) {
          load_idx(p_idx, ix[c]);
          p_idx.advance(GS, nch, g_last);
        }
#pragma unroll
        for (int c = RC; c < RC + 4; ++c) {
          load_idx(p_idx, idx[c & 3]);
          p_idx.advance(GS, nch, g_last);
        }
        float4v r0[NB];
        load_rows(p_rows, 0, ix[0], r0);
#pragma unroll
        for (int s = 1; s < RD; ++s) {
          if ((s & 1) == 0) p_rows.advance(GS, nch, g_last);
          load_rows(p_rows, s & 1, ix[s >> 1], rows[s]);
        }
        p_rows.advance(GS, nch, g_last);
        load_rows(p_rows, 0, idx[RC & 3], rows[0]);
        store_rows(0, r0);
      }
      // (tile rows of the chunk's group, negative unless it ends with the group: read a chunk ahead)
      int tile_rows = grp_meta[(int64_t)(g_begin + GS - 1) * 8 + 5];
      asm volatile("" : "+s"(tile_rows));  // (here: a load still out would be waited for in the loop)
      __syncthreads();  // stage 0 is there
      // Chunk c, stages s and s + 1: the rows of s + 1 and s + 2 are staged, those of s + 1 + RD
      // (chunk c + RC) and s + 2 + RD and the offsets of chunk c + RC + 4 are asked for.
      auto chunk = [&](auto phase) __attribute__((always_inline)) {
        constexpr int ph = decltype(phase)::value;  // == c % 4
        constexpr int r1 = (2 * ph + 1) % RD, r2 = (2 * ph + 2) % RD, i1 = (ph + RC) & 3,
                      i2 = (ph + RC + 1) & 3;
        const int g_cur = p_cur.g, n_rows = tile_rows;
        const bool last = n_rows > 0 && p_cur.cc == nch - 1;
        p_cur.advance(GS, nch, g_last);
        tile_rows = grp_meta[(int64_t)(p_cur.g + GS - 1) * 8 + 5];
        store_rows(1, rows[r1]);
        __builtin_amdgcn_sched_barrier(0);
        load_rows(p_rows, 1, idx[i1], rows[r1]);
        p_rows.advance(GS, nch, g_last);
        load_idx(p_idx, idx[i1]);
        p_idx.advance(GS, nch, g_last);
        __syncthreads();
        store_rows(0, rows[r2]);
        __builtin_amdgcn_sched_barrier(0);
        load_rows(p_rows, 0, idx[i2], rows[r2]);
        __syncthreads();
        if (last) {
          __syncthreads();
          __syncthreads();
          const int32_t *m = grp_meta + (int64_t)g_cur * 8;
          flush_tile(m[4], n_rows, m[6]);
          __syncthreads();
        }
      };
      int c = 0;
      for (; c + 4 <= n_ck; c += 4) {
        chunk(std::integral_constant<int, 0>());
        chunk(std::integral_constant<int, 1>());
        chunk(std::integral_constant<int, 2>());
        chunk(std::integral_constant<int, 3>());
      }
      if (c < n_ck) chunk(std::integral_constant<int, 0>());
      if (c + 1 < n_ck) chunk(std::integral_constant<int, 1>());
      if (c + 2 < n_ck) chunk(std::integral_constant<int, 2>());
    } else {
      // stages whose filters are in registers, and how far ahead they are asked for (a stage of
      // four row blocks lasts twice as long and leaves fewer registers)
      constexpr int WR = NB == 2 ? 4 : 2, AHEAD = WR - 1;
      const int g = lane >> 4, l16 = lane & 15;
      const int wr = wave >> 1, wc = wave & 1;
      const int parts_at = (int)(packed_bytes / (4096u + kPartFragBytes) * 4096u);
      const int cb0 = min(col0 / 16 + 2 * wc, ncb - 1), cb1 = min(col0 / 16 + 2 * wc + 1, ncb - 1);
      const int w_base[2] = {parts_at + cb0 * nch * kPartFragBytes,
                             parts_at + cb1 * nch * kPartFragBytes};
      const char *const a_base = abytes + wr * NB * 3072 + g * 256 + (l16 ^ swizzle(g)) * 16;
      typedef __attribute__((address_space(3))) float4v lds_float4v;
      const int acc_base = (int)(size_t)(__attribute__((address_space(3))) char *)acc;
      auto lds_load4 = [](int addr) -> float4v { return *(lds_float4v *)(size_t)addr; };
      auto lds_store4 = [](int addr, const float4v &v) { *(lds_float4v *)(size_t)addr = v; };
      const int acc_lane = acc_base + (wc * 32 + g * 4) * 4;  // (and 64 bytes on: the second group)
      // rings; the loop is unrolled over two chunks (four stages):
      //   w[s % WR]    filters of stage s [column group][part]
      //   a[b & 1]     rows of row block b [part], read from LDS one block ahead
      //   orow[c & 1]  accumulator rows of this lane's pairs in the group of chunk c
      int4v w[WR][2][3], a[2][3];
      int orow[2][NB];
      // sums [row block][column group]: of this chunk; of the group's chunks before or, during a
      // group's first chunk, of the group before; accumulators as they were read
      float4v t[NB][2], sum[NB][2], x[2][2];
      bool pending = false;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          t[b][i] = sum[b][i] = x[b & 1][i] = float4v{0.f, 0.f, 0.f, 0.f};
      auto kof_of = [&](const PartsPos &pos) -> int {
        return grp_meta[(int64_t)pos.g * 8 + (NB == 2 ? 2 * wr : 8 * wr)];
      };
      // byte offset of a chunk's filters but for the column group's part (packed as floats an
      // offset's filters are k_scale bytes, in parts 3/2 of that)
      auto soff_of = [](int kof, int cc) -> int { return (int)((unsigned)kof / 2u * 3u) + cc * kPartFragBytes; };
      auto load_w = [&](int soff, int ks, int i, int p) __attribute__((always_inline)) -> int4v {
        return __builtin_bit_cast(
            int4v, buf_load4(rs_w, lane * 16 + ks * 3072 + p * 1024, soff + w_base[i]));
      };
      auto load_orow = [&](const PartsPos &pos, int (&o)[NB]) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
          o[b] = buf_load1(rs_out, l16 * 4 + (wr * NB + b) * 64, pos.g * 256);
      };
      auto read_a = [&](int buf, int b, int part) __attribute__((always_inline)) -> int4v {
        return *reinterpret_cast<const int4v *>(a_base + buf * kStageB + b * 3072 + part * 1024);
      };
      PartsPos p_cur = {g_begin, 0}, p_next = {g_begin, 0}, p_f = {g_begin, 0};
      p_next.advance(GS, nch, g_last);
      int soff = soff_of(kof_of(p_f), 0);  // filters of the chunk that are asked for next
      p_f.advance(GS, nch, g_last);
#pragma unroll
      for (int st = 0; st < AHEAD; ++st)  // in the loop's order: stage by stage, part by part
#pragma unroll
        for (int p = 2; p >= 0; --p)
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            if (st == 2 && p == 2 && i == 0) {
              soff = soff_of(kof_of(p_f), p_f.cc);
              p_f.advance(GS, nch, g_last);
            }
            w[st][i][p] = load_w(soff, st & 1, i, p);
          }
      load_orow(p_cur, orow[0]);
      int kof = kof_of(p_f);  // of the chunk behind soff's
      int tile_rows = grp_meta[(int64_t)(g_begin + GS - 1) * 8 + 5];  // (as in the producers)
      asm volatile("" : "+s"(tile_rows), "+s"(kof));
      __syncthreads();
#pragma unroll
      for (int p = 0; p < 3; ++p) a[0][p] = read_a(0, 0, p);
      // two row blocks of the group before: h = 0 or 1
      auto commit_read = [&](const int (&o)[NB], int h) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 2; ++i) x[b][i] = lds_load4(o[2 * h + b] + acc_lane + i * 64);
      };
      auto commit_write = [&](const int (&o)[NB], int h) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 2; ++i)
            lds_store4(o[2 * h + b] + acc_lane + i * 64, x[b][i] + sum[2 * h + b][i]);
      };
      // the products of parts, the smallest first
      constexpr int kWp[6] = {2, 0, 1, 1, 0, 0}, kAp[6] = {0, 2, 1, 0, 1, 0};
      // One chunk.  Everything a stage needs besides its products lies between them, and the
      // branches in it are short: what they hold shares no registers with loads in flight.
      auto chunk = [&](auto phase) __attribute__((always_inline)) {
        constexpr int cp = decltype(phase)::value;  // == c % 2
        const int g_cur = p_cur.g, n_rows = tile_rows;
        const bool grp_first = p_cur.cc == 0, grp_last = p_cur.cc == nch - 1;
        const bool commit = pending && grp_first;
        // (a first chunk's products take the place of the sums: a factor and no branch)
        const float keep = grp_first ? 0.f : 1.f;
        auto add_up = [&](int b, int i) __attribute__((always_inline)) {
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[b][i][e] = __builtin_fmaf(sum[b][i][e], keep, t[b][i][e]);
        };
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const int cur = (2 * cp + ks) % WR, nxt = (2 * cp + ks + AHEAD) % WR;
          const bool turn = commit && wr == ks;
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            if (b == NB - 1) __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int p = 0; p < 6; ++p) {
#pragma unroll
              for (int i = 0; i < 2; ++i)
                t[b][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(bf16x8, w[cur][i][kWp[p]]),
                    __builtin_bit_cast(bf16x8, a[b & 1][kAp[p]]),
                    ks == 0 && p == 0 ? float4v{0.f, 0.f, 0.f, 0.f} : t[b][i], 0, 0, 0);
              if (p < 3) {  // the next row block's rows
                constexpr int kRead[3] = {0, 2, 1};
                a[(b + 1) & 1][kRead[p]] =
                    b < NB - 1 ? read_a(ks, b + 1, kRead[p]) : read_a(ks ^ 1, 0, kRead[p]);
              }
              if (b == 0 && p >= 1 && p < 4) {  // the filters of stage s + AHEAD
#pragma unroll
                for (int i = 0; i < 2; ++i)
                  w[nxt][i][3 - p] = load_w(soff, (ks + AHEAD) & 1, i, 3 - p);
              }
              if (b < NB / 2 && p == 0 && turn) commit_read(orow[cp ^ 1], b);
              if (b < NB / 2 && p == 4 && turn) commit_write(orow[cp ^ 1], b);
              if (ks == 1 && b > 0 && (p == 2 || p == 3)) add_up(b - 1, p - 2);
              if (ks == 1 && b == NB - 1 && p == 4) load_orow(p_next, orow[cp ^ 1]);
              if (ks == 0 && b == NB - 2 && p == 3) {
                // from here on the next chunk's filters are asked for, or its successor's (stage
                // s + AHEAD); the next chunk's tile.  (Scalar loads: behind the row block's last
                // wait for LDS data, which they would turn into a wait for everything.)
                soff = soff_of(kof, p_f.cc);
                p_f.advance(GS, nch, g_last);
                kof = kof_of(p_f);
                tile_rows = grp_meta[(int64_t)(p_next.g + GS - 1) * 8 + 5];
              }
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) add_up(NB - 1, i);
        p_cur.advance(GS, nch, g_last);
        p_next.advance(GS, nch, g_last);
        if (commit) pending = false;
        if (grp_last) pending = true;
        if (grp_last && n_rows > 0) {
#pragma unroll
          for (int r = 0; r < 2; ++r) {
            if (wr == r) {
#pragma unroll
              for (int h = 0; h < NB / 2; ++h) {
                commit_read(orow[cp], h);
                commit_write(orow[cp], h);
              }
            }
            __syncthreads();
          }
          pending = false;
          const int32_t *m = grp_meta + (int64_t)g_cur * 8;
          flush_tile(m[4], n_rows, m[6]);
          // (nothing of these is wanted behind a tile: no registers for them while it is written)
#pragma unroll
          for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < 2; ++i) sum[b][i] = x[b & 1][i] = float4v{0.f, 0.f, 0.f, 0.f};
          __syncthreads();
        }
      };
      int c = 0;
      for (; c + 2 <= n_ck; c += 2) {
        chunk(std::integral_constant<int, 0>());
        chunk(std::integral_constant<int, 1>());
      }
      if (c < n_ck) chunk(std::integral_constant<int, 0>());
    }
    // (all waves are behind the last tile's last barrier: every range ends with a tile's end)
    if (check.odd()) odd_s[0] = 1;
    __syncthreads();
    if (odd_s[0] == 0) return;
    unscale = 1.f;
    // The workgroup's tiles again, on float instructions: consumer wave w has columns 16 w .. of
    // the 64 and walks the row blocks in order, operands straight from memory.  Rare, and 3.4 times
    // as slow as the float form; its sums are no further off (128 -> 64 channels, every row: 1.8e-7
    // against 2.0e-7; with all chunks of a group in one chain 2.3e-7).
    {
      const int g = lane >> 4, l16 = lane & 15;
      const int w_base = min(col0 / 16 + (producer ? 0 : wave), ncb - 1) * nch * 4096;
      float *const acc_lane = acc + (producer ? 0 : wave) * 16 + g * 4;
      for (int gi = g_begin; gi < g_end; ++gi) {
        if (!producer) {
          float4v d[4];
          int in_off[4], out_off[4], kof[4];
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            d[b] = float4v{0.f, 0.f, 0.f, 0.f};
            in_off[b] = sched_in[(int64_t)gi * 64 + b * 16 + l16];
            out_off[b] = sched_out[(int64_t)gi * 64 + b * 16 + l16];
            kof[b] = grp_meta[(int64_t)gi * 8 + b];
          }
          for (int cc = 0; cc < nch; ++cc)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
              float4v av[4], wv[4], t = {0.f, 0.f, 0.f, 0.f};  // (a chunk's products by themselves)
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                int off = in_off[b];
                if (GATHER == 2 && cc * 64 + q * 16 + g * 4 >= cin) off = (int)kGatherPad;
                av[q] = buf_load4(rs_feat, off + q * 64 + g * 16, cc * 256);
                wv[q] = buf_load4(rs_w, lane * 16 + q * 1024, kof[b] + w_base + cc * 4096);
              }
#pragma unroll
              for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                  t = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[q][j], av[q][j], t, 0, 0, 0);
              d[b] += t;
            }
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            float4v *to = reinterpret_cast<float4v *>(reinterpret_cast<char *>(acc_lane) + out_off[b]);
            *to += d[b];
          }
        }
        const int32_t *m = grp_meta + (int64_t)gi * 8;
        if (m[5] > 0) {
          __syncthreads();
          flush_tile(m[4], m[5], m[6]);
          __syncthreads();
        }
      }
    }
    return;
  }

  if (producer) {
    // ------------------------------------------------------------------ producer
    const int pt = tid - NCW * 64;
    constexpr int RD = kRowsAhead, ID = kIdxAhead;
    static_assert(RD == 4 && ID == 2, "the rings below are sized for these distances");
    const __amdgpu_buffer_rsrc_t rs_in =
        __builtin_amdgcn_make_buffer_rsrc((void *)sched_in, 0, (int)sched_bytes, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t rs_feat =
        __builtin_amdgcn_make_buffer_rsrc((void *)features, 0, (int)feat_bytes, kRsrcFlags);
    const int idx_voff = (pt >> 4) * 4;    // this thread's slot (plus 16 slots per element)
    const int piece = pt & 15;                  // this thread's 4 channels of a row chunk
    const int chunk_off = piece * 4 * kEB;
    // the chunk has no such piece (fewer than 16 steps), or, in the last chunk, the piece
    // lies beyond Cin
    const bool no_piece = !kHalf && piece >= NS;
    const bool beyond_cin = (nch - 1) * kChunk + piece * 4 >= cin;
    // a piece of the partly used quarter is staged one channel per lane group
    const bool spread = !kHalf && kQRem != 0 && piece >= 4 * kQFull && piece < NS;
    typedef Raw Held;
    int idx[ID][NE];
    Held rows[RD][NE];
    // Rings indexed by stage number: rows of stage st in rows[st & 3], gather offsets
    // in idx[st & 1].  The loop is unrolled four times so that every ring index is a
    // compile-time constant: rotating a ring through register moves would read
    // registers that loads are still writing, and so wait for those loads one
    // iteration after their issue.
    auto load_idx = [&](const StagePos &pos, int s, int (&ix)[NE]) {
#pragma unroll
      for (int j = 0; j < NE; ++j) {
        int v = buf_load1(rs_in, idx_voff + j * 64, pos.g * 256);
        if (GATHER == 0) v = s < nstages ? v : -1;  // the pointer gather is not range-checked
        ix[j] = v;
      }
    };
    auto load_rows = [&](const StagePos &pos, const int (&ix)[NE], Held (&r)[NE]) {
#pragma unroll
      for (int j = 0; j < NE; ++j) {
        if constexpr (GATHER == 1) {
          r[j] = Io<IO>::gather(rs_feat, ix[j] + chunk_off, pos.cc * (kChunk * kEB));
        } else if constexpr (GATHER == 2) {
          const int off =
              (no_piece || (pos.cc == nch - 1 && beyond_cin)) ? (int)kGatherPad : ix[j];
          r[j] = Io<IO>::gather(rs_feat, off + chunk_off, pos.cc * (kChunk * kEB));
        } else {
          const int ch = pos.cc * kChunk + piece * 4;
          const int row = ix[j] < 0 ? 0 : ix[j];  // padding slots read row 0 and drop it
          const IO *fp = features + (int64_t)row * cin + ch;
          Held v = Io<IO>::zero();
          if ((cin & 3) == 0) {
            if (ch < cin) v = Io<IO>::load(fp);
          } else {  // rows are not aligned: one element at a time
            v = Io<IO>::load_first(fp, cin - ch);
          }
          if (ix[j] < 0 || no_piece) v = Io<IO>::zero();
          r[j] = v;
        }
      }
    };
    // where this thread's piece goes in a staged row: its own 16 bytes, or, for a piece of
    // the partly used quarter, element (piece - 4 kQFull) of each lane group's 16 bytes
    const int r16 = pt >> 4;  // the rows' number in their row blocks
    char *const st_base = reinterpret_cast<char *>(abuf) + r16 * kRowB +
                          (spread  ? (piece - 4 * kQFull) * kEB
                           : kHalf ? staged_piece<true>(piece >> 1, r16) + (piece & 1) * 8
                                   : staged_piece<false>(piece, r16));
    int spread_at[4];  // pieces of the four lane groups in the partly used quarter
#pragma unroll
    for (int i = 0; i < 4; ++i) spread_at[i] = staged_piece<false>((4 * kQFull + i) & 15, r16);
    auto store_rows = [&](int parity, const Held (&r)[NE]) {
#pragma unroll
      for (int j = 0; j < NE; ++j) {
        char *dst = st_base + (parity * kStage + j * 16) * kRowB;
        if constexpr (!kHalf && kQRem != 0) {
          if (spread) {
            const float4v v = __builtin_bit_cast(float4v, r[j]);
#pragma unroll
            for (int i = 0; i < 4; ++i) *reinterpret_cast<float *>(dst + spread_at[i]) = v[i];
            continue;
          }
        }
        if (!no_piece) *reinterpret_cast<Held *>(dst) = r[j];
      }
    };
    // Prologue.  Loads are issued in the order the loop will wait for them (offsets,
    // then rows, oldest stage first): the wait counts of the loop are static, so
    // they must also be right on its first trip.
    StagePos p_rows = {g_begin, 0};  // stage whose rows are loaded next
    StagePos p_idx = {g_begin, 0};   // stage whose gather offsets are loaded next
    StagePos p_cur = {g_begin, 0};   // stage the consumers are working on
    {
      int ix[RD + 1][NE];
#pragma unroll
      for (int j = 0; j <= RD; ++j) {
        load_idx(p_idx, j, ix[j]);
        p_idx.advance(nch);
      }
#pragma unroll
      for (int j = 1; j <= ID; ++j) {
        load_idx(p_idx, RD + j, idx[(RD + j) & 1]);
        p_idx.advance(nch);
      }
      Held r0[NE];
      load_rows(p_rows, ix[0], r0);
      p_rows.advance(nch);
#pragma unroll
      for (int j = 1; j <= RD; ++j) {
        load_rows(p_rows, ix[j], rows[j & 3]);
        p_rows.advance(nch);
      }
      store_rows(0, r0);
    }
    __syncthreads();
    // Iteration s stages the rows of stage s+1 and issues the loads of stages s+5
    // (rows) and s+7 (gather offsets).
    auto iteration = [&](int s, auto phase) {
      constexpr int ph = decltype(phase)::value;  // == s & 3
      int t_row0, t_rows, t_slot0;
      const bool last = tile_end(p_cur, t_row0, t_rows, t_slot0);
      p_cur.advance(nch);
      store_rows((ph + 1) & 1, rows[(ph + 1) & 3]);
      load_rows(p_rows, idx[(ph + 1 + RD) & 1], rows[(ph + 1 + RD) & 3]);
      p_rows.advance(nch);
      load_idx(p_idx, s + 1 + RD + ID, idx[(ph + 1 + RD + ID) & 1]);
      p_idx.advance(nch);
      __syncthreads();
      if (last) {
        if constexpr (FIVE) {  // the consumers add the last group's fifth-group products
#pragma unroll
          for (int i = 0; i < 4; ++i) __syncthreads();
        }
        flush_tile(t_row0, t_rows, t_slot0);
        __syncthreads();
      }
    };
    // Whole groups of four stages first, the remainder after the loop: an early exit
    // from the middle of the unrolled body would share the loop's back edge, and the
    // static wait counts at the top of the body would then have to allow for a trip
    // that follows a shorter one.
    int s = 0;
    for (; s + 4 <= nstages; s += 4) {
      iteration(s, std::integral_constant<int, 0>());
      iteration(s + 1, std::integral_constant<int, 1>());
      iteration(s + 2, std::integral_constant<int, 2>());
      iteration(s + 3, std::integral_constant<int, 3>());
    }
    if (s < nstages) iteration(s, std::integral_constant<int, 0>());
    if (s + 1 < nstages) iteration(s + 1, std::integral_constant<int, 1>());
    if (s + 2 < nstages) iteration(s + 2, std::integral_constant<int, 2>());
  } else {
    // ------------------------------------------------------------------ consumer
    const int g = lane >> 4;
    const int l16 = lane & 15;
    // A column group beyond Cout multiplies with the last real one's fragments; its
    // accumulator columns are never written out.
    // (The one-column-group form: every wave multiplies with the fragments of that group.)
    const int cb = TAIL ? col_base / 16 : min(col0 / 16 + wave, ncb - 1);
    const __amdgpu_buffer_rsrc_t rs_w =
        __builtin_amdgcn_make_buffer_rsrc((void *)packed, 0, (int)packed_bytes, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t rs_out =
        __builtin_amdgcn_make_buffer_rsrc((void *)sched_out, 0, (int)sched_bytes, kRsrcFlags);
    // 16-byte pieces of operands a lane handles per row block: weight fragment loads, and
    // as many reads of its staged row (float: 4 MFMA steps of 4 channels each, a quarter
    // of the chunk; half: one MFMA step of 32 channels, lane group g has 8 of them)
    constexpr int NF = kHalf ? 2 : (NS + 3) / 4;
    typedef std::conditional_t<kHalf, int4v, float4v> Frag;
    const int w_voff = lane * 16;  // this lane's 16 bytes of a KiB of fragments
    constexpr int kWStep = 1024;   // from one 16-byte piece to the next
    const int w_soff0 = cb * nch * kFragB;  // fragments of this wave's column block
    // this lane's 16 bytes of quarter q of its row in a row block
    const char *a_base[NF];
#pragma unroll
    for (int q = 0; q < NF; ++q)
      a_base[q] = reinterpret_cast<const char *>(abuf) + l16 * kRowB +
                  staged_piece<kHalf>(4 * q + g, l16);
    // The accumulators are addressed with 32-bit LDS byte addresses (acc_lane includes
    // the base of acc): no pointer arithmetic left for the vector ALU.
    typedef __attribute__((address_space(3))) float4v lds_float4v;
    const int acc_base = (int)(size_t)(__attribute__((address_space(3))) char *)acc;
    auto lds_load4 = [](int addr) -> float4v { return *(lds_float4v *)(size_t)addr; };
    auto lds_store4 = [](int addr, const float4v &v) { *(lds_float4v *)(size_t)addr = v; };

    const __amdgpu_buffer_rsrc_t rs_meta =
        __builtin_amdgcn_make_buffer_rsrc((void *)grp_meta, 0, (int)meta_bytes, kRsrcFlags);
    // Per-lane state of the consumer pipeline.  Row blocks are numbered through the
    // stages (block 4s+m is block m of stage s); rings are indexed with the block or
    // stage number, and the loop is unrolled over two stages so that every ring index
    // is a compile-time constant.
    //   w[b & 3][q]   weight fragments of block b (four 16-byte loads), fetched three
    //                 blocks ahead: while block b multiplies, the slot of block b-1 is
    //                 refilled for block b+3
    //   orow[b & 3]   LDS byte offset of the accumulator row of this lane's pair in block b
    //   rec[s & 1]    the schedule record (offsets of the 4 blocks, rows of the tile)
    //                 of stage s, the same in every lane.  It travels through vector
    //                 loads and v_readfirstlane rather than scalar loads: scalar loads
    //                 return out of order, and one in flight would turn every partial
    //                 wait for LDS data below into a wait for everything.
    Frag w[4][NF];
    int orow[4];
    int4v rec[2][2];
    // Second half of a record: only its first three words are used.  A 12-byte load:
    // a wider one would still write the unused register when it lands, and whatever
    // the compiler keeps there in the meantime would have to wait for it.
    auto load_rec_tail = [&](const StagePos &pos) -> int4v {
      const int3v t = buf_load3(rs_meta, 16, pos.g * 32);
      return int4v{t.x, t.y, t.z, 0};
    };
    // First row and rows of the tile of a stage, and whether the tile ends with the
    // stage, from the second half of its record.
    struct TileEnd {
      int row0, rows, slot0;
      bool last;
    };
    auto tile_end_of = [&](const int4v &tail, const StagePos &pos) -> TileEnd {
      TileEnd e;
      e.row0 = __builtin_amdgcn_readfirstlane(tail.x);
      const int r = __builtin_amdgcn_readfirstlane(tail.y);
      e.rows = r < 0 ? -r : r;
      e.slot0 = __builtin_amdgcn_readfirstlane(tail.z);
      e.last = r > 0 && pos.cc == nch - 1;
      return e;
    };
    auto load_rec = [&](const StagePos &pos, int4v (&r)[2]) {
      r[0] = __builtin_bit_cast(int4v, buf_load4(rs_meta, 0, pos.g * 32));
      r[1] = load_rec_tail(pos);
    };
    // Byte offset of the weight fragments of a block: the offset's part comes from the
    // schedule record (0 for empty blocks and, the loads being range-checked, for
    // records beyond the schedule), `base` is the part of this wave and channel chunk.
    auto frag_soff = [&](int rec_lane, int base) -> int {
      return __builtin_amdgcn_readfirstlane(rec_lane) + base;
    };
    auto rec_k = [](const int4v &v, int b) -> int {
      return b == 0 ? v.x : b == 1 ? v.y : b == 2 ? v.z : v.w;
    };
    auto fetch_frag = [&](Frag &dst, int soff, int q) {
      if constexpr (!kHalf && kQRem != 0) {
        if (q == kQFull) {  // the partly used quarter: kQRem floats per lane, densely packed
          const int voff = kQFull * kWStep + lane * (4 * kQRem);
          // The wider loads are cast to float vectors as a whole: with per-element casts
          // of an integer vector this compiler shrinks the load to its first element.
          if constexpr (kQRem == 1) {
            dst.x = __builtin_bit_cast(float, buf_load1(rs_w, voff, soff));
          } else if constexpr (kQRem == 2) {
            const float2v t = __builtin_bit_cast(
                float2v, __builtin_amdgcn_raw_buffer_load_b64(rs_w, voff, soff, 0));
            dst.x = t.x;
            dst.y = t.y;
          } else {
            const float3v t = __builtin_bit_cast(
                float3v, __builtin_amdgcn_raw_buffer_load_b96(rs_w, voff, soff, 0));
            dst.x = t.x;
            dst.y = t.y;
            dst.z = t.z;
          }
          return;
        }
      }
      dst = __builtin_bit_cast(Frag, buf_load4(rs_w, w_voff + q * kWStep, soff));
    };
    auto fetch_w = [&](int soff, int slot, int q) { fetch_frag(w[slot][q], soff, q); };
    auto fetch_orow = [&](const StagePos &pos, int m, int slot) {
      orow[slot] = buf_load1(rs_out, l16 * 4 + m * 64, pos.g * 256);
    };
    // An accumulator update whose write is still to come: row address, the row as it
    // was read, and the product to add.
    struct Pending {
      int addr;
      float4v accr, d;
    };
    // LDS address of this lane's 4 columns in accumulator row 0
    const int acc_lane = acc_base + (wave * 16 + g * 4) * 4;
    const int dummy_addr = T * kAS * 4 + acc_lane;
    if constexpr (TAIL) {
      // One column group for four consumer waves: wave m multiplies row block m of every
      // group and keeps its products in the 16 accumulator columns it owns (a partial sum
      // of the group's columns over the pairs of its blocks; flush_tile adds the four up).
      // A stage is 1 row block of NS MFMAs per wave instead of 4; the products of a group's
      // chunks stay in registers and reach the accumulators once per group.
      // Rings indexed by stage number (the loop is unrolled over four stages):
      //   w[s & 3]     fragments of stage s, fetched three stages ahead
      //   kof[s & 3]   fragment offset of the block's kernel offset, loaded seven stages
      //                ahead (four before the fetch that needs it)
      //   orow[s & 3]  accumulator row of this lane's pair, tl[s & 3] the tile of the stage:
      //                loaded four stages ahead, into the slot the stage before just used
      int kof[4];
      int4v tl[4];
      auto load_kof = [&](const StagePos &pos) -> int {
        return buf_load1(rs_meta, wave * 4, pos.g * 32);
      };
      StagePos p_cur = {g_begin, 0};  // stage being multiplied
      StagePos p_f = {g_begin, 0};    // stage whose fragments are fetched next
      StagePos p_k = {g_begin, 0};    // stage whose fragment offset is loaded next
      StagePos p_m = {g_begin, 0};    // stage whose accumulator rows and tile are loaded next
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        kof[j] = load_kof(p_k);
        p_k.advance(nch);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        fetch_orow(p_m, wave, j);
        tl[j] = load_rec_tail(p_m);
        p_m.advance(nch);
      }
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const int soff = frag_soff(kof[j], w_soff0 + p_f.cc * kFragB);
#pragma unroll
        for (int q = 0; q < NF; ++q) fetch_w(soff, j, q);
        p_f.advance(nch);
        kof[j] = load_kof(p_k);
        p_k.advance(nch);
      }
      float4v d = float4v{0.f, 0.f, 0.f, 0.f};
      __syncthreads();
      auto stage = [&](auto phase) {
        constexpr int ph = decltype(phase)::value;  // == stage number & 3
        constexpr int nx = (ph + 3) & 3;
        {
          const int soff = frag_soff(kof[nx], w_soff0 + p_f.cc * kFragB);
#pragma unroll
          for (int q = 0; q < NF; ++q) fetch_w(soff, nx, q);
          p_f.advance(nch);
          kof[nx] = load_kof(p_k);
          p_k.advance(nch);
        }
        Frag a[NF];
#pragma unroll
        for (int q = 0; q < NF; ++q)
          a[q] = *reinterpret_cast<const Frag *>(a_base[q] + (wave * 16 + (ph & 1) * kStage) * kRowB);
        const bool commit = p_cur.cc == nch - 1;  // the group's last chunk
        const int addr = commit ? orow[ph] + acc_lane : dummy_addr;
        const float4v accr = lds_load4(addr);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NS; ++i)
          d = __builtin_amdgcn_mfma_f32_16x16x4f32(w[ph][i >> 2][i & 3], a[i >> 2][i & 3], d, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        const TileEnd e = tile_end_of(tl[ph], p_cur);
        if (commit) {
          lds_store4(addr, accr + d);
          d = float4v{0.f, 0.f, 0.f, 0.f};
        }
        fetch_orow(p_m, wave, ph);
        tl[ph] = load_rec_tail(p_m);
        p_m.advance(nch);
        p_cur.advance(nch);
        __syncthreads();
        if (e.last) {
          flush_tile(e.row0, e.rows, e.slot0);
          __syncthreads();
        }
      };
      // whole groups of four stages first, the remainder after the loop (see the producers)
      int s = 0;
      for (; s + 4 <= nstages; s += 4) {
        stage(std::integral_constant<int, 0>());
        stage(std::integral_constant<int, 1>());
        stage(std::integral_constant<int, 2>());
        stage(std::integral_constant<int, 3>());
      }
      if (s < nstages) stage(std::integral_constant<int, 0>());
      if (s + 1 < nstages) stage(std::integral_constant<int, 1>());
      if (s + 2 < nstages) stage(std::integral_constant<int, 2>());
    } else {
    // The five-group form.  Besides its own column group, of
    // which it multiplies the four row blocks of a stage, wave w multiplies row block w with
    // the fragments of a fifth group (output columns xcol .., accumulator columns kCN ..):
    // five blocks of MFMAs per stage and wave instead of four, and no SIMD that multiplies
    // for a column block of one group.  The products of a row block stay in registers over
    // the chunks of its group (dx).  Two row blocks of a group may hold the same output row,
    // so the four waves must not add to the fifth group's accumulators between the same two
    // barriers: wave w adds its products of a finished group (dprev, at aprev) during chunk
    // w of the next group (nch >= 4, the host launches the form for such layers only), in
    // the order of the row blocks, as the other column groups see their offsets; when a
    // tile ends they are added at once, a barrier between each two waves.
    //   wx[s & 1]  fragments of the fifth group for stage s, fetched one stage ahead
    //   kofx       fragment offset of row block `wave` of the next stage
    //   orowx      accumulator row of this lane's pair in row block `wave` of this stage
    Frag wx[2][NF];
    int kofx = 0, orowx = 0;
    float4v dx = float4v{0.f, 0.f, 0.f, 0.f}, dprev = float4v{0.f, 0.f, 0.f, 0.f};
    const int acc_lane_x = acc_base + (kCN + g * 4) * 4;
    const int dummy_x = T * kAS * 4 + acc_lane_x;
    int aprev = dummy_x;
    bool x_pending = false;
    constexpr bool x_on = FIVE;  // (a launch of the form has a fifth group: xcol >= 0)
    const int w_soffx = (x_on ? xcol / 16 : 0) * nch * kFragB;
    auto load_kofx = [&](const StagePos &pos) -> int {
      return buf_load1(rs_meta, wave * 4, pos.g * 32);
    };
    auto load_orowx = [&](const StagePos &pos) -> int {
      return buf_load1(rs_out, l16 * 4 + wave * 64, pos.g * 256);
    };
    Pending pend;  // nothing pending yet: the first write adds zero to the dummy row
    pend.addr = dummy_addr;
    pend.accr = float4v{0.f, 0.f, 0.f, 0.f};
    pend.d = float4v{0.f, 0.f, 0.f, 0.f};
    // One stage = 4 row blocks of 16 MFMAs each, software-pipelined by hand.  A wave
    // issues at most one instruction every few cycles, and a dependent MFMA can only
    // issue when its predecessor is through the pipeline, so between two MFMAs of a
    // chain a handful of other instructions issue for free -- and no more than that:
    // everything else a block needs is therefore spread, one small piece per gap,
    // over the 16 gaps of the block, and scheduling barriers pin it there:
    // (gap numbers for NS = 16, i.e. 16 MFMAs a block)
    //   gap 2      fragment offset of block b+3 (from the schedule record); accumulator
    //              update of the previous block: add, write; once per stage, tile and
    //              last-of-tile of the next stage
    //   gap 3      accumulator read of this block (LDS operations of a wave execute
    //              in order, so it sees the write of gap 2 when both blocks touch
    //              the same output row)
    //   gaps 4,7,9,12  the four fragment loads of block b+3 (the slot of block b-1)
    //   gap 5      output rows of block b+3
    //   gaps 6,8,10,11  the staged rows of block m+1
    //   gaps 13,14 once per stage: the record of the stage after the next
    // The update of a stage's last block waits, across the barrier, for the first
    // block of the next stage, unless the tile ends here.
    //   cur / next / after: positions of this stage and the two that follow;
    //   returns the tile rows and last-of-tile of the NEXT stage.
    auto run_stage = [&](auto parity, bool last_cur, const StagePos &cur, const StagePos &next,
                         const StagePos &after, TileEnd &end_next) {
      constexpr int par = decltype(parity)::value;
      const int base_cur = w_soff0 + cur.cc * kFragB;
      const int base_next = w_soff0 + next.cc * kFragB;
      // Staged rows in registers: of this block and the next.  Half: of all four blocks, read
      // as the stage begins -- two MFMAs are shorter than an LDS read takes, so a block's rows
      // read during the block before would be waited for in every block instead of once
      // (64 -> 128 channels, 1.54 M pairs: 166 -> 160 us).
      constexpr int kARing = kHalf ? 4 : 2;
      Frag a[kARing][NF];
      auto load_a = [&](int m, int q, Frag (&av)[NF]) {
        av[q] = *reinterpret_cast<const Frag *>(a_base[q] + (par * kStage + m * 16) * kRowB);
      };
#pragma unroll
      for (int m = 0; m < (kHalf ? 4 : 1); ++m)
#pragma unroll
        for (int q = 0; q < NF; ++q) load_a(m, q, a[m]);
      // gaps of the pieces of a block (see above); with fewer than 16 MFMAs they move
      // closer together, in the same order
      // half: two MFMAs a block, so the pieces sit behind the first or the second
      constexpr int kSteps = kHalf ? 2 : NS;
      constexpr bool kFull = !kHalf && NS == 16;
      // no piece may be placed behind the last MFMA
      constexpr int kLast = kSteps - 1;
      auto at = [](int gap) constexpr { return gap < (kHalf ? 1 : NS - 1) ? gap : (kHalf ? 1 : NS - 1); };
      constexpr int kGapAlu = kHalf ? 0 : kFull ? 2 : at(1), kGapAcc = kHalf ? 0 : at(kGapAlu + 1);
      constexpr int kGapW[4] = {kHalf ? 0 : kFull ? 4 : at(2), kHalf ? 1 : kFull ? 7 : at(3),
                                kFull ? 9 : at(4), at(12)};
      constexpr int kGapRow = kHalf ? 0 : kFull ? 5 : at(2);  // after fragment load 0 in the same gap
      constexpr int kGapA[4] = {kHalf ? 1 : kFull ? 6 : at(kSteps / 2),
                                kHalf ? 1 : kFull ? 8 : at(kSteps / 2 + 1),
                                kFull ? 10 : at(kSteps / 2 + 2), at(11)};
      constexpr int kGapRec0 = kHalf ? 1 : kFull ? 13 : (kSteps >= 2 ? kSteps - 2 : 0);
      constexpr int kGapRec1 = kHalf ? 1 : kFull ? 14 : kLast;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int slot = m;                 // == (4 * s + m) & 3
        const int tslot = (m + 3) & 3;      // slot of block b+3 == slot of block b-1
        const int tm = (m + 3) & 3;         // index of block b+3 inside its stage
        const bool tnext = m > 0;           // block b+3 belongs to the next stage
        float4v d = float4v{0.f, 0.f, 0.f, 0.f};
        int soff = 0;
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (kHalf) {
            d = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8v, w[slot][i]),
                                                       __builtin_bit_cast(half8v, a[m][i]), d,
                                                       0, 0, 0);
          } else {
            const int q = i >> 2, j = i & 3;
            d = __builtin_amdgcn_mfma_f32_16x16x4f32(w[slot][q][j], a[m & 1][q][j], d, 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
          // all vector-ALU work of the block in one gap: a vector-ALU instruction
          // next to the matrix chain costs about ten cycles for leaving and re-entering
          // the chain, whatever follows it in the same gap is cheap
          if (i == kGapAlu) {
            soff = tnext ? frag_soff(rec_k(rec[par ^ 1][0], tm), base_next)
                         : frag_soff(rec_k(rec[par][0], tm), base_cur);
            if (m == 3) end_next = tile_end_of(rec[par ^ 1][1], next);
            // pend.d = out[pair l16][channels 4g .. 4g+3] of the previous block
            lds_store4(pend.addr, pend.accr + pend.d);
            pend.addr = orow[slot] + acc_lane;
          }
          if (i == kGapAcc) pend.accr = lds_load4(pend.addr);
          if (i == kGapW[0]) fetch_w(soff, tslot, 0);
          if (i == kGapRow) fetch_orow(tnext ? next : cur, tm, tslot);
#pragma unroll
          for (int qq = 1; qq < NF; ++qq)
            if (i == kGapW[qq]) fetch_w(soff, tslot, qq);
          if constexpr (kHalf) {
            // (read already)
          } else if (m < 3) {
#pragma unroll
            for (int qq = 0; qq < NF; ++qq)
              if (i == kGapA[qq]) load_a(m + 1, qq, a[(m + 1) & 1]);
          } else if constexpr (FIVE) {  // row block `wave`, for the fifth group
#pragma unroll
            for (int qq = 0; qq < NF; ++qq)
              if (i == kGapA[qq])
                a[0][qq] = *reinterpret_cast<const Frag *>(a_base[qq] +
                                                           (par * kStage + wave * 16) * kRowB);
          }
          // this stage's record was last used by block 0: refill it for the stage
          // after the next
          if (m == 1 && i == kGapRec0)
            rec[par][0] = __builtin_bit_cast(int4v, buf_load4(rs_meta, 0, after.g * 32));
          if (m == 1 && i == kGapRec1) rec[par][1] = load_rec_tail(after);
        }
        __builtin_amdgcn_sched_barrier(0);
        pend.d = d;
      }
      if constexpr (FIVE) {
        if (x_on) {
          // gaps: 0 read of the accumulator row this wave adds to in this stage (the dummy
          // row in other stages); 3 that update, fragment offset of the next stage;
          // 4, 6, 8, 10 its fragments; 11, 12 the next offset and accumulator row
          const bool mine = x_pending && cur.cc == wave;
          const int caddr = mine ? aprev : dummy_x;
          float4v accx = float4v{0.f, 0.f, 0.f, 0.f};
          int soffx = 0;
          constexpr int kGapXW[4] = {at(4), at(6), at(8), at(10)};
#pragma unroll
          for (int i = 0; i < kSteps; ++i) {
            __builtin_amdgcn_sched_barrier(0);
            dx = __builtin_amdgcn_mfma_f32_16x16x4f32(wx[par][i >> 2][i & 3], a[0][i >> 2][i & 3],
                                                      dx, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (i == at(0)) accx = lds_load4(caddr);
            if (i == at(3)) {
              soffx = frag_soff(kofx, w_soffx + next.cc * kFragB);
              lds_store4(caddr, accx + dprev);
            }
#pragma unroll
            for (int qq = 0; qq < NF; ++qq)
              if (i == kGapXW[qq]) fetch_frag(wx[par ^ 1][qq], soffx, qq);
            if (i == at(11)) kofx = load_kofx(after);
          }
          __builtin_amdgcn_sched_barrier(0);
          if (cur.cc == nch - 1) {  // the group is complete
            dprev = dx;
            aprev = orowx + acc_lane_x;
            dx = float4v{0.f, 0.f, 0.f, 0.f};
            x_pending = true;
          }
          orowx = load_orowx(next);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (last_cur) {  // the tile is written out after this stage: finish its last update
        lds_store4(pend.addr, pend.accr + pend.d);
        pend.addr = dummy_addr;
      }
    };
    StagePos p_cur = {g_begin, 0};    // stage being multiplied
    StagePos p_next = {g_begin, 0};   // the stage after it
    StagePos p_after = {g_begin, 0};  // and the one after that
    p_next.advance(nch);
    p_after.advance(nch);
    p_after.advance(nch);
    TileEnd end, end_next;
    {
      // what the first stage needs before it starts: its record and the next one,
      // fragments and rows of its blocks 0..2
      load_rec(p_cur, rec[0]);
      load_rec(p_next, rec[1]);
      end = tile_end_of(rec[0][1], p_cur);
      // Loads are issued in the order of the loop (fragment 0, the output rows, the other
      // fragments, block after block) and pinned there: the wait counts of the
      // loop are static and must hold on its first trip as well, so a load that the
      // prologue issued late would make every trip wait for nearly all loads in flight.
#pragma unroll
      for (int b = 0; b < 3; ++b) {
        const int soff = frag_soff(rec_k(rec[0][0], b), w_soff0 + p_cur.cc * kFragB);
        __builtin_amdgcn_sched_barrier(0);
        fetch_w(soff, b, 0);
        __builtin_amdgcn_sched_barrier(0);
        fetch_orow(p_cur, b, b);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 1; q < NF; ++q) {
          fetch_w(soff, b, q);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if constexpr (FIVE) {
        if (x_on) {  // in the loop's order: fragments, next offset, accumulator row
          kofx = load_kofx(p_cur);
          const int soffx = frag_soff(kofx, w_soffx + p_cur.cc * kFragB);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int q = 0; q < NF; ++q) fetch_frag(wx[0][q], soffx, q);
          __builtin_amdgcn_sched_barrier(0);
          kofx = load_kofx(p_next);
          orowx = load_orowx(p_cur);
        }
      }
    }
    __syncthreads();
    auto step = [&](auto parity) {
      run_stage(parity, end.last, p_cur, p_next, p_after, end_next);
      p_cur.advance(nch);
      p_next.advance(nch);
      p_after.advance(nch);
      __syncthreads();
      if (end.last) {
        if constexpr (FIVE) {
          // the last group's products of the fifth group, wave after wave
#pragma unroll
          for (int wv = 0; wv < 4; ++wv) {
            if (x_on && wave == wv) lds_store4(aprev, lds_load4(aprev) + dprev);
            __syncthreads();
          }
          x_pending = false;
        }
        flush_tile(end.row0, end.rows, end.slot0);
        __syncthreads();
      }
      end = end_next;
    };
    // pairs of stages first, an odd last stage after the loop (see the producer's loop)
    int s = 0;
    for (; s + 2 <= nstages; s += 2) {
      step(std::integral_constant<int, 0>());
      step(std::integral_constant<int, 1>());
    }
    if (s < nstages) step(std::integral_constant<int, 0>());
    }
  }
}

struct ConvPlan {
  int ncb, nch, T, ncw, n_wg, n_colblk;  // T: rows of the accumulator window
  int n_rng;  // ranges of output rows: one for every workgroup of a column block, or two
  int tile_rows;                         // largest tile height
  int gather;  // conv_fwd_kernel's GATHER
  int ns;      // conv_fwd_kernel's NS: MFMA steps per chunk
  int64_t n_tiles, n_fine, words_per_k, grp_cap;  // n_tiles: upper bound
  int granule;  // rows per cell of the grid the work split places its boundaries on
  size_t lds_bytes;
  // Launches.  As a rule one, over all column blocks (n_colblk of them side by side, the
  // CUs shared out among them).  A last column group that would be alone in its block of
  // four (Cout = 72: 5 groups) behind at most two full blocks gets no column block, where
  // three of four consumer waves would multiply for nothing: the full blocks take one launch
  // each over all CUs (n_launch of them, n_colblk = 1) and the kernel's one-column-group
  // form a last one (has_tail), all over the same plan.
  // Or, for layers of four or more channel chunks, the last full block's launch takes the
  // lone group along as a fifth one (five): every launch is then of the five-group form,
  // whose accumulator rows are 16 columns wider (acc_cols), xcol >= 0 in the last only.
  int n_launch;
  bool has_tail, five;
  bool rebalance;  // the work split is made twice, the second time from the first one's counts
  int acc_cols;  // accumulator columns of a workgroup: 64, or 80 in the five-group form
  // a layer of a handful of input channels: no schedule, no matrix kernel -- the plan is a
  // table of every output row's input rows and the rows are computed by conv_small_kernel
  bool small;
  // the bfloat16-parts form
  bool parts;
  bool parts_packed;  // the packed filters have the parts behind the floats
  int blk;  // pairs of an offset to a block: 16, in the parts form 32 or 64
  int kvol;           // kernel volume and number of output rows the plan was made for
  int64_t out_rows;
};

// conv_small.hip
bool conv_small_applies(int K, int c_in, int c_out, int elem_bytes);
int conv_small_build_table(const int32_t *flag, bool in_order, const int32_t *pairs,
                           const int32_t *sorted, int64_t pair_stride, int plane_s,
                           const int32_t *pair_num, int K, int64_t n_out, int32_t *table,
                           hipStream_t s);
int conv_small_run(const float *features, int c_in, const void *packed, int ncb, int ns,
                   const int32_t *table, int K, float *out, int c_out, int64_t n_out,
                   const ConvEpilogue &epi, hipStream_t s);

// Device buffers of a convolution call, in three groups with different lifetimes:
//   packed   the filters in MFMA fragment order: as long as the filters keep their values;
//   plan     what the convolution kernel reads besides features and filters (the row-block
//            schedule and the tile ranges of the workgroups): as long as the rulebook, the
//            channel counts, the element type and the direction (`inverse`) stay the same;
//   scratch  intermediate tables of the kernels that build the plan: until it is built.
struct ConvWs {
  void *packed;
  // plan
  int32_t *wg_tile, *wg_grp;  // first tile of every range; first and end group of every workgroup
  int32_t *sched_in, *sched_out, *grp_meta;
  int32_t *small_table;  // [K, n_out] (plans of ConvPlan::small, which have nothing else)
  // scratch
  int32_t *flag;
  int32_t *segs;
  int32_t *sorted;
  uint32_t *bits;
  int32_t *prefix;
  int32_t *tile_loc, *tile_nmb, *kofs, *tile_rng, *range_grp, *range_row1, *range_g0;
  int32_t *fine_segs, *range_row0, *range_row0_alt, *tile_row0, *n_tiles_dev;
  int32_t *spill_end, *tile_slot0, *spill, *share_first, *share_cnt;
};

// (switched by ssc_conv_tuning, for measurements)
inline bool g_conv_by_column = true;  // one column block per XCD for large filters

template <typename IO, int GATHER, int NCW, int NS, bool EPI, int FORM>
inline int launch_conv(const ConvPlan &p, const ConvWs &w, const IO *features, int64_t n_in,
                       int c_in, int K, IO *out, int c_out, int col_base, int xcol,
                       const ConvEpilogue &epi, hipStream_t s) {
  static bool attr_set = false;
  if (!attr_set) {
    SSC_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(conv_fwd_kernel<IO, GATHER, NCW, NS, EPI, FORM>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    attr_set = true;
  }
  const uint64_t packed_bytes = (uint64_t)K * p.ncb * p.nch *
                                (FORM >= 4 ? Io<IO>::kFragBytes + kPartFragBytes : Io<IO>::kFragBytes);
  const uint64_t sched_bytes = (uint64_t)p.grp_cap * 256;
  SSC_CHECK(packed_bytes < ((uint64_t)1 << 32) && sched_bytes < ((uint64_t)1 << 32), SSC_ERUNTIME,
            "convolution too large for 32-bit buffer offsets (filters %llu B, schedule %llu B)",
            (unsigned long long)packed_bytes, (unsigned long long)sched_bytes);
  const unsigned feat_bytes = GATHER != 0 ? (unsigned)((uint64_t)n_in * c_in * sizeof(IO)) : 0u;
  SSC_CHECK(p.n_wg >= 1 && p.n_colblk >= 1 && col_base % 16 == 0 &&
                col_base + (p.n_colblk - 1) * 16 * NCW < c_out,
            SSC_ERUNTIME, "convolution launch outside the output columns");
  SSC_CHECK(FORM == 2 ? (xcol >= 0 && xcol % 16 == 0 && xcol < c_out && p.nch >= 4 &&
                         p.n_colblk == 1 && p.five)
                      : (xcol < 0 && p.five == (FORM == 3)),
            SSC_ERUNTIME, "convolution launch with a fifth column group it is not built for");
  dim3 grid((unsigned)p.n_wg, (unsigned)p.n_colblk);
  // one column block per XCD when the packed filters are larger than an L2 can keep
  // (4 MiB per XCD) and the grid divides that way (256 -> 256 channels, 7 MiB: 2.44 ->
  // 2.24 ms on the 64^3 benchmark geometry; 128 -> 256 at stride 2, 3.5 MiB, is 5 % slower
  // that way and stays with the row-major mapping)
  const uint64_t walked_bytes = (uint64_t)K * p.ncb * p.nch *
                                (FORM >= 4 ? kPartFragBytes : Io<IO>::kFragBytes);
  const bool by_column = walked_bytes > ((uint64_t)4 << 20) && p.n_colblk > 1 &&
                         8 % p.n_colblk == 0 && (p.n_wg * p.n_colblk) % 8 == 0 &&
                         g_conv_by_column;
  // (-1: a grid that is no multiple of 8 wide takes the kernel's mapping for any grid)
  const bool big = walked_bytes > ((uint64_t)4 << 20) && p.n_colblk > 1 && g_conv_by_column;
  const int cols_per_xcd = by_column ? 8 / p.n_colblk
                           : ((p.n_wg & 7) != 0 && p.n_wg * p.n_colblk >= 16) ? (big ? -2 : -1) : 0;
  hipLaunchKernelGGL((conv_fwd_kernel<IO, GATHER, NCW, NS, EPI, FORM>), grid, dim3((NCW + 4) * 64), p.lds_bytes, s, features, c_in,
                     feat_bytes, w.packed, (unsigned)packed_bytes, w.sched_in, w.sched_out,
                     w.grp_meta, (unsigned)sched_bytes, (unsigned)(p.grp_cap * 32), w.wg_grp,
                     p.nch, p.ncb, out, c_out, p.T, cols_per_xcd, col_base, xcol, epi);
  SSC_LAUNCH_CHECK("conv_fwd");
  return SSC_OK;
}

// The instances on float rows that conv.hip does not compile itself (conv_instances.h):
// with the epilogue, and the one-column-group and five-group forms with and without it.
template <int GATHER, int NS, bool EPI, int FORM>
int launch_conv_f32(const ConvPlan &p, const ConvWs &w, const float *features, int64_t n_in,
                    int c_in, int K, float *out, int c_out, int col_base, int xcol,
                    const ConvEpilogue &epi, hipStream_t s);

}  // namespace ssc
