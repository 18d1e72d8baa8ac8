// Steerable kernel synthesis: dense kernel = sum_beta weight * basis, written
// straight into the contiguous [K, Cin, Cout] layout the convolution consumes.
// One thread per output element; the per-channel descriptor tables replace the
// reference's loop over irrep pairs, its einsum, both concatenations and the
// permute.  The sum over beta runs in ascending order.
#include "combine_element.h"
#include "ssc_common.h"

#include <algorithm>

namespace ssc {

__global__ void __launch_bounds__(256)
    combine_kernel(const float *__restrict__ weight, const float *__restrict__ basis,
                   const int32_t *__restrict__ chan_out, const int32_t *__restrict__ chan_in,
                   const int32_t *__restrict__ blocks, int n_j, int K, int cin, int cout,
                   float *__restrict__ out) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t total = (int64_t)K * cin * cout;
  if (idx >= total) return;
  int co = (int)(idx % cout);
  int64_t r = idx / cout;
  int ci = (int)(r % cin);
  int k = (int)(r / cin);
  const float acc = combine_element(weight, basis, chan_out, chan_in, blocks, n_j, K, k, ci, co);
  out[idx] = acc;
}

// Gradient with respect to the weights: d_weight[u][v][n] of block (i, j) is the sum over the
// offsets k and the components a, b of d_dense[k][(j,v,b)][(i,u,a)] * basis_ij[n][a][b][k].
// A workgroup per pair of an output field (i, u) and an input field (j, v): its threads run
// along the basis elements as they lie in memory (k fastest), eight basis functions at a time
// (further eights beside them, grid z), and the threads' sums are added in a fixed order.
// Bound by the latency of its few loads (442 KB of d_dense for 64 -> 64 channels and kernel
// 3): 11 us there, where matrix products block by block took 49 launches, 200 us and as much
// again of host time.  Kernel 5, orders 0 to 4, eight fields each: 156 -> 97 us by the loads
// without branches and the eights beside each other; 16 fields of order 2, kernel 7: 168 -> 46.
constexpr int kBwdBeta = 8;
__global__ void __launch_bounds__(256)
    combine_bwd_kernel(const float *__restrict__ d_dense, const float *__restrict__ basis,
                       const int32_t *__restrict__ chan_out, const int32_t *__restrict__ chan_in,
                       const int32_t *__restrict__ blocks, const int32_t *__restrict__ first_out,
                       const int32_t *__restrict__ first_in, int n_j, int K, int cin, int cout,
                       float *__restrict__ d_weight) {
  __shared__ float part[4][kBwdBeta];
  const int co0 = first_out[blockIdx.x], ci0 = first_in[blockIdx.y];
  const int i = chan_out[co0 * 3], u = chan_out[co0 * 3 + 1];
  const int j = chan_in[ci0 * 3], v = chan_in[ci0 * 3 + 1];
  const int32_t *blk = blocks + (i * n_j + j) * 6;
  const int w_off = blk[0], b_off = blk[1], n_beta = blk[2], m_in = blk[3], d_out = blk[4],
            d_in = blk[5];
  const int elems = d_out * d_in * K;
  const float *bs = basis + b_off;
  const float *g = d_dense + (int64_t)ci0 * cout + co0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int n0 = blockIdx.z * kBwdBeta; n0 < n_beta; n0 += gridDim.z * kBwdBeta) {
    const int n = min(kBwdBeta, n_beta - n0);
    float acc[kBwdBeta];
    // (functions beyond the last: the last one, not stored -- a load behind a branch of its
    // own would be waited for before the next)
    const float *fn[kBwdBeta];
#pragma unroll
    for (int t = 0; t < kBwdBeta; ++t) {
      acc[t] = 0.f;
      fn[t] = bs + (int64_t)min(n0 + t, n_beta - 1) * elems;
    }
    for (int e = threadIdx.x; e < elems; e += 256) {
      const int ab = e / K, k = e - ab * K;
      const int a = ab / d_in, b = ab - a * d_in;
      const float x = g[((int64_t)k * cin + b) * cout + a];
#pragma unroll
      for (int t = 0; t < kBwdBeta; ++t) acc[t] += x * fn[t][e];
    }
#pragma unroll
    for (int t = 0; t < kBwdBeta; ++t) {
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) acc[t] += __shfl_xor(acc[t], d, 64);
      if (lane == 0) part[wave][t] = acc[t];
    }
    __syncthreads();
    if (threadIdx.x < n) {
      const int t = threadIdx.x;
      d_weight[w_off + (u * m_in + v) * n_beta + n0 + t] =
          (part[0][t] + part[1][t]) + (part[2][t] + part[3][t]);
    }
    __syncthreads();
  }
}

// The same for layers of many fields.  There the kernel above pays a workgroup for every pair
// (2.1 ns of dispatch each), fetches a line of d_dense for one value and the basis anew for
// every pair.  Here a wave takes 16 output fields by 4 input fields, a pair to a lane:
// neighbouring fields are neighbours in memory, and the basis is the same for all lanes of a
// block (i, j), so that it comes through the scalar cache.  Bound by the latency of a tile's
// chain of loads, and by dispatch where tiles are many: 512 -> 512 scalars, kernel 3: 60 us
// (a workgroup to a pair 559, one matrix product 68); orders 0 to 2, 32 fields each, kernel
// 7: 198 (874, 393).  With SHARED the sixteen waves of
// a workgroup share out the offsets k of one tile and their sums are added in a fixed order;
// without (few offsets) each has a tile of its own.  Tiles of more than one block are taken
// block by block.
constexpr int kWideWaves = 16, kWideOut = 16, kWideIn = 4;
template <bool SHARED>
__global__ void __launch_bounds__(kWideWaves * 64)
    combine_bwd_wide_kernel(const float *__restrict__ d_dense, const float *__restrict__ basis,
                            const int32_t *__restrict__ chan_out,
                            const int32_t *__restrict__ chan_in,
                            const int32_t *__restrict__ blocks,
                            const int32_t *__restrict__ first_out, int n_out,
                            const int32_t *__restrict__ first_in, int n_in, int n_j, int K,
                            int cin, int cout, float *__restrict__ d_weight) {
  __shared__ float part[SHARED ? kWideWaves : 1][kBwdBeta][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int per = SHARED ? (K + kWideWaves - 1) / kWideWaves : K;
  const int k_lo = SHARED ? min(K, wave * per) : 0, k_hi = min(K, k_lo + per);
  const int tiles = SHARED ? 1 : kWideWaves;  // of the workgroup, along the input fields
  const int64_t plane = (int64_t)cin * cout;
  for (int in0 = blockIdx.y * tiles * kWideIn; in0 < n_in; in0 += gridDim.y * tiles * kWideIn) {
    const int fo = blockIdx.x * kWideOut + lane % kWideOut;
    const int fi = in0 + (SHARED ? 0 : wave * kWideIn) + lane / kWideOut;
    const bool live = fo < n_out && fi < n_in;
    int co0 = 0, ci0 = 0, of = -1, u = 0, v = 0;
    if (live) {
      co0 = first_out[fo];
      ci0 = first_in[fi];
      of = chan_out[co0 * 3] * n_j + chan_in[ci0 * 3];  // the pair's block
      u = chan_out[co0 * 3 + 1];
      v = chan_in[ci0 * 3 + 1];
    }
    const float *g = d_dense + (int64_t)ci0 * cout + co0;
    // (SHARED: the lanes of all waves hold the same pairs, every wave makes the same rounds)
    for (unsigned long long left = __ballot(live); left != 0;) {
      const int now = __builtin_amdgcn_readlane(of, __ffsll(left) - 1);
      const bool mine = of == now;
      left &= ~__ballot(mine);
      const int32_t *blk = blocks + now * 6;
      const int w_off = blk[0], b_off = blk[1], n_beta = blk[2], m_in = blk[3], d_out = blk[4],
                d_in = blk[5];
      const int elems = d_out * d_in * K;
      float *dst = d_weight + w_off + (u * m_in + v) * n_beta;
      for (int n0 = blockIdx.z * kBwdBeta; n0 < n_beta; n0 += gridDim.z * kBwdBeta) {
        float acc[kBwdBeta];
        const float *bs[kBwdBeta];  // (functions beyond the last: the last one, not stored)
#pragma unroll
        for (int t = 0; t < kBwdBeta; ++t) {
          acc[t] = 0.f;
          bs[t] = basis + b_off + (int64_t)min(n0 + t, n_beta - 1) * elems;
        }
        if (mine) {
          for (int k = k_lo; k < k_hi; ++k) {
            float of_k[kBwdBeta];  // summed offset by offset: shorter chains of roundings
#pragma unroll
            for (int t = 0; t < kBwdBeta; ++t) of_k[t] = 0.f;
            for (int b = 0; b < d_in; ++b) {
              const float *row = g + k * plane + b * cout;
#pragma unroll 4
              for (int a = 0; a < d_out; ++a) {
                const float x = row[a];
                const int e = (a * d_in + b) * K + k;
#pragma unroll
                for (int t = 0; t < kBwdBeta; ++t) of_k[t] += x * bs[t][e];
              }
            }
#pragma unroll
            for (int t = 0; t < kBwdBeta; ++t) acc[t] += of_k[t];
          }
        }
        if constexpr (SHARED) {
#pragma unroll
          for (int t = 0; t < kBwdBeta; ++t) part[wave][t][lane] = acc[t];
          __syncthreads();
          if (wave < kBwdBeta && mine && n0 + wave < n_beta) {
            float sum[4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
              sum[q] = (part[q * 4][wave][lane] + part[q * 4 + 1][wave][lane]) +
                       (part[q * 4 + 2][wave][lane] + part[q * 4 + 3][wave][lane]);
            dst[n0 + wave] = (sum[0] + sum[1]) + (sum[2] + sum[3]);
          }
          __syncthreads();
        } else {
#pragma unroll
          for (int t = 0; t < kBwdBeta; ++t)
            if (mine && n0 + t < n_beta) dst[n0 + t] = acc[t];
        }
      }
    }
  }
}

}  // namespace ssc

extern "C" int ssc_kernel_combine_bwd_f32(const float *d_dense, const float *basis,
                                          const int32_t *chan_out, const int32_t *chan_in,
                                          const int32_t *blocks, const int32_t *first_out,
                                          int32_t n_fields_out, const int32_t *first_in,
                                          int32_t n_fields_in, int32_t n_irreps_in,
                                          int32_t kernel_volume, int32_t c_in, int32_t c_out,
                                          float *d_weight, ssc_stream_t stream) {
  SSC_CHECK(d_dense && basis && chan_out && chan_in && blocks && first_out && first_in && d_weight,
            SSC_EINVAL, "NULL pointer argument");
  SSC_CHECK(n_irreps_in >= 1 && kernel_volume >= 1 && c_in >= 1 && c_out >= 1, SSC_EINVAL,
            "sizes must be positive");
  SSC_CHECK(n_fields_out >= 1 && n_fields_out <= c_out && n_fields_in >= 1 && n_fields_in <= c_in,
            SSC_EINVAL, "field counts out of range");
  // chunks of eight basis functions, as many as the default radial window makes of a block
  // (5, 11, 19 and 28 functions for kernels of size 3, 5, 7 and 9); the kernels walk the rest
  const unsigned chunks =
      kernel_volume <= 27 ? 1 : kernel_volume <= 125 ? 2 : kernel_volume <= 343 ? 3 : 4;
  const int64_t n_pairs = (int64_t)n_fields_out * n_fields_in;
  const int64_t elems = (int64_t)kernel_volume * c_in * c_out / n_pairs;  // of a function, on average
  auto launch = [&](auto kernel, dim3 grid, int threads, auto... fields) {
    hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, (hipStream_t)stream, d_dense, basis,
                       chan_out, chan_in, blocks, fields..., n_irreps_in, kernel_volume, c_in,
                       c_out, d_weight);
  };
  // A workgroup to a pair while the pairs are few: with kernel 3 and orders 0 to 3, 4096 pairs
  // take 19 us that way and 30 the other, 9216 pairs 35 and 49, 12544 pairs 47 and 51, 16384
  // pairs 61 and 31.  With long basis functions the pair form is bound by reading them for
  // every pair: kernel 5, orders 0 to 3, 6400 pairs 244 and 206, 9216 pairs 327 and 202, 16384
  // pairs 699 and 143; tiles that cut fields of many blocks would be slower below that.
  if (n_pairs > (elems >= 1024 ? 4096 : 14336)) {
    // (grid rows beyond 65535 are walked by the kernel; up to 8 offsets sixteen waves would
    // have none to share)
    const bool shared = kernel_volume > 8;
    const int fields = ssc::kWideIn * (shared ? 1 : ssc::kWideWaves);
    const dim3 grid((unsigned)ssc::ceil_div(n_fields_out, ssc::kWideOut),
                    (unsigned)std::min(65535, (int)ssc::ceil_div(n_fields_in, fields)), chunks);
    launch(shared ? ssc::combine_bwd_wide_kernel<true> : ssc::combine_bwd_wide_kernel<false>, grid,
           ssc::kWideWaves * 64, first_out, n_fields_out, first_in, n_fields_in);
  } else {
    launch(ssc::combine_bwd_kernel, dim3((unsigned)n_fields_out, (unsigned)n_fields_in, chunks),
           256, first_out, first_in);
  }
  SSC_LAUNCH_CHECK("combine_bwd");
  return SSC_OK;
}

extern "C" int ssc_kernel_combine_f32(const float *weight, const float *basis,
                                      const int32_t *chan_out, const int32_t *chan_in,
                                      const int32_t *blocks, int32_t n_irreps_in,
                                      int32_t kernel_volume, int32_t c_in, int32_t c_out,
                                      float *out, ssc_stream_t stream) {
  SSC_CHECK(weight && basis && chan_out && chan_in && blocks && out, SSC_EINVAL,
            "NULL pointer argument");
  SSC_CHECK(n_irreps_in >= 1 && kernel_volume >= 1 && c_in >= 1 && c_out >= 1, SSC_EINVAL,
            "sizes must be positive");
  int64_t total = (int64_t)kernel_volume * c_in * c_out;
  hipLaunchKernelGGL(ssc::combine_kernel, dim3((unsigned)ssc::ceil_div(total, 256)), dim3(256), 0,
                     (hipStream_t)stream, weight, basis, chan_out, chan_in, blocks, n_irreps_in,
                     kernel_volume, c_in, c_out, out);
  SSC_LAUNCH_CHECK("combine");
  return SSC_OK;
}
