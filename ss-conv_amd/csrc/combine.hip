// Steerable kernel synthesis: dense kernel = sum_beta weight * basis, written
// straight into the contiguous [K, Cin, Cout] layout the convolution consumes.
// One thread per output element; the per-channel descriptor tables replace the
// reference's loop over irrep pairs, its einsum, both concatenations and the
// permute.  The sum over beta runs in ascending order.
#include "combine_element.h"
#include "ssc_common.h"

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
// along the basis elements as they lie in memory (k fastest), eight basis functions at a time,
// and the threads' sums are added in a fixed order.  Bound by the latency of its few loads
// (442 KB of d_dense for 64 -> 64 channels and kernel 3): 13 us there, where matrix products
// block by block took 49 launches, 200 us and as much again of host time.
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
  for (int n0 = 0; n0 < n_beta; n0 += kBwdBeta) {
    const int n = min(kBwdBeta, n_beta - n0);
    float acc[kBwdBeta];
#pragma unroll
    for (int t = 0; t < kBwdBeta; ++t) acc[t] = 0.f;
    for (int e = threadIdx.x; e < elems; e += 256) {
      const int ab = e / K, k = e - ab * K;
      const int a = ab / d_in, b = ab - a * d_in;
      const float x = g[((int64_t)k * cin + b) * cout + a];
#pragma unroll
      for (int t = 0; t < kBwdBeta; ++t)
        if (t < n) acc[t] += x * bs[(int64_t)(n0 + t) * elems + e];
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
  SSC_CHECK(n_fields_out >= 1 && n_fields_out <= c_out && n_fields_in >= 1 && n_fields_in <= c_in &&
                n_fields_in <= 65535,
            SSC_EINVAL, "field counts out of range");
  hipLaunchKernelGGL(ssc::combine_bwd_kernel, dim3((unsigned)n_fields_out, (unsigned)n_fields_in),
                     dim3(256), 0, (hipStream_t)stream, d_dense, basis, chan_out, chan_in, blocks,
                     first_out, first_in, n_irreps_in, kernel_volume, c_in, c_out, d_weight);
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
