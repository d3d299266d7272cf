// The sums that end a weight gradient of wgrad_gemm.hip, as a block of 256 threads makes them: in a launch of their own, or in
// the last launch of the same layer's input gradient, which waits for memory just as long.
#pragma once

#include "mellin_common.hpp"

namespace mellin {

// W[m, j] = sum over the S partial blocks, in a fixed order.  A block of 256
// threads handles 16 outputs: 16 threads per output add every 16th partial,
// then thread 0 of each output adds the 16 sums in pairs.  Behind the M J weights
// come, with bias_ws, the M sums of grad_out: gb[m] of the partial sums bias_ws[s, m].
template <typename O>                                  // O: float, or _Float16 (rounded once)
__device__ __forceinline__ void wgrad_reduce_block(const float *__restrict__ ws, O *__restrict__ W, int S, int M, int J, int M_pad,
                                                   int J_pad, const float *__restrict__ bias_ws, O *__restrict__ gb, unsigned block) {
  __shared__ float part[16][17];
  const int el = threadIdx.x & 15, ph = threadIdx.x >> 4;
  const int e = block * 16 + el, outputs = M * J + (bias_ws ? M : 0);
  float sum = 0.f;
  if (e < outputs) {
    const int m = e / J, j = e - m * J;
    const bool weight = e < M * J;
    const float *src = weight ? ws + (i64)m * J_pad + j : bias_ws + (e - M * J);
    const i64 stride = weight ? (i64)M_pad * J_pad : M_pad;
    int s = ph;
    for (; s + 48 < S; s += 64) {
      const float v0 = src[(i64)s * stride], v1 = src[(i64)(s + 16) * stride];
      const float v2 = src[(i64)(s + 32) * stride], v3 = src[(i64)(s + 48) * stride];
      sum += (v0 + v1) + (v2 + v3);
    }
    for (; s < S; s += 16) sum += src[(i64)s * stride];
  }
  part[ph][el] = sum;
  __syncthreads();
  if (ph == 0 && e < outputs) {
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = part[k][el];
#pragma unroll
    for (int n = 8; n > 0; n >>= 1)
#pragma unroll
      for (int k = 0; k < n; ++k) v[k] += v[k + n];
    const float tot = v[0];
    (e < M * J ? W[e] : gb[e - M * J]) = (O)tot;
  }
}

__device__ __forceinline__ void wgrad_reduce_block(const WgradReduce &r, unsigned block) {
  wgrad_reduce_block<float>(r.ws, r.W, r.S, r.M, r.J, r.M_pad, r.J_pad, r.bias_ws, r.gb, block);
}

}  // namespace mellin
