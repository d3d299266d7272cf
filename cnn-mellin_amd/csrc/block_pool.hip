// Maximum over pairs of neighbouring columns (frequency pooling) on channel-blocked tensors (block_gemm.hpp), forward and
// backward: streaming passes, a unit (eight channels of a position) of the smaller tensor to a thread.  The backward pass
// also applies the ReLU in front of the pooling, whose sign the pooled value has, and sums the gradients of each channel;
// so nothing of the unpooled tensor is needed.  64 channels of 32 x 780 x 41, fp32: 125 and 190 us, where the kernels on
// tensors as they lie (four bytes a value instead of six, no sums, no ReLU) take 106 and 93 and the pooled tensor would
// take another 128 to lay out.
#include <algorithm>

#include "block_gemm.hpp"
#include "tile_stage.hpp"

namespace mellin {

namespace {

constexpr int kPoolThreads = 256;

template <bool F16>
__device__ __forceinline__ void load_unit(const char *p, uintx4 (&u)[F16 ? 1 : 3]) {
#pragma unroll
  for (int i = 0; i < (F16 ? 1 : 3); ++i) u[i] = ((const uintx4 *)p)[i];
}
template <bool F16>
__device__ __forceinline__ float value(const uintx4 (&u)[F16 ? 1 : 3], int c) {
  const int sh = 16 * (c & 1);
  if constexpr (F16) {
    return (float)__builtin_bit_cast(_Float16, (unsigned short)(u[0][c >> 1] >> sh));
  } else {
    float v[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) v[i] = __uint_as_float((u[i][c >> 1] >> sh) << 16);
    return (v[0] + v[1]) + v[2];                       // (exact: the parts of one fp32 value)
  }
}

struct PoolArgs {
  const char *x, *y, *gy;
  char *out;
  unsigned char *which;
  float *partial;
  int groups, channels, batch, rows, cols, half_cols, chunks;
};

template <bool F16>
__global__ __launch_bounds__(kPoolThreads) void block_pool_kernel(PoolArgs a) {
  constexpr int PARTS = F16 ? 1 : 3, UB = 16 * PARTS;
  const i64 ng = blockIdx.y + (i64)blockIdx.z * gridDim.y;       // (image, group)
  const int plane_x = a.rows * a.cols, plane_y = a.rows * a.half_cols;
  const int j = blockIdx.x * kPoolThreads + threadIdx.x;
  if (j > plane_y) return;
  char *y = a.out + (ng * (plane_y + 1) + j) * UB;
  if (j == plane_y) {                                  // the unit of zeros
    const uintx4 zero = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < PARTS; ++i) ((uintx4 *)y)[i] = zero;
    return;
  }
  const int row = j / a.half_cols, col = j - row * a.half_cols;
  uintx4 u[PARTS], w[PARTS];
  const char *x = a.x + (ng * (plane_x + 1) + row * a.cols + 2 * col) * UB;
  load_unit<F16>(x, u);
  load_unit<F16>(x + UB, w);
  unsigned long long which = 0;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const float p = value<F16>(u, c), q = value<F16>(w, c);
    if (q > p || q != q) {
      which |= 1ull << (8 * c);
      const unsigned m = c & 1 ? 0xFFFF0000u : 0xFFFFu;
#pragma unroll
      for (int i = 0; i < PARTS; ++i) u[i][c >> 1] = (u[i][c >> 1] & ~m) | (w[i][c >> 1] & m);
    }
  }
#pragma unroll
  for (int i = 0; i < PARTS; ++i) ((uintx4 *)y)[i] = u[i];
  if (a.which) ((unsigned long long *)a.which)[ng * plane_y + j] = which;
}

template <bool F16>
__global__ __launch_bounds__(kPoolThreads) void block_pool_grad_kernel(PoolArgs a) {
  constexpr int PARTS = F16 ? 1 : 3, UB = 16 * PARTS;
  __shared__ float red[kPoolThreads / 64][8];
  const int group = blockIdx.y, n = blockIdx.z;
  const i64 ng = group + (i64)n * gridDim.y;
  const int plane_x = a.rows * a.cols, plane_y = a.rows * a.half_cols;
  const uintx4 zero = {0, 0, 0, 0};
  float sum[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) sum[c] = 0.f;
#pragma unroll 1
  for (int turn = 0; turn < 4; ++turn) {
    const int j = (blockIdx.x * 4 + turn) * kPoolThreads + threadIdx.x;
    if (j > plane_y) break;
    if (j == plane_y) {
      uintx4 *z = (uintx4 *)(a.out + (ng * (plane_x + 1) + plane_x) * UB);
#pragma unroll
      for (int i = 0; i < PARTS; ++i) z[i] = zero;
      break;
    }
    const int row = j / a.half_cols, col = j - row * a.half_cols;
    uintx4 g[PARTS];
    load_unit<F16>(a.gy + (ng * (plane_y + 1) + j) * UB, g);
    const uintx4 y = *(const uintx4 *)(a.y + (ng * (plane_y + 1) + j) * UB);
    const unsigned long long which = ((const unsigned long long *)a.which)[ng * plane_y + j];
    uintx4 first[PARTS], second[PARTS];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      unsigned keep = 0, to = 0;                       // channels whose value passed the ReLU; whose second value was taken
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const unsigned m = h ? 0xFFFF0000u : 0xFFFFu;
        if ((short)(y[k] >> (16 * h)) > 0) keep |= m;
        if ((which >> (8 * (2 * k + h))) & 1) to |= m;
      }
#pragma unroll
      for (int i = 0; i < PARTS; ++i) {
        g[i][k] &= keep;
        first[i][k] = g[i][k] & ~to;
        second[i][k] = g[i][k] & to;
      }
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) sum[c] += value<F16>(g, c);
    uintx4 *o = (uintx4 *)(a.out + (ng * (plane_x + 1) + row * a.cols + 2 * col) * UB);
#pragma unroll
    for (int i = 0; i < PARTS; ++i) {
      o[i] = first[i];
      o[PARTS + i] = second[i];
    }
    if (2 * col + 3 == a.cols) {                       // an odd last column takes no part
#pragma unroll
      for (int i = 0; i < PARTS; ++i) o[2 * PARTS + i] = zero;
    }
  }
  // sums in a fixed order: a shuffle tree per wavefront, the wavefronts in order
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum[c] += __shfl_down(sum[c], o);
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int c = 0; c < 8; ++c) red[threadIdx.x >> 6][c] = sum[c];
  __syncthreads();
  const int c = group * 8 + (int)threadIdx.x;
  if (threadIdx.x < 8 && c < a.channels) {
    float s = 0.f;
    for (int w = 0; w < kPoolThreads / 64; ++w) s += red[w][threadIdx.x];
    a.partial[((i64)c * a.batch + n) * a.chunks + blockIdx.x] = s;
  }
}

int pool_chunks(i64 rows, i64 cols) { return (int)(rows * (cols / 2) / (4 * kPoolThreads) + 1); }      // (with the unit of zeros)

PoolArgs pool_args(i64 batch, i64 channels, i64 rows, i64 cols) {
  PoolArgs a = {};
  a.groups = (int)((channels + 7) / 8);
  a.channels = (int)channels; a.batch = (int)batch; a.rows = (int)rows; a.cols = (int)cols; a.half_cols = (int)(cols / 2);
  a.chunks = pool_chunks(rows, cols);
  return a;
}

}  // namespace

size_t pool_partial_count(i64 batch, i64 channels, i64 rows, i64 cols) { return (size_t)(batch * channels * pool_chunks(rows, cols)); }

hipError_t launch_block_pool(bool f16, const void *x, i64 batch, i64 channels, i64 rows, i64 cols, void *y, void *which, hipStream_t stream) {
  PoolArgs a = pool_args(batch, channels, rows, cols);
  a.x = (const char *)x; a.out = (char *)y; a.which = (unsigned char *)which;
  const dim3 grid((unsigned)(rows * (cols / 2) / kPoolThreads + 1), (unsigned)a.groups, (unsigned)batch);
  if (f16) hipLaunchKernelGGL(block_pool_kernel<true>, grid, dim3(kPoolThreads), 0, stream, a);
  else hipLaunchKernelGGL(block_pool_kernel<false>, grid, dim3(kPoolThreads), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_block_pool_grad(bool f16, const void *grad_y, const void *y, const void *which, i64 batch, i64 channels, i64 rows,
                                  i64 cols, void *grad_x, float *partial, hipStream_t stream) {
  PoolArgs a = pool_args(batch, channels, rows, cols);
  a.gy = (const char *)grad_y; a.y = (const char *)y; a.which = (unsigned char *)which; a.out = (char *)grad_x; a.partial = partial;
  const dim3 grid((unsigned)a.chunks, (unsigned)a.groups, (unsigned)batch);
  if (f16) hipLaunchKernelGGL(block_pool_grad_kernel<true>, grid, dim3(kPoolThreads), 0, stream, a);
  else hipLaunchKernelGGL(block_pool_grad_kernel<false>, grid, dim3(kPoolThreads), 0, stream, a);
  return hipGetLastError();
}

}  // namespace mellin
