// Maximum over pairs of neighbouring columns (frequency pooling) of a channel-blocked tensor (block_gemm.hpp): a streaming
// pass, a unit (eight channels of a position) of the smaller tensor to a thread, behind layers whose own kernel cannot store the
// maxima in the order of sums that it has without the pooling (make_block_plan; elsewhere it does).  64 channels of 32 x 780
// x 41, fp32: 125 us, bound by the bytes (six a value).
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
  const char *x;
  char *out;
  unsigned char *which;
  int rows, cols, half_cols;
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

}  // namespace

hipError_t launch_block_pool(bool f16, const void *x, i64 batch, i64 channels, i64 rows, i64 cols, void *y, void *which, hipStream_t stream) {
  const PoolArgs a = {(const char *)x, (char *)y, (unsigned char *)which, (int)rows, (int)cols, (int)(cols / 2)};
  const dim3 grid((unsigned)(rows * (cols / 2) / kPoolThreads + 1), (unsigned)((channels + 7) / 8), (unsigned)batch);
  if (f16) hipLaunchKernelGGL(block_pool_kernel<true>, grid, dim3(kPoolThreads), 0, stream, a);
  else hipLaunchKernelGGL(block_pool_kernel<false>, grid, dim3(kPoolThreads), 0, stream, a);
  return hipGetLastError();
}

}  // namespace mellin
