// Operands of the channel-blocked matrix kernels (block_gemm.hpp): the signal with eight channels
// of a position side by side, and the filter as fragments.
//
// Both are streaming passes.  Signal: a thread owns one position of a group of eight channels,
// reads its eight values (consecutive threads: consecutive words of a channel), cuts them once
// into bf16 parts (fp32) and writes 48 or 16 consecutive bytes.  It replaces the cuts that a
// matrix kernel reading fp32 words makes per use -- kx * ky times per element and tile of output
// channels -- which kept those kernels' vector pipe as busy as their matrix pipe.  Where the
// layer's backward pass also wants the bias gradient and the backward of a fused ReLU, they
// ride along: the gradient is read once, and its masked form is written in this layout only.
#include <algorithm>

#include "block_gemm.hpp"
#include "tile_stage.hpp"

namespace mellin {

namespace {

constexpr int kPackThreads = 256;
constexpr int kPackPositions = 4;                  // per thread

template <bool F16, bool MASK, bool SUM>
__global__ __launch_bounds__(kPackThreads) void pack_signal_kernel(const void *__restrict__ xv, const void *__restrict__ maskv,
                                                                   int channels, int plane, char *__restrict__ blocked,
                                                                   float *__restrict__ partial) {
  typedef typename std::conditional<F16, _Float16, float>::type T;
  constexpr int UB = F16 ? 16 : 48;
  const int groups = gridDim.y, cg = blockIdx.y, n = blockIdx.z, batch = gridDim.z;
  const int c0 = cg * 8, live = min(8, channels - c0);
  const T *x = (const T *)xv + ((i64)n * channels + c0) * plane;
  const T *mk = MASK ? (const T *)maskv + ((i64)n * channels + c0) * plane : nullptr;
  char *out = blocked + ((i64)n * groups + cg) * (i64)(plane + 1) * UB;
  float sum[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) sum[c] = 0.f;
  const int q0 = blockIdx.x * (kPackThreads * kPackPositions) + threadIdx.x;
#pragma unroll
  for (int i = 0; i < kPackPositions; ++i) {
    const int q = q0 + i * kPackThreads;
    if (q < plane) {
      T v[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = c < live ? x[(i64)c * plane + q] : (T)0;
      if (MASK) {
#pragma unroll
        for (int c = 0; c < 8; ++c)
          if (c < live) v[c] = mk[(i64)c * plane + q] > (T)0 ? v[c] : (T)0;
      }
      if (SUM) {
#pragma unroll
        for (int c = 0; c < 8; ++c) sum[c] += (float)v[c];
      }
      uintx4 *o = (uintx4 *)(out + (i64)q * UB);
      if constexpr (F16) {
        uintx4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          w[j] = (unsigned)__builtin_bit_cast(unsigned short, v[2 * j]) | ((unsigned)__builtin_bit_cast(unsigned short, v[2 * j + 1]) << 16);
        o[0] = w;
      } else {
        uintx4 hi, mid, lo;
        split8(v, hi, mid, lo);
        o[0] = hi;
        o[1] = mid;
        o[2] = lo;
      }
    } else if (q == plane) {
      uintx4 *o = (uintx4 *)(out + (i64)q * UB);
      const uintx4 zero = {0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < UB / 16; ++j) o[j] = zero;
    }
  }
  if (SUM) {
    // sums in a fixed order: a shuffle tree per wavefront, the wavefronts in order
    __shared__ float red[kPackThreads / 64][8];
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) sum[c] += __shfl_down(sum[c], o);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
      for (int c = 0; c < 8; ++c) red[threadIdx.x >> 6][c] = sum[c];
    __syncthreads();
    if ((int)threadIdx.x < live) {
      float a = 0.f;
      for (int w = 0; w < kPackThreads / 64; ++w) a += red[w][threadIdx.x];
      partial[((i64)(c0 + threadIdx.x) * batch + n) * gridDim.x + blockIdx.x] = a;
    }
  }
}

// Fragment of (32 output channels mt, group of eight contracted channels cg, filter row fx, filter
// column fy): the eight values of row r as part p at
//   frag[((mt * (CG * nfx * nfy + 1) + (cg * nfx + fx) * nfy + fy) * parts + p) * 32 + r]   (16-byte words)
// and a unit of zeros behind each tile of 32 channels.
template <bool F16>
__global__ __launch_bounds__(kPackThreads) void pack_filter_kernel(BlockPlan pl, int channels, const void *__restrict__ fv,
                                                                   uintx4 *__restrict__ frag) {
  typedef typename std::conditional<F16, _Float16, float>::type T;
  const i64 idx = (i64)blockIdx.x * kPackThreads + threadIdx.x;
  const int taps = pl.nfx * pl.nfy, per_tile = pl.CG * taps + 1;
  const i64 total = (i64)pl.m_tiles * pl.wm * pl.mt * per_tile * 32;
  if (idx >= total) return;
  const int r = (int)(idx & 31);
  const int unit = (int)(idx >> 5);
  const int mt = unit / per_tile, ct = unit - mt * per_tile;
  const int cg = ct / taps, tap = ct - cg * taps;                      // (cg == CG: the zeros)
  const int fx = tap / pl.nfy, fy = tap - fx * pl.nfy;
  const int m = mt * 32 + r;
  const T *f = (const T *)fv + (i64)m * pl.f_m + fx * pl.f_pitch + pl.f_off + fy;
  T v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (m < pl.M && cg < pl.CG && cg * 8 + i < channels) ? f[(i64)(cg * 8 + i) * pl.f_c] : (T)0;
  uintx4 *o = frag + (i64)unit * (F16 ? 32 : 96) + r;
  if constexpr (F16) {
    uintx4 w;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      w[j] = (unsigned)__builtin_bit_cast(unsigned short, v[2 * j]) | ((unsigned)__builtin_bit_cast(unsigned short, v[2 * j + 1]) << 16);
    o[0] = w;
  } else {
    uintx4 hi, mid, lo;
    split8(v, hi, mid, lo);
    o[0] = hi;
    o[32] = mid;
    o[64] = lo;
  }
}

i64 pack_chunks(i64 plane) { return plane / (kPackThreads * kPackPositions) + 1; }     // (plane + 1 units)

}  // namespace

size_t pack_partial_count(i64 batch, i64 channels, i64 plane) {
  return (size_t)(batch * channels * pack_chunks(plane));
}

hipError_t launch_pack_signal(const void *x, const void *relu_out, bool f16, i64 batch, i64 channels, i64 plane,
                              void *blocked, float *partial, hipStream_t stream) {
  const dim3 grid((unsigned)pack_chunks(plane), (unsigned)((channels + 7) / 8), (unsigned)batch);
#define MELLIN_PACK_CASE(F_, M_, S_)                                                                                     \
  if (f16 == F_ && (relu_out != nullptr) == M_ && (partial != nullptr) == S_)                                            \
    hipLaunchKernelGGL((pack_signal_kernel<F_, M_, S_>), grid, dim3(kPackThreads), 0, stream, x, relu_out, (int)channels, \
                       (int)plane, (char *)blocked, partial);
  MELLIN_PACK_CASE(false, false, false)
  MELLIN_PACK_CASE(false, false, true)
  MELLIN_PACK_CASE(false, true, false)
  MELLIN_PACK_CASE(false, true, true)
  MELLIN_PACK_CASE(true, false, false)
  MELLIN_PACK_CASE(true, false, true)
  MELLIN_PACK_CASE(true, true, false)
  MELLIN_PACK_CASE(true, true, true)
#undef MELLIN_PACK_CASE
  return hipGetLastError();
}

hipError_t launch_pack_filter(const BlockPlan &pl, int channels, const void *f, void *frag, hipStream_t stream) {
  const i64 total = (i64)pl.m_tiles * pl.wm * pl.mt * ((i64)pl.CG * pl.nfx * pl.nfy + 1) * 32;
  const dim3 grid((unsigned)((total + kPackThreads - 1) / kPackThreads));
  if (pl.f16)
    hipLaunchKernelGGL(pack_filter_kernel<true>, grid, dim3(kPackThreads), 0, stream, pl, channels, f, (uintx4 *)frag);
  else
    hipLaunchKernelGGL(pack_filter_kernel<false>, grid, dim3(kPackThreads), 0, stream, pl, channels, f, (uintx4 *)frag);
  return hipGetLastError();
}

}  // namespace mellin
