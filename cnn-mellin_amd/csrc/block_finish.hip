// The sums that end a pass of the channel-blocked kernels (block_gemm.hpp), in one launch: weight
// gradients from their partial blocks, bias gradients from the packing pass's partial sums, and the
// output of a pass whose contracted channels were dealt to several workgroups.  Each is a short
// streaming sum in a fixed order; on small layers a launch of its own (3-5 us each) cost more than
// the sum, so they share one -- those of all layers of a stack, as far as their partial sums are kept.
#include <algorithm>

#include "block_gemm.hpp"
#include "tile_stage.hpp"

namespace mellin {

namespace {

constexpr int kFinishThreads = 256;
constexpr int kSliceValues = kFinishThreads * 4;       // values of a tile that a block adds up

// (JOBS: 1 or kFinishJobs: a layer's launch does not carry a stack's arguments; measured at kPackFilters)
struct SliceSums {
  BlockPlan s;
  BlockGemmArgs sa;
  const int2 *s_rows;
};
template <int JOBS>
struct FinishArgs : SliceSums {
  int n_weights, n_biases;
  WeightSums w[JOBS];
  BiasSums b[JOBS];
};
static_assert(sizeof(FinishArgs<kFinishJobs>) <= 4096, "kernel arguments are limited to 4 KB");

// p[0] + p[step] + .. + p[(count - 1) step], added to `s` in that order.  Eight loads are on their way at a time: a sum is a
// chain of trips to memory, and with one or four the sums of a few channels over an image's many tiles took 20-27 us a
// launch, whatever their size (16000 partial sums of each of 32 channels: 22 -> 6 us).
__device__ __forceinline__ float add_chain(const float *__restrict__ p, i64 step, int count, float s) {
  constexpr int kAtOnce = 8;
  int k = 0;
  for (; k + kAtOnce <= count; k += kAtOnce, p += kAtOnce * step) {
    float v[kAtOnce];
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i) v[i] = p[i * step];
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i) s += v[i];
  }
  float v[kAtOnce];
#pragma unroll
  for (int i = 0; i < kAtOnce - 1; ++i) v[i] = k + i < count ? p[i * step] : 0.f;
#pragma unroll
  for (int i = 0; i < kAtOnce - 1; ++i)
    if (k + i < count) s += v[i];
  return s;
}

// The same of four values side by side, eight of them added pairwise at a time (which rounds less than one after the other).
__device__ __forceinline__ float4 add_chain4(const float *__restrict__ p, i64 step, int count) {
  constexpr int kAtOnce = 8;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int k = 0; k < count; k += kAtOnce, p += kAtOnce * step) {
    float4 v[kAtOnce];
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i) v[i] = k + i < count ? *(const float4 *)(p + i * step) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int n = kAtOnce / 2; n > 0; n /= 2)
#pragma unroll
      for (int i = 0; i < n; ++i) {
        v[i].x += v[i + n].x; v[i].y += v[i + n].y; v[i].z += v[i + n].z; v[i].w += v[i + n].w;
      }
    s.x += v[0].x; s.y += v[0].y; s.z += v[0].z; s.w += v[0].w;
  }
  return s;
}

// gw[m, c, fx, fy] = the sum of its partial sums.  A block owns an output channel and 32 input channels with `tap_chunk` of their
// taps, which it writes side by side; eight threads add the partial sums of a tap over one of `parts` of the slices, 16 bytes a
// thread, and the parts are added in order.  What bounds it is reading the partial sums, 64 KB of each of the weight
// gradient's workgroups.  A block of 32 weights of one tap, or all slices a thread, four bytes at a time, took up to twice the
// time, and wrote four bytes of every line: half, 128 -> 128 channels, 4 x 4 taps 20.6 -> 14.2 us, 256 -> 256 25 -> 14.3 and 128 ->
// 256, 3 x 3 taps, fp32 28 -> 22.
template <typename T>
__device__ void finish_weight(const WeightSums &pl, int b, float *__restrict__ red) {
  constexpr int kRow = 33;
  const int all_taps = pl.nfx * pl.nfy, c_tiles = (pl.C + 31) / 32;
  const int m = b % pl.M;
  b /= pl.M;
  const int chunk = b / c_tiles, c_tile = b - chunk * c_tiles, tap0 = chunk * pl.tap_chunk, taps = min(pl.tap_chunk, all_taps - tap0);
  const int parts = pl.parts, t = threadIdx.x, c4 = (t & 7) * 4, part = (t >> 3) / taps, tap = (t >> 3) - part * taps;
  if (part < parts) {
    const int fx = (tap0 + tap) / pl.nfy, fy = tap0 + tap - fx * pl.nfy, slices = pl.slices[fx];
    const int lo = slices * part / parts, hi = slices * (part + 1) / parts;
    const int mb = m / pl.m_t, ml = m - mb * pl.m_t, cb = c_tile / pl.ctb, ct = c_tile - cb * pl.ctb;
    const int cols = pl.ctb * pl.nfy * 32, blocks = pl.m_blocks * pl.c_blocks;
    const i64 stride = (i64)blocks * pl.m_t * cols;
    const float4 s = add_chain4(pl.partial + ((i64)pl.slice0[fx] * blocks + mb * pl.c_blocks + cb) * (i64)pl.m_t * cols + (i64)ml * cols +
                                    (ct * pl.nfy + fy) * 32 + c4 + lo * stride,
                                stride, hi - lo);
    float *to = red + (part * taps + tap) * kRow + c4;
    to[0] = s.x; to[1] = s.y; to[2] = s.z; to[3] = s.w;
  }
  __syncthreads();
  const int live = min(32, pl.C - c_tile * 32) * taps;
  T *out = (T *)pl.grad + ((i64)m * pl.C + c_tile * 32) * pl.nfx * pl.f_pitch + pl.f_off;
  for (int i = t; i < live; i += kFinishThreads) {
    const int c = i / taps, tp = i - c * taps, fx = (tap0 + tp) / pl.nfy, fy = tap0 + tp - fx * pl.nfy;
    float a = red[tp * kRow + c];
    for (int k = 1; k < parts; ++k) a += red[(k * taps + tp) * kRow + c];
    out[(c * pl.nfx + fx) * pl.f_pitch + fy] = (T)a;
  }
}

// Eight values as a unit of a blocked tensor.
template <typename T>
__device__ __forceinline__ void make_unit(const float (&v)[8], uintx4 (&u)[sizeof(T) == 2 ? 1 : 3]) {
  if constexpr (sizeof(T) == 2) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      u[0][j] = (unsigned)__builtin_bit_cast(unsigned short, (_Float16)v[2 * j]) | ((unsigned)__builtin_bit_cast(unsigned short, (_Float16)v[2 * j + 1]) << 16);
  } else {
    split8(v, u[0], u[1], u[2]);
  }
}

// Tiles in slices whose output is blocked or passes a ReLU: a thread makes a unit (eight channels of a position) -- of pooled
// ones the maxima of two positions, or both positions that a maximum was taken from; a block has 256 of a tile's, the positions
// side by side.
template <typename T>
__device__ void finish_units(const SliceSums &a, int b, float (*red)[32]) {
  constexpr bool F16 = sizeof(T) == 2;
  constexpr int PARTS = F16 ? 1 : 3, UB = 16 * PARTS;
  const BlockPlan &pl = a.s;
  const bool pool = pl.pool == 1, unpool = pl.pool == 2;
  const int m_t = pl.wm * pl.mt * 32, P = kWaves / pl.wk / pl.wm * pl.nt * 32, each_p = pool ? 2 : 1, PU = P / each_p, units = m_t / 8 * PU;
  const int chunks = (units + kFinishThreads - 1) / kFinishThreads;
  const int tm = b / chunks, at = (b - tm * chunks) * kFinishThreads + (int)threadIdx.x;      // (tile, tile of channels), unit in it
  const int r = tm / pl.m_tiles, g_t = at / PU, p = (at - g_t * PU) * each_p, group = (tm - r * pl.m_tiles) * (m_t / 8) + g_t;
  const int id = pl.whole + r, qt = id / pl.tile_batch, q0 = qt * P, count = min(P, pl.tile_q - q0);
  int n = id - qt * pl.tile_batch;
  const bool live = at < units && group < pl.out_groups && p < count;
  float v[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) v[c] = 0.f;
  if (live) {
    const i64 slice = (i64)pl.rest * pl.m_tiles * m_t * P;
    const float *from = a.sa.sums + (i64)tm * m_t * P + (i64)g_t * 8 * P + p;
    auto add_slices = [&](const float *from, float (&v)[8]) {
      for (int k = 0; k < pl.slices; ++k)
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] += from[k * slice + c * P];
      // (channels past the last have no sums: the matrix kernel's stores end with the last channel, and what the workspace
      // held there must not become a blocked tensor's padding)
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = group * 8 + c < pl.M ? v[c] : 0.f;
      if (!a.sa.grad && pl.relu)
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] = fmaxf(v[c], 0.f);
    };
    add_slices(from, v);
    int row = (q0 + p) / pl.noy;
    const int oy = q0 + p - row * pl.noy;
    if (pl.joint) { n = row % pl.batch; row /= pl.batch; }
    if (a.s_rows) row = a.s_rows[row].x;
    const int q = row * pl.noy + oy;
    const i64 of_group = (i64)n * pl.out_groups + group;
    const i64 unit = of_group * (pl.out_q + 1) + (pool ? q / 2 : unpool ? row * pl.out_cols + 2 * oy : q);
    unsigned long long which = 0;
    if (a.sa.grad) {
      const uintx4 x = *(const uintx4 *)((const char *)a.sa.mask + (of_group * (pl.Q + 1) + q) * UB);
#pragma unroll
      for (int c = 0; c < 8; ++c)
        if (!((short)(x[c >> 1] >> (16 * (c & 1))) > 0)) v[c] = 0.f;
      if (unpool) which = ((const unsigned long long *)a.sa.which)[of_group * pl.Q + q];
    }
    if (pool) {
      float w[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) w[c] = 0.f;
      add_slices(from + 1, w);
#pragma unroll
      for (int c = 0; c < 8; ++c)
        if ((T)w[c] > (T)v[c]) {                       // (of the values as they would be stored)
          which |= 1ull << (8 * c);
          v[c] = w[c];
        }
      if (a.sa.which) ((unsigned long long *)a.sa.which)[of_group * pl.out_q + q / 2] = which;
    }
    const uintx4 zero = {0, 0, 0, 0};
    if (a.sa.blocked) {
      uintx4 *o = (uintx4 *)((char *)a.sa.out + unit * UB), u[PARTS];
      make_unit<T>(v, u);
      if (unpool) {
#pragma unroll
        for (int i = 0; i < PARTS; ++i) {
          uintx4 m;
#pragma unroll
          for (int j = 0; j < 4; ++j) m[j] = ((which >> (16 * j)) & 1 ? 0xFFFFu : 0u) | ((which >> (16 * j + 8)) & 1 ? 0xFFFF0000u : 0u);
          o[i] = u[i] & ~m;
          o[PARTS + i] = u[i] & m;
          if (oy == pl.noy - 1 && (pl.out_cols & 1)) o[2 * PARTS + i] = zero;
        }
      } else {
#pragma unroll
        for (int i = 0; i < PARTS; ++i) o[i] = u[i];
      }
      // the unit of zeros behind the image
      if (pl.joint ? q == pl.Q - 1 : q0 + p + each_p == pl.Q) {
        uintx4 *z = (uintx4 *)((char *)a.sa.out + (of_group * (pl.out_q + 1) + pl.out_q) * UB);
#pragma unroll
        for (int i = 0; i < PARTS; ++i) z[i] = zero;
      }
    } else {
      T *o = (T *)a.sa.out + n * pl.h_n + (i64)group * 8 * pl.h_m + q;
#pragma unroll
      for (int c = 0; c < 8; ++c)
        if (group * 8 + c < pl.M) o[c * pl.h_m] = (T)v[c];
    }
  }
  if (a.sa.grad) {
    // channel sums of 32 positions, then of the nt * 32 (or 32) that share a place
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int o = 16; o > 0; o >>= 1) v[c] += __shfl_xor(v[c], o);
    const int hw = (int)threadIdx.x >> 5, each = pl.wk > 1 ? 1 : pl.nt;
    if ((threadIdx.x & 31) == 0)
#pragma unroll
      for (int c = 0; c < 8; ++c) red[c][hw] = v[c];
    __syncthreads();
    if ((threadIdx.x & 31) < 8 && hw % each == 0 && at < units && group < pl.out_groups) {
      const int c = threadIdx.x & 31, slots = P / 32 / each;
      float s = red[c][hw];
      for (int i = 1; i < each; ++i) s += red[c][hw + i];
      if (group * 8 + c < pl.M) a.sa.chan_sums[(i64)(group * 8 + c) * pl.chan_slots + (i64)id * slots + (p & ~31) / (32 * each)] = s;
    }
  }
}

template <typename T, typename TG, int JOBS>           // tensors, gradients of the parameters
__global__ __launch_bounds__(kFinishThreads) void block_finish_kernel(FinishArgs<JOBS> a) {
  __shared__ float red[8][32], weight_sums[kFinishThreads / 8 * 33];
  const int tid = threadIdx.x;
  unsigned b = blockIdx.x;
  for (int i = 0; i < a.n_weights; ++i) {
    const WeightSums &w = a.w[i];
    if (b < w.blocks) {
      finish_weight<TG>(w, (int)b, weight_sums);
      return;
    }
    b -= w.blocks;
    if (b < w.zero_blocks) {                           // filter columns that have no tap at all: zeros
      const i64 at = (i64)b * kFinishThreads + tid;
      const int fy = (int)(at % w.f_pitch);
      if (at < (i64)w.M * w.C * w.nfx * w.f_pitch && (fy < w.f_off || fy >= w.f_off + w.nfy)) ((TG *)w.grad)[at] = (TG)0;
      return;
    }
    b -= w.zero_blocks;
  }
  for (int i = 0; i < a.n_biases; ++i) {
    const BiasSums &c = a.b[i];
    if (b < c.channels) {
      // one channel: thread sums, a shuffle tree per wavefront, the wavefronts in order
      const float *p = c.partial + (i64)b * c.count;
      float s = tid < c.count ? add_chain(p + tid, kFinishThreads, (int)((c.count - tid + kFinishThreads - 1) / kFinishThreads), 0.f) : 0.f;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o);
      if ((tid & 63) == 0) red[0][tid >> 6] = s;
      __syncthreads();
      if (tid == 0) ((TG *)c.grad)[b] = (TG)(red[0][0] + red[0][1] + red[0][2] + red[0][3]);
      return;
    }
    b -= c.channels;
  }
  if (a.sa.blocked || a.sa.grad) {
    finish_units<T>(a, (int)b, red);
    return;
  }
  // a block: kSliceValues values of a tile, four positions of a channel a thread, the slices in order
  const BlockPlan &pl = a.s;
  const int m_t = pl.wm * pl.mt * 32, P = kWaves / pl.wk / pl.wm * pl.nt * 32, chunks = m_t * P / kSliceValues;
  const int tm = (int)b / chunks, at = ((int)b - tm * chunks) * kSliceValues + tid * 4;   // (tile, tile of channels), value in it
  const int r = tm / pl.m_tiles, c = at / P, p = at - c * P, m = (tm - r * pl.m_tiles) * m_t + c;
  const int id = pl.whole + r, qt = id / pl.tile_batch, n = id - qt * pl.tile_batch, q0 = qt * P, count = min(P, pl.tile_q - q0) - p;
  if (m >= pl.M || count <= 0) return;
  const i64 slice = (i64)pl.rest * pl.m_tiles * m_t * P;
  const float *from = a.sa.sums + (i64)tm * m_t * P + at;
  float4 v = *(const float4 *)from;
#pragma unroll 4
  for (int k = 1; k < pl.slices; ++k) {
    const float4 w = *(const float4 *)(from + k * slice);
    v.x += w.x; v.y += w.y; v.z += w.z; v.w += w.w;
  }
  if (pl.relu) v = make_float4(fmaxf(v.x, 0.f), fmaxf(v.y, 0.f), fmaxf(v.z, 0.f), fmaxf(v.w, 0.f));
  const float o[4] = {v.x, v.y, v.z, v.w};
  int row = (q0 + p) / pl.noy, oy = q0 + p - row * pl.noy;
  T *out = (T *)a.sa.out + n * pl.h_n + m * pl.h_m;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int at = pl.joint ? row / pl.batch : row;
    if (i < count) out[(pl.joint ? (row - at * pl.batch) * pl.h_n : 0) + (a.s_rows ? a.s_rows[at].x : at) * pl.noy + oy] = (T)o[i];
    if (++oy == pl.noy) { oy = 0; ++row; }
  }
}

}  // namespace

void BlockFinish::add_weight(const BlockWgradPlan &pl, const void *partial, void *grad) {
  WeightSums &w = weight[n_weights++];
  w = WeightSums{(const float *)partial, grad, pl.M, pl.C, pl.nfx, pl.nfy, pl.f_pitch, pl.f_off, pl.ctb, pl.wm * pl.mt * 32, pl.m_blocks,
                 pl.c_blocks, 0, 0, 0, 0, {}, {}};
  for (int f = 0; f < pl.nfx; ++f) {
    w.slice0[f] = (unsigned short)pl.row[f].slice0;
    w.slices[f] = (unsigned short)pl.row[f].slices;
  }
  // as many taps to a block as its threads hold -- longer runs of weights -- and leave two blocks a CU, or four where a thread's
  // share of the slices would be more than the eight loads that are on their way at a time (64 -> 64 channels, 5 x 3 taps, 100
  // slices a filter row: 10.0 -> 9.2 us with four; 41 -> 128 channels, 8 taps, 8 slices: 4.6 -> 5.5)
  const int taps = pl.nfx * pl.nfy;
  const i64 tiles = (i64)pl.M * ((pl.C + 31) / 32);
  w.tap_chunk = std::min(taps, kFinishThreads / 8);
  auto few = [&](int chunk) {
    const i64 blocks = tiles * ((taps + chunk - 1) / chunk);
    return blocks < 512 || (blocks < 1024 && pl.slices > pl.nfx * 8 * (kFinishThreads / 8 / chunk));
  };
  while (w.tap_chunk > 1 && few(w.tap_chunk)) w.tap_chunk = (w.tap_chunk + 1) / 2;
  w.parts = kFinishThreads / 8 / w.tap_chunk;
  w.blocks = (unsigned)(tiles * ((taps + w.tap_chunk - 1) / w.tap_chunk));
  if (pl.nfy != pl.f_pitch) w.zero_blocks = (unsigned)(((i64)pl.M * pl.C * pl.nfx * pl.f_pitch + kFinishThreads - 1) / kFinishThreads);
}

template <int JOBS>
static hipError_t launch_finish(bool f16, bool wide, const BlockFinish &job, hipStream_t stream) {
  FinishArgs<JOBS> a = {};
  i64 blocks = 0;
  a.n_weights = job.n_weights;
  a.n_biases = job.n_biases;
  for (int i = 0; i < job.n_weights; ++i) {
    a.w[i] = job.weight[i];
    blocks += (i64)a.w[i].blocks + a.w[i].zero_blocks;
  }
  for (int i = 0; i < job.n_biases; ++i) {
    a.b[i] = job.bias[i];
    blocks += a.b[i].channels;
  }
  i64 s_blocks = 0;
  if (job.slices && job.slices->rest > 0) {
    a.s = *job.slices;
    a.sa = job.args;
    if (a.s.kind_x == AX_MCORR || a.s.kind_x == AX_MCONV) a.s_rows = (const int2 *)((const char *)job.args.frag + a.s.rows_off);
    const i64 values = (i64)a.s.wm * a.s.mt * 32 * (kWaves / a.s.wk / a.s.wm * a.s.nt * 32);
    const i64 each = a.sa.blocked || a.sa.grad ? kFinishThreads * 8 : kSliceValues;
    s_blocks = (i64)a.s.rest * a.s.m_tiles * ((values + each - 1) / each);
  }
  blocks += s_blocks;
  if (blocks == 0) return hipSuccess;
  const dim3 grid((unsigned)blocks), threads(kFinishThreads);
  if (f16 && wide) hipLaunchKernelGGL((block_finish_kernel<_Float16, float, JOBS>), grid, threads, 0, stream, a);
  else if (f16) hipLaunchKernelGGL((block_finish_kernel<_Float16, _Float16, JOBS>), grid, threads, 0, stream, a);
  else hipLaunchKernelGGL((block_finish_kernel<float, float, JOBS>), grid, threads, 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_block_finish(bool f16, bool wide, const BlockFinish &job, hipStream_t stream) {
  return job.n_weights <= 1 && job.n_biases <= 1 ? launch_finish<1>(f16, wide, job, stream) : launch_finish<kFinishJobs>(f16, wide, job, stream);
}

}  // namespace mellin
