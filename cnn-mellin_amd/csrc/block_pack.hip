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
//
// All that a pass reads is packed by one launch: small layers are bound by launches, and the
// filter's few blocks hide behind the signal's.
#include <algorithm>

#include "block_gemm.hpp"
#include "tile_stage.hpp"

namespace mellin {

namespace {

constexpr int kPackThreads = 256;
constexpr int kPackPositions = 4;                  // per thread at most
// Positions that a thread takes one after the other, by the blocks that four would leave (30 signals each, 33 to 128 channels, us
// with four over us with one).  Few blocks wait for memory as often as they have positions: one in half below 1024 blocks
// (1.02 to 1.38 up to 780 of them; 0.97 to 1.04 from 1040 to 1280, 0.74 to 1.02 from 1560 to 19200: 128 channels of 32 x 256 x
// 41, 44.2 and 45.8) and in fp32 below 512 (0.98 to 1.12).  From there to the 2048 blocks that the chip holds at a time, four in
// fp32 (0.77 to 1.05); beyond, one, whose last round leaves less of the chip empty (1.05 to 1.46: 128 channels of 32 x 256 x 41,
// 104 and 81).  With sums: four, the order of sums that gives a bias gradient the same bits whether the input gradient is asked
// for beside it or not.
constexpr i64 kHalfBlocks = 1024, kFloatBlocks = 512, kResidentBlocks = 2048;

struct PackPart {                                  // a signal, dealt to blocks as (image, group, chunk of its plane)
  PackSignal s;
  int groups, positions, chunks;
  unsigned blocks;
};

template <bool F16, bool MASK, bool SUM>
__device__ __forceinline__ void pack_signal(const PackPart &pt, unsigned block, float (*red)[8]) {
  typedef typename std::conditional<F16, _Float16, float>::type T;
  constexpr int UB = F16 ? 16 : 48;
  const int groups = pt.groups, chunks = pt.chunks, plane = pt.s.plane, channels = pt.s.channels;
  const int row = (int)(block / (unsigned)chunks), chunk = (int)(block - (unsigned)row * (unsigned)chunks);
  const int n = row / groups, cg = row - n * groups;
  const int c0 = cg * 8, live = min(8, channels - c0);
  const T *x = (const T *)pt.s.x + ((i64)n * channels + c0) * plane;
  const T *mk = MASK ? (const T *)pt.s.relu_out + ((i64)n * channels + c0) * plane : nullptr;
  char *out = pt.s.blocked + ((i64)n * groups + cg) * (i64)(plane + 1) * UB;
  float sum[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) sum[c] = 0.f;
  const int q0 = chunk * (kPackThreads * pt.positions) + threadIdx.x;
#pragma unroll
  for (int i = 0; i < kPackPositions; ++i) {
    if (i >= pt.positions) break;
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
      pt.s.partial[((i64)(c0 + threadIdx.x) * pt.s.batch + n) * chunks + chunk] = a;
    }
  }
}

// Fragment of (32 output channels mt, group of eight contracted channels cg, filter row fx, filter
// column fy): the eight values of row r as part p at
//   frag[((mt * (CG * nfx * nfy + 1) + (cg * nfx + fx) * nfy + fy) * parts + p) * 32 + r]   (16-byte words)
// and a unit of zeros behind each tile of 32 channels.
template <bool F16, typename From>
__device__ __forceinline__ void pack_fragments(const PackFilterHead &pl, i64 idx) {
  typedef typename std::conditional<F16, _Float16, float>::type T;
  const int taps = pl.nfx * pl.nfy, per_tile = pl.CG * taps + 1;
  const i64 total = (i64)pl.tiles * per_tile * 32;
  if (idx >= total) return;
  const int r = (int)(idx & 31);
  const int unit = (int)(idx >> 5);
  const int mt = unit / per_tile, ct = unit - mt * per_tile;
  const int cg = ct / taps, tap = ct - cg * taps;                      // (cg == CG: the zeros)
  const int fx = tap / pl.nfy, fy = tap - fx * pl.nfy;
  const int m = mt * 32 + r;
  const From *f = (const From *)pl.f + (i64)m * pl.f_m + fx * pl.f_pitch + pl.f_off + fy;
  T v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (m < pl.M && cg < pl.CG && cg * 8 + i < pl.channels) ? (T)f[(i64)(cg * 8 + i) * pl.f_c] : (T)0;
  uintx4 *o = (uintx4 *)pl.frag + (i64)unit * (F16 ? 32 : 96) + r;
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

// Output row `row` of a Mellin axis in the order of its classes, with the filter rows that have a tap for it.
__device__ __forceinline__ int2 class_row(const PackFilterHead &pl, const BlockClass *cls, int row) {
  int ox = row;
  for (int k = 0; k < pl.n_classes; ++k)
    if (row >= cls[k].start) ox = cls[k].first + (row - cls[k].start) * pl.cls_stride;
  int mask = 0;
  for (int f = 0; f < pl.nfx; ++f)
    if (mellin_tap32(pl.kind_x, ox, f, pl.ngx, pl.sx, pl.dx, pl.px + 1, pl.ux, pl.mg_p1) >= 0) mask |= 1 << f;
  return make_int2(ox, mask);
}

// The filters of a stack of 16 layers and their classes go with one launch: with the classes of each at their most, six did,
// and ten layers took two (one utterance through ten Mellin layers 226.6 -> 223.4 us).
// A layer's launch has room for its one filter only: with a stack's arguments, 3.6 KB each of them and of the sums' launch,
// that are copied and fetched, 41 -> 128 channels on one axis took 85.0 us a step instead of 83.7, a half layer's output 49.0
// instead of 48.3.
constexpr int kPackFilters = 16, kPackClasses = 96;

template <int FILTERS>
struct PackArgs {
  static constexpr int kClasses = FILTERS == 1 ? kBlockClasses : kPackClasses;
  PackPart a, b;
  PackFilterHead filter[FILTERS];
  unsigned rows[FILTERS], fragments[FILTERS], copies[FILTERS];      // blocks
  short cls_at[FILTERS];
  int n_filters;
  BlockClass cls[kClasses];
};
static_assert(kPackClasses >= kBlockClasses && sizeof(PackArgs<kPackFilters>) <= 4096, "kernel arguments are limited to 4 KB");

template <bool F16, int FILTERS>
__global__ __launch_bounds__(kPackThreads) void block_pack_kernel(PackArgs<FILTERS> args) {
  __shared__ float red[kPackThreads / 64][8];
  unsigned b = blockIdx.x;
  for (int i = 0; i < args.n_filters; ++i) {
    const PackFilterHead &fl = args.filter[i];
    if (b < args.rows[i]) {
      const int row = (int)(b * kPackThreads + threadIdx.x);
      if (row < fl.nox) ((int2 *)(fl.frag + fl.rows_off))[row] = class_row(fl, args.cls + args.cls_at[i], row);
      return;
    }
    b -= args.rows[i];
    if (b < args.fragments[i]) {
      const i64 idx = (i64)b * kPackThreads + threadIdx.x;
      if (!F16 || fl.wide) pack_fragments<F16, float>(fl, idx);
      else pack_fragments<F16, _Float16>(fl, idx);
      return;
    }
    b -= args.fragments[i];
    if (b < args.copies[i]) {
      const i64 at = ((i64)b * kPackThreads + threadIdx.x) * 4;
      for (i64 k = at; k < min(at + 4, fl.copy_count); ++k) ((_Float16 *)fl.copy)[k] = (_Float16)((const float *)fl.f)[k];
      return;
    }
    b -= args.copies[i];
  }
  const bool second = b >= args.a.blocks;
  const PackPart &pt = second ? args.b : args.a;
  if (second) b -= args.a.blocks;
  if (pt.s.relu_out) {
    if (pt.s.partial) pack_signal<F16, true, true>(pt, b, red);
    else pack_signal<F16, true, false>(pt, b, red);
  } else {
    if (pt.s.partial) pack_signal<F16, false, true>(pt, b, red);
    else pack_signal<F16, false, false>(pt, b, red);
  }
}

i64 pack_chunks(i64 plane, int positions) { return plane / (kPackThreads * positions) + 1; }     // (plane + 1 units)
int pack_positions(bool half, const PackSignal &s, int groups) {
  if (s.partial) return kPackPositions;
  const i64 blocks = (i64)s.batch * groups * pack_chunks(s.plane, kPackPositions);
  return blocks < (half ? kHalfBlocks : kFloatBlocks) || (!half && blocks >= kResidentBlocks) ? 1 : kPackPositions;
}

bool pack_part(bool half, const PackSignal *s, PackPart &pt) {
  pt = PackPart{};
  if (!s) return true;
  pt.s = *s;
  pt.groups = (s->channels + 7) / 8;
  pt.positions = pack_positions(half, *s, pt.groups);
  pt.chunks = (int)pack_chunks(s->plane, pt.positions);
  const i64 blocks = (i64)s->batch * pt.groups * pt.chunks;
  pt.blocks = (unsigned)blocks;
  return blocks < (i64)1 << 30;
}

}  // namespace

size_t pack_partial_count(i64 batch, i64 channels, i64 plane) {
  return (size_t)(batch * channels * pack_chunks(plane, kPackPositions));
}

PackFilter pack_filter(const BlockPlan &pl, int channels, const void *f, void *frag, void *copy, i64 copy_count) {
  PackFilter pf = {{f, (char *)frag, copy, copy_count, pl.f_m, pl.f_c, pl.rows_off, channels, pl.wide, pl.M, pl.CG, pl.nfx, pl.nfy,
                   pl.f_pitch, pl.f_off, pl.m_tiles * pl.wm * pl.mt, pl.kind_x, pl.nox, pl.ngx, pl.sx, pl.dx, pl.px, pl.ux, pl.mg_p1,
                    pl.n_classes, pl.cls_stride}, {}};
  std::copy(pl.cls, pl.cls + kBlockClasses, pf.cls);
  return pf;
}

template <int FILTERS>
static hipError_t launch_pack(bool f16, const PackSignal *a, const PackSignal *b, const PackFilter *filters, int n_filters,
                              hipStream_t stream) {
  PackArgs<FILTERS> args = {};
  if (!pack_part(f16, a, args.a) || !pack_part(f16, b, args.b)) return hipErrorInvalidValue;
  do {
    unsigned blocks = args.a.blocks + args.b.blocks;
    int i = 0, classes = 0;
    for (; i < std::min(n_filters, FILTERS) && classes + filters[i].n_classes <= args.kClasses; ++i) {
      const PackFilter &fl = filters[i];
      args.filter[i] = fl;
      args.cls_at[i] = (short)classes;
      std::copy(fl.cls, fl.cls + fl.n_classes, args.cls + classes);
      classes += fl.n_classes;
      const i64 units = (i64)fl.tiles * ((i64)fl.CG * fl.nfx * fl.nfy + 1) * 32;
      args.fragments[i] = (unsigned)((units + kPackThreads - 1) / kPackThreads);
      args.rows[i] = fl.kind_x == AX_MCORR || fl.kind_x == AX_MCONV ? (unsigned)((fl.nox + kPackThreads - 1) / kPackThreads) : 0;
      args.copies[i] = fl.copy ? (unsigned)((fl.copy_count + 4 * kPackThreads - 1) / (4 * kPackThreads)) : 0;
      blocks += args.rows[i] + args.fragments[i] + args.copies[i];
    }
    args.n_filters = i;
    if (blocks) {
      if (f16) hipLaunchKernelGGL((block_pack_kernel<true, FILTERS>), dim3(blocks), dim3(kPackThreads), 0, stream, args);
      else hipLaunchKernelGGL((block_pack_kernel<false, FILTERS>), dim3(blocks), dim3(kPackThreads), 0, stream, args);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
    args.a.blocks = args.b.blocks = 0;                 // (the signals went with the first launch)
    filters += args.n_filters;
    n_filters -= args.n_filters;
  } while (n_filters > 0);
  return hipSuccess;
}

hipError_t launch_block_pack(bool f16, const PackSignal *a, const PackSignal *b, const PackFilter *filters, int n_filters,
                             hipStream_t stream) {
  return n_filters <= 1 ? launch_pack<1>(f16, a, b, filters, n_filters, stream) : launch_pack<kPackFilters>(f16, a, b, filters, n_filters, stream);
}

}  // namespace mellin
