// Weight gradient of layers with many channels, from channel-blocked tensors (block_gemm.hpp) on
// the bf16 / f16 matrix cores.
//
//   W[m, c, fx, fy] = sum_{n, ox, oy} A[n, m, ox, oy] * G[n, c, tap_x(ox, fx), tap_y(oy, fy)]
//
// A = grad_out and G = the layer's input, both blocked.  The contracted index runs over output
// positions; a matrix operand wants eight consecutive ones of a channel per lane while the blocked
// tensors hold eight channels of a position, so operands come out of LDS through the transposing
// read (ds_read_b64_tr_b16: sixteen lanes read four positions x sixteen channels and each receives
// four positions of one channel).  A position's unit of the input serves every filter column: a
// tap is an offset of whole units.
//
// A workgroup owns one filter row fx, MB * 32 output channels and CB * 32 input channels with all
// filter columns, for a slice of the rows of all images that have a tap of fx -- those rows and no
// others: on a Mellin axis no row is staged or multiplied without its tap (the kernel that ran along
// whole rows, wgrad_pos.hip, multiplied every pair).  A stage is KS positions, in the order
// (image, row, column) and across images, so nothing is padded but the slice's end.  Input units are
// staged once per position and row piece: the row's columns and the filter's reach behind them.
// Both operands come by direct global->LDS loads (16 bytes per lane) from source tables in LDS that
// are worked out two stages ahead, one entry per thread.  There are no register loads in the loop,
// so the only wait for memory is the one at a stage's start, for loads issued a whole stage before.
//
// Every workgroup writes its sums as one partial block; block_finish.hip adds a weight's partial
// sums in slice order (bit-reproducible).
//
// Measured against wgrad_pos.hip, 128 -> 256 channels, 3 x 3 taps, 32 x 256 x 41 positions: fp32, linear rows 1171 -> 1000 us;
// half, Mellin rows 356 -> 112 us.  64 -> 64 channels, 4 x 4 taps, 32 x 780 x 20, fp32: Mellin rows 477 -> 200 us.
// Bound by what a stage costs beside its products (tables, loads' issue, the first operands after the barrier): a wavefront
// has 2 x 24 matrix instructions a stage in fp32 (1536 cycles), 4 x 8 in half (1024).  256 -> 256 channels, 4 x 4 taps,
// 32 x 780 x 5, fp32: 970 us with tables from divisions, 860 now (46 % of the cycles multiply), 660 without tables and loads.
#include <algorithm>
#include <type_traits>

#include "block_gemm.hpp"
#include "tile_stage.hpp"

namespace mellin {

namespace {

typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) shortx4 *lds_short4_ptr;
typedef const __attribute__((address_space(4))) BlockWgradPlan ConstWgradPlan;

// four values of k for this lane's channel (see above) from the LDS byte address `at`
__device__ __forceinline__ void read_transposed(unsigned at, unsigned &lo, unsigned &hi) {
  const shortx4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(size_t)at);
  const uint2 w = __builtin_bit_cast(uint2, v);
  lo = w.x;
  hi = w.y;
}

// Tiles of a wavefront that leave registers for separate sums of the small products (block_multiply_low).  Error of the
// weight gradient against 64 bits, 64 -> 64 channels, 4 x 4 taps, 8 x 390 x 20 positions: 2.7e-7 -> 1.3e-7, at the same time.
constexpr int kLowTiles = 4;

// NW: wavefronts of a workgroup -- four, two workgroups to a CU, or eight where a stage's operands leave room for
// one workgroup only
// Wavefronts of a SIMD that registers allow: more than two where tiles are small, whose stages are all latency.
constexpr int waves_per_simd(int mt, int nt, bool f16) { return f16 ? (mt * nt <= 4 ? 4 : mt * nt == 6 ? 3 : 2) : mt * nt == 1 ? 4 : mt * nt == 2 ? 3 : 2; }

template <int MT, int NT, int NW, bool F16>
__global__ __launch_bounds__(NW * 64, waves_per_simd(MT, NT, F16)) void block_wgrad_kernel(BlockWgradPlan plan_arg, const char *__restrict__ A,
                                                                  const char *__restrict__ G, float *__restrict__ ws) {
  constexpr int PARTS = F16 ? 1 : 3, UB = 16 * PARTS, KS = F16 ? 64 : 32, KSP = KS + 4;
  extern __shared__ __align__(16) char bw_lds[];
  ConstWgradPlan *plp = (ConstWgradPlan *)__builtin_amdgcn_kernarg_segment_ptr();
#define pl (*plp)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int WM = pl.wm;
  const int wm = wave % WM, wn = wave / WM;
  // this workgroup's filter row and slice, output-channel and input-channel block
  const int blocks = pl.m_blocks * pl.c_blocks;
  int fx, slice, block;
  {
    // XCD k (workgroups k, k + 8, ...) takes an eighth of the items without a gap: the blocks of a slice read the same rows
    // through one L2 (256 -> 256 channels, 4 x 4 taps, 32 x 780 x 5, fp32: misses 4.0 GB -> 1.3 GB)
    const int items = pl.slices * blocks, xcd = blockIdx.x & 7, item = xcd * (items >> 3) + min(xcd, items & 7) + (blockIdx.x >> 3);
    int at = item / blocks, left = pl.slices;
    block = item - at * blocks;
    // the filter rows' slices in turn, each row's spread evenly over those of the rows behind it
    for (fx = 0; fx + 1 < pl.nfx; ++fx) {
      const int n = pl.row[fx].slices, before = at * n / left;
      if ((at + 1) * n >= (before + 1) * left) { at = before; break; }
      at -= before;
      left -= n;
    }
    slice = at;
  }
  const int slices = pl.row[fx].slices;
  const int mb = block / pl.c_blocks, cb = block - mb * pl.c_blocks;
  const int mg0 = mb * pl.mgt, cg0 = cb * pl.cgt;
  const int mgs = min(pl.mgt, pl.MG - mg0), cgs = min(pl.cgt, pl.CG - cg0);
  const int ox_first = pl.row[fx].ox0, ox_step = pl.row[fx].step, gx0 = pl.row[fx].gx0, gx_step = pl.row[fx].gstep;
  const int count = pl.row[fx].count, noy = pl.noy;
  const int total = pl.batch * count * noy;            // positions (blocked tensors of < 2^32 bytes: fewer than 2^28)
  const int units = (total + KS - 1) / KS;
  const unsigned mg_noy = pl.mg_noy, mg_count = pl.row[fx].mg_count;
  const int u_lo = (int)((i64)units * slice / slices), u_hi = (int)((i64)units * (slice + 1) / slices);
  const int VP = pl.VP, a_bytes = pl.mgt * KSP * UB, buf_bytes = a_bytes + pl.cgt * VP * UB;
  const unsigned lds0 = lds_address((const float *)bw_lds);
  int *tabs = (int *)(bw_lds + 2 * buf_bytes);         // [3][KS (grad_out source) + KS (LDS unit) + VP (input source)]
  const int tab_words = 2 * KS + VP;
  const i64 a_plane = (i64)(pl.q_out + 1) * UB, g_plane = (i64)(pl.plane + 1) * UB;
  const char *A0 = A + (i64)mg0 * a_plane, *G0 = G + (i64)cg0 * g_plane;

  // The sources of a stage, one entry per thread (KS + VP <= threads): a position's units of grad_out and of the staged
  // input, or one of the staged units' source.  Threads keep their place (image, row, column) from stage to stage and add
  // KS positions to it with two carries: worked out from the stage's number, with divisions and products, the tables took
  // a fifth of the fp32 kernels' time and up to two fifths of half kernels'.
  const int full = pl.ay * (noy - 1) + pl.by_span + 1;                 // virtual units of a row
  const int wrap = full - pl.ay * noy;                                 // what a row's end adds to those of its positions
  const int rows_on = udiv(KS, noy, mg_noy), k_col = KS - rows_on * noy;
  const int k_image = udiv(rows_on, count, mg_count), k_row = rows_on - k_image * count;
  const unsigned a_image = (unsigned)pl.MG * (unsigned)(pl.q_out + 1) * UB, a_row = (unsigned)(ox_step * noy * UB);
  const unsigned g_image = (unsigned)pl.CG * (unsigned)(pl.plane + 1) * UB, g_row = (unsigned)(gx_step * pl.ngy * UB);
  int first_col;                                       // of the stage whose table is next
  int at_col, at_row, at_n;                            // (position: at_n its LDS address)
  unsigned at_source;                                  // input: of the row's first unit
  {
    const int first = u_lo * KS, row0 = udiv(first, noy, mg_noy);
    first_col = first - row0 * noy;
    int row = row0;
    if (tid < KS) {
      row = udiv(first + tid, noy, mg_noy);
      at_col = first + tid - row * noy;
    } else {
      at_col = tid - KS + pl.ay * first_col;
      const int r = at_col / full;
      at_col -= r * full;
      row += r;
    }
    const int n = udiv(row, count, mg_count);
    at_row = row - n * count;
    if (tid < KS) {
      at_source = (unsigned)n * a_image + (unsigned)(ox_first * noy * UB) + (unsigned)at_row * a_row + (unsigned)(at_col * UB);
      at_n = (pl.ay * (at_col - first_col) + (row - row0) * full) * UB;
    } else {
      at_source = (unsigned)n * g_image + (unsigned)(gx0 * pl.ngy * UB) + (unsigned)at_row * g_row;
      at_n = tid - KS < pl.zero_unit ? n : 1 << 30;    // (an image that is not there: zeros)
    }
  }
  auto build_tables = [&](int u) {                     // (called for u_lo, u_lo + 1, ...)
    int *t = tabs + (u % 3) * tab_words;
    const int next_col = first_col + k_col;
    const bool first_wraps = next_col >= noy;
    first_col = first_wraps ? next_col - noy : next_col;
    if (tid < KS) {
      const bool live = u * KS + tid < total;
      t[tid] = (int)(live ? at_source : (unsigned)(pl.q_out * UB));
      t[KS + tid] = live ? at_n : pl.zero_unit * UB;
      at_col += k_col;
      at_row += k_row;
      at_source += k_image * a_image + k_row * a_row + k_col * UB;
      at_n -= first_wraps ? wrap * UB : 0;
      if (at_col >= noy) { at_col -= noy; ++at_row; at_source += a_row - noy * UB; at_n += wrap * UB; }
      if (at_row >= count) { at_row -= count; at_source += a_image - count * a_row; }
    } else if (tid < KS + VP) {
      const int vy = pl.cy + at_col;
      int gy = vy;
      if (pl.uy != 1) {
        gy = vy / pl.uy;
        if (gy * pl.uy != vy) gy = -1;
      }
      const bool live = vy >= 0 && (unsigned)gy < (unsigned)pl.ngy && at_n < pl.batch;
      t[KS + tid] = (int)(live ? at_source + gy * UB : (unsigned)(pl.plane * UB));
      at_col += pl.ay * k_col + (first_wraps ? wrap : 0);              // (0 <= what is added < full)
      at_row += k_row;
      at_n += k_image;
      at_source += k_image * g_image + k_row * g_row;
      if (at_col >= full) { at_col -= full; ++at_row; at_source += g_row; }
      if (at_row >= count) { at_row -= count; ++at_n; at_source += g_image - count * g_row; }
    }
  };
  // the loads of stage u into buffer b: groups of channels dealt to the wavefronts
  auto issue = [&](int u, int b) {
    const int *t = tabs + (u % 3) * tab_words;
    const unsigned to = lds0 + (unsigned)(b * buf_bytes);
    constexpr int kSlots = KS * PARTS, kA = (kSlots + 63) / 64, kG = 4;
    const int slots = VP * PARTS;
    auto unit_of = [&](int slot) { return F16 ? slot : slot / 3; };
    auto part_of = [&](int slot) { return F16 ? 0 : (slot - slot / 3 * 3) * 16; };
    // every source that is needed (lanes without a slot: a slot that is there), then the loads: one wait for the tables
    unsigned a_src[kA], g_src[kG];
#pragma unroll
    for (int k = 0; k < kA; ++k) { const int slot = min(k * 64 + lane, kSlots - 1); a_src[k] = (unsigned)t[unit_of(slot)] + part_of(slot); }
#pragma unroll
    for (int k = 0; k < kG; ++k)
      if (k * 64 < slots) { const int slot = min(k * 64 + lane, slots - 1); g_src[k] = (unsigned)t[2 * KS + unit_of(slot)] + part_of(slot); }
    auto load_a = [&](int k) {
      const char *from = A0 + wave * a_plane;
      for (int g = wave; g < mgs; g += NW, from += NW * a_plane)
        load16_to_lds_at((const float *)from, a_src[k], to + (unsigned)(g * KSP * UB + k * 1024));
    };
    auto load_g = [&](int k, unsigned src) {
      const char *from = G0 + wave * g_plane;
      for (int g = wave; g < cgs; g += NW, from += NW * g_plane)
        load16_to_lds_at((const float *)from, src, to + (unsigned)(a_bytes + g * VP * UB + k * 1024));
    };
#pragma unroll
    for (int k = 0; k < kA; ++k)
      if (k * 64 + lane < kSlots) load_a(k);
#pragma unroll
    for (int k = 0; k < kG; ++k)
      if (k * 64 + lane < slots) load_g(k, g_src[k]);
    for (int k = kG; k * 64 < slots; ++k) {
      const int slot = k * 64 + lane;
      if (slot < slots) load_g(k, (unsigned)t[2 * KS + unit_of(slot)] + part_of(slot));
    }
  };

  floatx16 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][t][r] = 0.f;
  // fp32: sums of their own for the small products, where registers allow
  constexpr bool LOW = !F16 && MT * NT <= kLowTiles;
  floatx16 low[LOW ? MT : 1][LOW ? NT : 1];
  if constexpr (LOW)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t) low[i][t] = acc[i][t];

  // transposing reads: lane -> position (4 in a read), channel pair of groups and half unit
  const int j16 = lane >> 4, l16 = lane & 15;
  const int k_pos = (j16 >> 1) * 8 + (l16 >> 2);       // position of the lane's first read; the second is four further on
  const int grp = (j16 & 1) * 2 + ((l16 & 3) >> 1), sub = (l16 & 1) * 8;
  unsigned a_off[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) a_off[i] = (unsigned)((((wm * MT + i) * 4 + grp) * KSP + k_pos) * UB + sub);
  unsigned b_off[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int tile = min(wn * NT + t, pl.ctb * pl.nfy - 1), ct = tile / pl.nfy, fy = tile - ct * pl.nfy;
    b_off[t] = (unsigned)(a_bytes + ((ct * 4 + grp) * VP + pl.by * fy) * UB + sub);
  }

  if (u_lo < u_hi) {
    build_tables(u_lo);
    if (u_lo + 1 < u_hi) build_tables(u_lo + 1);
    __syncthreads();
    issue(u_lo, 0);
  }
  for (int u = u_lo; u < u_hi; ++u) {
    const int b = (u - u_lo) & 1;
    // every wavefront's loads for this stage have landed, and every wavefront is done with the other buffer
    wait_and_barrier<0>();
    const int *vt = tabs + (u % 3) * tab_words + KS + k_pos;
    const unsigned base = lds0 + (unsigned)(b * buf_bytes);
    struct Ops { uintx4 a[MT][PARTS], b[NT][PARTS]; };
    auto fetch = [&](int s, Ops &o) {
      const unsigned v0 = base + (unsigned)vt[16 * s], v1 = base + (unsigned)vt[16 * s + 4];
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int p = 0; p < PARTS; ++p) {
          const unsigned at = base + a_off[i] + (unsigned)(16 * s * UB + p * 16);
          unsigned w0, w1, w2, w3;
          read_transposed(at, w0, w1);
          read_transposed(at + 4 * UB, w2, w3);
          o.a[i][p] = uintx4{w0, w1, w2, w3};
        }
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int p = 0; p < PARTS; ++p) {
          unsigned w0, w1, w2, w3;
          read_transposed(v0 + b_off[t] + p * 16, w0, w1);
          read_transposed(v1 + b_off[t] + p * 16, w2, w3);
          o.b[t][p] = uintx4{w0, w1, w2, w3};
        }
    };
    auto multiply = [&](const Ops &o) {
      if constexpr (LOW) block_multiply_low<MT, NT>(acc, low, o.a, o.b);
      else block_multiply<MT, NT, PARTS>(acc, o.a, o.b);
    };
    Ops o0, o1;
    fetch(0, o0);                                      // (on its way while the next stage's loads are issued)
    __builtin_amdgcn_sched_barrier(0);
    if (u + 1 < u_hi) issue(u + 1, b ^ 1);
#pragma unroll
    for (int s = 0; s < KS / 16; s += 2) {
      fetch(s + 1, o1);
      __builtin_amdgcn_sched_barrier(0);
      multiply(o0);
      __builtin_amdgcn_sched_barrier(0);
      if (s + 2 < KS / 16) fetch(s + 2, o0);
      __builtin_amdgcn_sched_barrier(0);
      multiply(o1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (u + 2 < u_hi) build_tables(u + 2);
  }

  if constexpr (LOW)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[i][t] += low[i][t];
  // ---- the partial block: [channel of the block][column tile (input channels, filter column)][32]
  const int l32 = lane & 31, half = lane >> 5;
  const int cols = pl.ctb * pl.nfy * 32;
  float *out = ws + ((i64)(pl.row[fx].slice0 + slice) * blocks + block) * (i64)(WM * MT * 32) * cols;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int tile = wn * NT + t;
    if (tile < pl.ctb * pl.nfy) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          out[(i64)((wm * MT + i) * 32 + (r >> 2) * 8 + half * 4 + (r & 3)) * cols + tile * 32 + l32] = acc[i][t][r];
    }
  }
#undef pl
}

template <int MT, int NT, int NW, bool F16>
hipError_t launch_wgrad_instance(const BlockWgradPlan &pl, const void *a, const void *g, float *ws, hipStream_t stream) {
  auto kern = block_wgrad_kernel<MT, NT, NW, F16>;
  static std::atomic<int> lds_allowed{0};
  hipError_t e = allow_large_lds((const void *)kern, pl.lds_bytes, lds_allowed);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)(pl.slices * pl.m_blocks * pl.c_blocks)), dim3(NW * 64), pl.lds_bytes, stream,
                     pl, (const char *)a, (const char *)g, ws);
  return hipGetLastError();
}

}  // namespace

bool make_block_wgrad_plan(const SepConv &fwd, bool f16, BlockWgradPlan &pl) {
  const Axis &X = fwd.x, &Y = fwd.y;
  const i64 lim = (i64)1 << 30;
  if (X.nf < 1 || Y.nf < 1 || X.nf > kBlockFilterRows || X.kind > AX_LCORR || X.kind == AX_MCONV || Y.kind != AX_LCORR) return false;
  const i64 plane = X.ng * Y.ng, Q = X.nh * Y.nh;
  if (fwd.batch < 1 || fwd.c_in < 1 || fwd.c_out < 1 || plane < 1 || Q < 1 || plane >= (i64)1 << 22 || Q >= (i64)1 << 22) return false;
  if (X.s > 4096 || X.d > 4096 || X.u > 4096 || X.p > 4096 || X.p < -lim || Y.s > 64 || Y.d > 4096 || Y.u > 64 || Y.p > lim || Y.p < -lim)
    return false;
  // 32-bit source offsets over whole tensors
  if (blocked_bytes(fwd.batch, fwd.c_in, plane, f16) >= ((size_t)1 << 32) || blocked_bytes(fwd.batch, fwd.c_out, Q, f16) >= ((size_t)1 << 32))
    return false;
  if (fwd.batch * Q >= (i64)1 << 31 || fwd.batch * X.nh >= (i64)1 << 21) return false;
  auto magic = [](i64 d) { return d <= 1 ? 0xFFFFFFFFu : (unsigned)(0x100000000ull / (unsigned)d); };
  const int parts = f16 ? 1 : 3, UB = 16 * parts, KS = f16 ? 64 : 32;
  pl.f16 = f16;
  pl.batch = (int)fwd.batch; pl.M = (int)fwd.c_out; pl.C = (int)fwd.c_in;
  pl.MG = (pl.M + 7) / 8; pl.CG = (pl.C + 7) / 8;
  pl.q_out = (int)Q; pl.plane = (int)plane; pl.noy = (int)Y.nh; pl.ngy = (int)Y.ng;
  i64 fy_lo = 0, fy_hi = Y.nf - 1;
  if (Y.u == 1) {
    const i64 span = Y.s * (Y.nh - 1), lo = -floor_div(-(Y.p - span), Y.d), hi = floor_div(Y.ng - 1 + Y.p, Y.d);
    if (std::max<i64>(lo, 0) <= std::min<i64>(hi, Y.nf - 1)) { fy_lo = std::max<i64>(lo, 0); fy_hi = std::min<i64>(hi, Y.nf - 1); }
  }
  pl.nfx = (int)X.nf; pl.nfy = (int)(fy_hi - fy_lo + 1); pl.f_pitch = (int)Y.nf; pl.f_off = (int)fy_lo;
  pl.mg_noy = magic(pl.noy);
  pl.ay = (int)Y.s; pl.by = (int)Y.d; pl.cy = (int)-(Y.p - Y.d * fy_lo); pl.uy = (int)Y.u;
  const i64 span = (i64)pl.by * (pl.nfy - 1);
  if (span > 64) return false;
  pl.by_span = (int)span;
  // rows of each filter row: output rows ox0, ox0 + step, ... with input rows gx0, gx0 + gstep, ...
  i64 work = 0;
  auto gcd = [](i64 a, i64 b) { while (b) { const i64 t = a % b; a = b; b = t; } return a; };
  for (i64 f = 0; f < X.nf; ++f) {
    BlockWgradRow &r = pl.row[f];
    i64 step, lo = 0, hi = X.nh - 1, num0, numk, den, off;       // input row = (num0 + numk ox) / den - off
    if (X.kind == AX_MCORR) { numk = f + X.d; num0 = X.s * numk; den = X.p + 1; off = X.u; }
    else { numk = X.s; num0 = X.d * f - X.p; den = X.u; off = 0; }
    step = den / gcd(numk, den);
    // first row with an exact division, then the first whose input row is not before 0 and the last not past the end
    i64 first = -1;
    for (i64 o = 0; o < step && o <= hi; ++o)
      if (((num0 + numk * o) % den + den) % den == 0) { first = o; break; }
    r = BlockWgradRow{0, 1, 0, 0, 0, 0, 0, 0};
    if (first < 0) continue;
    const i64 need_lo = off * den - num0, need_hi = (X.ng - 1 + off) * den - num0;   // numk ox in [need_lo, need_hi]
    lo = std::max<i64>(lo, -floor_div(-need_lo, numk));
    hi = std::min<i64>(hi, floor_div(need_hi, numk));
    if (lo > first) first += (lo - first + step - 1) / step * step;
    if (first > hi) continue;
    r.ox0 = (int)first; r.step = (int)step; r.count = (int)((hi - first) / step + 1);
    r.gx0 = (int)((num0 + numk * first) / den - off);
    r.gstep = (int)(numk * step / den);
    r.mg_count = magic(r.count);
    work += (i64)r.count * pl.noy * pl.batch;
  }
  if (work == 0) return false;
  // Block shape: wavefronts side by side along the output channels (wm) and along the column tiles, MT x NT tiles each.
  // What counts: the share of the tiles that are of use, and how often a fetched operand is (MT NT / (MT + NT)).
  const int ct_all = (pl.C + 31) / 32, mt_all = (pl.M + 31) / 32;
  const i64 R = (KS - 1 + pl.noy - 1) / pl.noy + 1;
  const i64 vu = std::max<i64>(pl.ay * (KS - 1) + span + 1, pl.ay * (KS - R) + R * (span + 1));
  const i64 vp = ((vu + span + 1 - 4 + 7) / 8) * 8 + 4;
  double best = 0;
  for (int nw = 4; nw <= 8; nw *= 2)
    for (int mt = 1; mt <= 2; ++mt)
      for (int wm = 1; wm <= nw; wm *= 2)
        for (int ctb = 1; ctb <= ct_all; ++ctb) {
          const int wn = nw / wm, tiles = ctb * pl.nfy, nt = (tiles + wn - 1) / wn;
          if (nt > (f16 || mt == 1 ? 4 : 3)) break;    // (fp32: registers)
          if (KS + vp > nw * 64) break;
          const i64 bytes = 2 * UB * ((i64)wm * mt * 4 * (KS + 4) + (i64)ctb * 4 * vp) + 12 * (2 * KS + vp);
          if (bytes > (nw == 4 ? 79 : 158) * 1024) continue;
          const int m_blocks = (mt_all + wm * mt - 1) / (wm * mt), c_blocks = (ct_all + ctb - 1) / ctb;
          const double use = (double)mt_all / (m_blocks * wm * mt) * (double)ct_all / (c_blocks * ctb) * (double)tiles / (nt * wn);
          // (eight wavefronts at one barrier have nothing to hide its wait behind)
          const double score = (nw == 4 ? 1.0 : 0.9) * use * (0.4 + (double)(mt * nt) / (mt + nt));
          if (score > best) {
            best = score;
            pl.nw = nw; pl.mt = mt; pl.wm = wm; pl.ctb = ctb; pl.nt = nt;
            pl.m_blocks = m_blocks; pl.c_blocks = c_blocks;
            pl.VP = (int)vp; pl.zero_unit = (int)vu;
            pl.lds_bytes = (size_t)bytes;
          }
        }
  if (best == 0) return false;
  pl.mgt = pl.wm * pl.mt * 4;
  pl.cgt = pl.ctb * 4;
  // slices: what a CU's registers and LDS hold of workgroups, dealt to the filter rows by their positions.  Small tiles have
  // a few hundred cycles of products a stage, and more than two workgroups to hide the rest behind: 32 -> 32 channels, 4 x 4
  // taps, 32 x 780 x 41, two workgroups and four: fp32 202 -> 147 us, half 111 -> 79 (their sums' launch 27 and 13 us either
  // way) -- as long as a slice has eight stages.  Twice as many, half as long, where a single accumulator takes all six
  // products of fp32 parts (128 -> 256 channels, 3 x 3 taps, 32 x 256 x 41 positions: error 2.9e-6 -> 2.1e-6, wgrad_pos.hip
  // 2.6e-6; its sums' launch 22 -> 28 us, 0.2 % of the step)
  const int blocks = pl.m_blocks * pl.c_blocks, turns = !f16 && pl.mt * pl.nt > kLowTiles ? 2 : 1;
  const int resident = std::min<int>(waves_per_simd(pl.mt, pl.nt, f16) * 4 / pl.nw, (int)(160 * 1024 / pl.lds_bytes));
  i64 want = 256 * resident * turns / blocks;
  if (resident > 2) want = std::max<i64>(512 / blocks, std::min<i64>(want, work / KS / 8));
  want = std::max<i64>(pl.nfx, want);
  int total = 0;
  for (int f = 0; f < pl.nfx; ++f) {
    const i64 k = (i64)pl.row[f].count * pl.noy * pl.batch, units = (k + KS - 1) / KS;
    pl.row[f].slice0 = total;
    pl.row[f].slices = (int)std::min<i64>(units, k ? std::max<i64>(1, want * k / work) : 0);
    total += pl.row[f].slices;
  }
  pl.slices = total;
  pl.ws_bytes = (size_t)total * blocks * (pl.wm * pl.mt * 32) * (size_t)(pl.ctb * pl.nfy * 32) * 4;
  return pl.ws_bytes <= ((size_t)1 << 30);
}

hipError_t launch_block_wgrad(const BlockWgradPlan &pl, const void *grad_out, const void *input, float *workspace,
                              hipStream_t stream) {
  hipError_t e = hipErrorInvalidValue;
#define MELLIN_BW_CASE(MT_, NT_)                                                                    \
  if (pl.mt == MT_ && pl.nt == NT_) {                                                               \
    if (pl.f16) {                                                                                   \
      e = pl.nw == 4 ? launch_wgrad_instance<MT_, NT_, 4, true>(pl, grad_out, input, workspace, stream)   \
                     : launch_wgrad_instance<MT_, NT_, 8, true>(pl, grad_out, input, workspace, stream);  \
    } else if constexpr (MT_ * NT_ < 8) {                                                           \
      e = pl.nw == 4 ? launch_wgrad_instance<MT_, NT_, 4, false>(pl, grad_out, input, workspace, stream)  \
                     : launch_wgrad_instance<MT_, NT_, 8, false>(pl, grad_out, input, workspace, stream); \
    }                                                                                               \
  }
  MELLIN_BW_CASE(1, 1)
  MELLIN_BW_CASE(1, 2)
  MELLIN_BW_CASE(1, 3)
  MELLIN_BW_CASE(1, 4)
  MELLIN_BW_CASE(2, 1)
  MELLIN_BW_CASE(2, 2)
  MELLIN_BW_CASE(2, 3)
  MELLIN_BW_CASE(2, 4)
#undef MELLIN_BW_CASE
  return e;
}

}  // namespace mellin
