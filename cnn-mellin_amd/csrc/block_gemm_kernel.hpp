// Forward pass and gather-form input gradient of layers with many channels, from the
// channel-blocked signal (block_gemm.hpp) on the bf16 / f16 matrix cores.
//
//   H[n, m, ox, oy] = bias[m] + sum_{fx, fy, c} F[m, c, fx, fy] * G[n, c, tap_x(ox, fx), tap_y(oy, fy)]
//
// The contracted index of a matrix instruction runs over CHANNELS of one tap (two groups of
// eight), so an operand of the signal is 16 consecutive bytes of one position: one LDS read per
// register quadruple, nothing to gather, pack or cut in the loop.  What bounded the kernel that
// reads the tensors as they lie (tile_gemm.hip: eight LDS reads and 44 vector instructions per
// 16 taps and 32 positions; matrix pipe 8-19 % busy on half tensors, 39-47 % on fp32) is paid
// once per element in block_pack.hip instead of once per tap and tile of output channels.
//
// Tile: P = WN * NT * 32 consecutive output positions of one image x MT * 32 output channels.
// A stage is F filter rows x G channel groups.  Its signal rows are copied by direct
// global->LDS loads (16 bytes per lane, any source) into virtual rows as in tile_gemm.hip:
//   Mellin axis   virtual row (filter row of the stage, output row): the row of that tap;
//   linear axis   virtual row = coordinate ax ox + bx fx + cx, all filter rows in one stage;
// positions without a source read the blocked tensor's unit of zeros, so nothing is cleared and
// a buffer needs no memory of what it held.  The sources of a tile's virtual positions are worked
// out once per tile into an LDS table.  While a stage multiplies, the next one's loads are issued
// a few at a time between the steps.  Filter fragments come from L1 / L2 straight to registers,
// two or four steps ahead: the WN wavefronts of a workgroup use the same ones at the same time.
//
// Mellin axes: output rows are taken in the order of the residue classes of the axis, so the rows
// of a tile have taps for the same filter rows and only those are staged and multiplied; filter
// rows none of whose taps lies inside the signal for the tile's rows are left out as well.
//
// Input gradients of small images on Mellin axes (JOINT): a tile's positions run over the images of an output row, whose rows
// have taps for the same filter rows; its virtual rows are those of (output row, image) pairs.
//
// Few tiles (one utterance, deep layers): WK = 4 wavefronts share the positions of a tile and
// take every fourth step of a stage; their sums are added in wavefront order through LDS.
//
// Measured against the kernels that read the tensors as they lie, 128 -> 256 channels, 3 x 3 taps, 32 x 256 x 41 positions
// (0.194 TFLOP): fp32, linear, forward and input gradient 1308 -> 905 us each (1075 with tiles of 64 channels x 256 positions
// instead of 128 x 128: make_block_plan) and 206 us a tensor for the cut (six bf16 products: 1.28 PF, at the 1.7 to 2.0 GHz
// the board's power leaves, where a plain bf16 product of 8192^3 reaches 1.34 PF); half, Mellin rows, forward 259 -> 181 us, input gradient 420 -> 181, and 71 us a tensor.
// One utterance (few tiles, WK = 4): 1039 -> 228 us for ten layers.
#pragma once

#include <type_traits>

#include "block_gemm.hpp"
#include "tile_stage.hpp"

namespace mellin {

namespace {

// What a launch makes of its sums: the tensor as it lies, or blocked (block_gemm.hpp) for the kernels that read it
// next; an output [relu](bias + sum), or a gradient, which passes the ReLU in front of the layer (where its blocked
// output `mask` is positive) and whose sums over the positions, the bias gradient of the layer before, go to `chan_sums`.
// Where pairs of neighbouring columns are pooled behind the layer, an output is stored as their maxima (OUT_POOLED; `which`:
// one byte a value, 1 where the second was the larger), and the gradient of such maxima as that of the values they were taken
// from (GRAD_POOLED): the unpooled output is never written, nor the gradient of the maxima.  (Passes of their own, 64
// channels, 32 x 780 x 41, moved 0.6 and 0.7 GB in fp32: 125 and 190 us; half 32 and 51 us.)
enum { OUT_PLAIN, OUT_BLOCKED, GRAD_PLAIN, GRAD_BLOCKED, OUT_POOLED, GRAD_POOLED };

// The plan stays in the kernel arguments and is read by scalar loads where it is used: held in
// registers for a whole stage its fields would not fit the scalar register file.
typedef const __attribute__((address_space(4))) BlockPlan ConstBlockPlan;

struct BlockTile {
  int n, q0, count, row_lo, rows;  // (rows of a joint tile: the (output row, image) pairs that it has positions of)
  int id;                          // the tile
  int c_first, c_end, slot, slice; // its channel groups; in slices: place in the workspace, which slice (whole tiles: -1, 0)
  int vx_min, vrows, units;        // linear axes: first coordinate; virtual rows and positions of the whole tile
  unsigned long long filter_rows;  // Mellin axes: the filter rows with a tap for some row of the tile, four bits each
  int nv;                          // how many
  int G, at_stage, group_bytes;    // channel groups of its stages, their place in the plan's table, LDS bytes of one
};

__device__ __forceinline__ int filter_row(const BlockTile &g, int j) { return (int)(g.filter_rows >> (4 * j)) & 15; }

// Item `id` of the launch: the images of a position tile lie side by side, so that the position tiles
// with the most filter rows come first for all images and every workgroup gets its share of them.
// `rows`: the output rows in the order of their classes, with their filter rows (Mellin axes).
template <int P, int PARTS, bool JOINT>
__device__ __forceinline__ BlockTile block_tile(ConstBlockPlan &pl, const int2 *__restrict__ rows, int id, bool mellin_x) {
  BlockTile g;
  g.c_first = 0;
  g.c_end = pl.CG;
  g.slot = -1;
  g.slice = 0;
  if (id >= pl.whole) {
    const int i = id - pl.whole, r = i / pl.slices, stages = pl.CG / pl.G;
    g.slice = i - r * pl.slices;
    g.slot = g.slice * pl.rest + r;
    g.c_first = g.slice * stages / pl.slices * pl.G;
    g.c_end = (g.slice + 1) * stages / pl.slices * pl.G;
    id = pl.whole + r;
  }
  g.id = id;
  const int qt = JOINT ? id : udiv(id, pl.batch, pl.mg_batch);
  g.n = JOINT ? 0 : id - qt * pl.batch;
  g.q0 = qt * P;
  g.count = min(P, (JOINT ? pl.tile_q : pl.Q) - g.q0);
  g.row_lo = udiv(g.q0, pl.noy, pl.mg_noy);
  g.rows = udiv(g.q0 + g.count - 1, pl.noy, pl.mg_noy) - g.row_lo + 1;
  g.vx_min = pl.ax * g.row_lo + pl.cx + pl.bx_min;
  g.filter_rows = 0;
  if (mellin_x) {
    int mask = 0;
    for (int r = (int)threadIdx.x & 63; r < g.rows; r += 64) {
      const int at = g.row_lo + r;
      mask |= rows[JOINT ? udiv(at, pl.batch, pl.mg_batch) : at].y;
    }
    g.nv = 0;
    for (int f = 0; f < pl.nfx; ++f)
      if (__ballot(mask >> f & 1)) g.filter_rows |= (unsigned long long)f << (4 * g.nv++);
    g.nv = max(g.nv, 1);                             // (no tap at all: a stage of zeros)
    g.vrows = g.nv * g.rows;
  } else {
    g.nv = pl.nfx;
    g.vrows = pl.ax * (g.rows - 1) + pl.bx_span + 1;
  }
  g.units = g.vrows * pl.RS;
  g.at_stage = (g.slot < 0 ? min(g.nv, pl.F) : pl.F) - 1;
  g.G = pl.stage[g.at_stage].G;
  g.group_bytes = mellin_x ? (min(g.nv, pl.F) * g.rows * pl.RS * PARTS + 63) >> 6 << 10 : pl.group_bytes;
  return g;
}

typedef unsigned uintx2 __attribute__((ext_vector_type(2)));

// Sums of sixteen values over the 32 lanes of each half of a wavefront: lane 16 a + 8 b + 4 c + 2 d + e of a half gets the
// sum of value 8 a + 4 b + 2 c + d (halves of the values exchanged at each step: 38 additions instead of 80).
__device__ __forceinline__ float lane_sums(const float (&v)[16], int lane) {
  auto other = [](float x, int step) {
    const int i = __float_as_int(x);
    return __int_as_float(step == 8 ? __builtin_amdgcn_mov_dpp(i, 0x128, 0xf, 0xf, true)        // lane + 8 of sixteen
                        : step == 4 ? __builtin_amdgcn_mov_dpp(i, 0x141, 0xf, 0xf, true)        // 7 - lane of eight
                        : step == 2 ? __builtin_amdgcn_mov_dpp(i, 0x4e, 0xf, 0xf, true) : __builtin_amdgcn_mov_dpp(i, 0xb1, 0xf, 0xf, true));
  };
  float a[8], b[4], c[2];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const bool up = lane & 16;
    const float keep = up ? v[i + 8] : v[i], send = up ? v[i] : v[i + 8];
    a[i] = keep + __shfl_xor(send, 16);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bool up = lane & 8;
    const float keep = up ? a[i + 4] : a[i], send = up ? a[i] : a[i + 4];
    b[i] = keep + other(send, 8);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const bool up = lane & 4;
    const float keep = up ? b[i + 2] : b[i], send = up ? b[i] : b[i + 2];
    c[i] = keep + other(send, 4);
  }
  const bool up = lane & 2;
  const float keep = up ? c[1] : c[0], send = up ? c[0] : c[1];
  const float d = keep + other(send, 2);
  return d + other(d, 1);
}

// A value, and a buffer descriptor of `bytes` at `base`, that are the same in every lane.  Said here: the compiler takes what
// comes from a tile's fields for values of a lane, and then repeats every store for each descriptor that it finds among the
// lanes (a dozen more instructions a store; 33 -> 67 channels, 5 x 3 taps, 7 x 333 x 37 half values: 39.7 us with that and
// stores of four transposed positions, 23.9 without).
__device__ __forceinline__ int wave_value(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ char *wave_value(const void *p) {
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)(size_t)p), hi = __builtin_amdgcn_readfirstlane((unsigned)((size_t)p >> 32));
  return (char *)((unsigned long long)hi << 32 | lo);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t wave_buffer(const void *base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(wave_value(base), 0, wave_value(bytes), 0x00020000);
}

template <int MT, int NT, int WM, int WK, bool F16, int OUT, bool JOINT>
__global__ __launch_bounds__(kThreads, 2) void block_gemm_kernel(BlockPlan plan_arg, const char *__restrict__ X,
                                                                 const char *__restrict__ AF, const void *__restrict__ bias,
                                                                 void *__restrict__ Hv, float *__restrict__ sums,
                                                                 const char *__restrict__ mask, float *__restrict__ chan_sums,
                                                                 unsigned char *__restrict__ which) {
  constexpr int PARTS = F16 ? 1 : 3, UB = 16 * PARTS;
  constexpr int WN = kWaves / WK / WM, P = WN * NT * 32, M_T = WM * MT * 32;
  // Steps that a filter fragment is requested ahead of its own: two, whose products in fp32 take longer than the trip to L2.  In
  // half they are a sixth, and a wavefront waited for its fragments in every step: four, where wavefronts do not share a tile.
  // 128 -> 128 channels, 4 x 4 taps, 32 x 774 x 7: 85.7 -> 78.3 us (67 where every step takes the same fragment, which then
  // comes out of L1); input gradient of 256 <- 128 on 771 x 5: 154 -> 131; ten linear layers' step 2903 -> 2682.
  constexpr int AD = deep_fragments(F16, WK) ? 4 : 2;
  constexpr int kALoads = AD * MT * PARTS;             // fragment loads of that many steps
  constexpr bool POOLED = OUT == OUT_POOLED, UNPOOLED = OUT == GRAD_POOLED;
  constexpr bool BLOCKED = OUT == OUT_BLOCKED || OUT == GRAD_BLOCKED || POOLED || UNPOOLED, GRAD = OUT == GRAD_PLAIN || OUT == GRAD_BLOCKED || UNPOOLED;
  extern __shared__ __align__(16) char blk_lds[];
  ConstBlockPlan *plp = (ConstBlockPlan *)__builtin_amdgcn_kernarg_segment_ptr();
#define pl (*plp)
  char *bufs = blk_lds;                                                    // [2][buf_bytes]
  float *Bs = (float *)(bufs + 2 * pl.buf_bytes);                          // [M_T]
  int *tab = (int *)(Bs + M_T);                                            // [tab_units] source byte offset in a group's plane
  int2 *ents = (int2 *)(tab + pl.tab_units);                               // [2][ents] (LDS offset, fragment offset) of a step's half
  int *row_src = (int *)(ents + 2 * pl.ents);                              // Mellin axes: [filter row of the tile][row] first source of the row
  const int2 *rows = (const int2 *)(AF + pl.rows_off);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  const int wk = WK > 1 ? wave : 0, wm = WM > 1 ? wave & (WM - 1) : 0, wn = WK > 1 ? 0 : wave / WM;
  const bool mellin_x = JOINT || pl.kind_x == AX_MCORR || pl.kind_x == AX_MCONV;
  const int taps = pl.nfx * pl.nfy;
  const int items = pl.whole + pl.rest * pl.slices;
  // Wavefronts that share a tile, 2, 4 or 8 tiles of channels: XCD k (workgroups k, k + 8, ...) takes one of those, and its
  // share of the filter is all that the XCD's L2 sees: one utterance of a Mellin stack, layers of 128 to 256 channels on 337 x
  // 10 and 337 x 5, 16.9, 17.9, 26.2 and 36.2 us -> 15.9, 16.8, 24.5 and 35.3.  (Filters below 1 MB: nothing gained;
  // 41 -> 128 channels on one axis 84.2 -> 86.0 us a step.  Other numbers of tiles do not divide the XCDs evenly: of three
  // the slowest would have two XCDs for a third of the work, 1.3 times an even share, of five, six and seven one for a fifth,
  // a sixth and a seventh, 1.6, 1.3 and 1.1 times.)  The position tiles are dealt to a tile of channels' XCDs in turn: those of a
  // class with many filter rows follow each other, and an eighth of all tiles without a gap left XCDs waiting (113 us).
  int m_tile = blockIdx.y, item = blockIdx.x;
  if constexpr (WK > 1)
    if (gridDim.y != (unsigned)pl.m_tiles) {
      const int xcd = item & 7, each = 8 / pl.m_tiles;
      m_tile = xcd / each;
      item = (item >> 3) * each + xcd - m_tile * each;
      if (item >= items) return;
    }
  const unsigned zero_frag = (unsigned)(pl.CG * taps * PARTS * 512);       // the tile's fragment of zeros, behind the others
  const unsigned af_tile = zero_frag + PARTS * 512;                        // bytes of 32 channels' fragments
  const char *AFm = AF + (i64)(m_tile * WM + wm) * MT * af_tile, *AFm1 = AFm + af_tile;
  const i64 plane_bytes = (i64)(pl.plane + 1) * UB;
  const unsigned lds0 = lds_address((const float *)blk_lds);
  const int my_tiles = WK > 1 ? 1 : (items - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;

  if (tid < M_T) {
    const int m = m_tile * M_T + tid;
    float b = 0.f;
    if (bias && m < pl.M) b = !F16 ? ((const float *)bias)[m] : (float)(pl.wide ? (_Float16)((const float *)bias)[m] : ((const _Float16 *)bias)[m]);
    Bs[tid] = b;
  }

  // the sources of a tile's virtual positions, and the operand offsets of its steps
  constexpr int kWrap = (AD == 4 ? 10 : 4) * WK;       // halves of the steps that a stage reads on, of every wavefront that shares a tile's
  auto stage_halves = [](int n) { return max((n + 2 * WK - 1) / (2 * WK) * (2 * WK), 2 * AD * WK); };
  auto build_tile = [&](const BlockTile &g, int parity, int2 *before) {
    // (fields of the plan, read together: one wait for the scalar loads instead of one each)
    int RS = pl.RS, cy = pl.cy + pl.by_min, uy = pl.uy, ux = pl.ux, ngx = pl.ngx, ngy = pl.ngy, tab_units = pl.tab_units, F = pl.F,
        G = g.G, nfx = pl.nfx, nfy = pl.nfy, none = pl.plane, group_bytes = g.group_bytes, n_before = pl.ents;
    asm volatile("" : "+s"(RS), "+s"(cy), "+s"(uy), "+s"(ux), "+s"(ngx), "+s"(ngy), "+s"(tab_units), "+s"(F), "+s"(G), "+s"(nfx),
                 "+s"(nfy), "+s"(none), "+s"(group_bytes), "+s"(n_before));
    int kx = pl.kind_x, sx = pl.sx, dx = pl.dx, px = pl.px, bx = pl.bx, bx_min = pl.bx_min, by = pl.by, by_min = pl.by_min;
    unsigned mg_p1 = pl.mg_p1, mg_full = pl.mg_full, mg_per_row = pl.stage[g.at_stage].mg_per_row, mg_G = pl.stage[g.at_stage].mg_G;
    asm volatile("" : "+s"(kx), "+s"(sx), "+s"(dx), "+s"(px), "+s"(bx), "+s"(bx_min), "+s"(by), "+s"(by_min), "+s"(mg_p1),
                 "+s"(mg_full), "+s"(mg_per_row), "+s"(mg_G));
    if (mellin_x) {
      const FastDiv by_rows(g.rows);
      for (int t = tid; t < g.nv * g.rows; t += kThreads) {
        int j, r, from = 0;
        by_rows.divmod(t, j, r);
        r += g.row_lo;
        if (JOINT) {
          const int pair = r;
          r = udiv(pair, pl.batch, pl.mg_batch);
          from = (pair - r * pl.batch) * pl.CG * (none + 1);               // the image's units
        }
        const int gx = mellin_tap32(kx, rows[r].x, filter_row(g, j), ngx, sx, dx, px + 1, ux, mg_p1);
        row_src[t] = gx >= 0 ? from + gx * ngy : -1;
      }
      lds_barrier();
    }
    // wavefronts take 64 / RS virtual rows (or a 64th piece of one) at a time: a lane keeps its column
    const int per = RS <= 64 ? 64 / RS : 1, vrows = g.vrows;
    const int lr = RS <= 64 ? lane / RS : 0;
    for (int col = lane - lr * RS; col < RS; col += RS <= 64 ? RS : 64) {
      const int vy = cy + col;
      int gy = -1;
      if (vy >= 0) {
        if (uy == 1) gy = vy;
        else { const int q = vy / uy; if (q * uy == vy) gy = q; }
        if (gy >= ngy) gy = -1;
      }
      if (lr < per)
        for (int vr = wave * per + lr; vr < vrows; vr += kWaves * per) {
          int first = -1;
          if (mellin_x) {
            first = row_src[vr];
          } else {
            const int vx = g.vx_min + vr;
            int gx = -1;
            if (vx >= 0) {
              if (ux == 1) gx = vx;
              else { const int q = vx / ux; if (q * ux == vx) gx = q; }
            }
            if (gx >= 0 && gx < ngx) first = gx * ngy;
          }
          tab[vr * RS + col] = (first >= 0 && gy >= 0 ? first + gy : none) * UB;
        }
    }
    if (tid < 64 && g.units + tid < tab_units) tab[g.units + tid] = none * UB;
    // Entries of the tile's stages one behind the other (a last odd half is paired with the fragment of zeros), then
    // the first steps again: a stage reads on into the one that follows it.  `before`: the first steps of
    // this tile also go behind the entries of the tile before it, whose last stage is running.
    int2 *out = ents + parity * n_before;
    const int per_row = nfy * G, full = stage_halves(F * per_row), subsets = (g.nv + F - 1) / F;
    const int tail = stage_halves((g.nv - (subsets - 1) * F) * per_row), n_ents = (subsets - 1) * full + tail;
    for (int e = tid; e < n_ents + kWrap; e += kThreads) {
      int at0 = e < n_ents ? e : e - n_ents;
      if (AD == 4 && at0 >= n_ents) at0 -= n_ents;                       // (a stage has AD steps or more)
      const int sub = min(udiv(at0, full, mg_full), subsets - 1), at = at0 - sub * full;
      const int n_e = min(F, g.nv - sub * F) * per_row, k = min(at, n_e - 1);
      const int jj = udiv(k, per_row, mg_per_row), rest = k - jj * per_row, fy = udiv(rest, G, mg_G), gi = rest - fy * G;
      const int fx = mellin_x ? filter_row(g, sub * F + jj) : jj;
      const int row = mellin_x ? jj * g.rows : bx * fx - bx_min;
      const int2 v = make_int2(gi * group_bytes + (row * RS + by * fy - by_min) * UB,
                               at < n_e ? ((gi * nfx + fx) * nfy + fy) * (PARTS * 512) : 0x40000000);
      out[e] = v;
      if (e < kWrap && before) before[e] = v;
    }
    return n_ents;
  };

  // the loads of a stage: 16-byte slots in blocks of 64, dealt to the wavefronts; the sources of four blocks are read
  // before the first is used
  auto issue = [&](const BlockTile &g, int c0, int j0, int buf) {
    const int nF = min(pl.F, g.nv - j0);
    const int units = mellin_x ? nF * g.rows * pl.RS : g.units, blocks = (units * PARTS + 63) >> 6;
    const int *from = tab + (mellin_x ? j0 * g.rows * pl.RS : 0);
    const char *src0 = X + ((i64)g.n * pl.CG + c0) * plane_bytes;
    const unsigned dst0 = lds0 + (unsigned)(buf * pl.buf_bytes);
    int groups = g.G, group_bytes = g.group_bytes;
    asm volatile("" : "+s"(groups), "+s"(group_bytes));      // (kept in registers: a scalar load in the loop would wait for LDS as well)
    for (int b = wave; b < blocks; b += 4 * kWaves) {
      unsigned at[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int slot = min(b + i * kWaves, blocks - 1) * 64 + lane, unit = F16 ? slot : slot / 3;
        at[i] = (unsigned)from[unit] + (F16 ? 0 : (slot - unit * 3) * 16);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (b + i * kWaves < blocks) {
          const char *src = src0;
          unsigned dst = dst0 + (unsigned)((b + i * kWaves) * 1024);
          for (int k = 0; k < groups; ++k) {
            load16_to_lds_at((const float *)src, at[i], dst);
            src += plane_bytes;
            dst += (unsigned)group_bytes;
          }
        }
    }
  };

  floatx16 acc[MT][NT];
  // fp32: sums of their own for the small products (of the largest tiles they take the last registers).  Error against 64
  // bits of 64 -> 128 channels, 5 x 3 taps, in the 2-norm: output 4.1e-7 -> 1.4e-7, input gradient 4.3e-7 -> 1.6e-7; time of
  // a ten-layer stack's step 13.57 -> 13.58 ms.
  constexpr bool LOW = !F16;
  floatx16 low[LOW ? MT : 1][LOW ? NT : 1];
  int lane_vpos[NT], lane_q[NT];
  struct Operands { uintx4 a[MT][PARTS]; };
  struct SignalOps { uintx4 b[NT][PARTS]; };
  Operands A0, A1, A2, A3;                             // (AD == 2: A0, A1)
  SignalOps B0, B1;

  const unsigned lane_frag = (unsigned)(l32 * 16), zero_at = zero_frag + lane_frag;
  auto fetch_a = [&](const int2 &e, unsigned af_c, Operands &o) {
    const unsigned off = min((unsigned)e.y + af_c + lane_frag, zero_at);
#pragma unroll
    for (int k = 0; k < MT; ++k)
#pragma unroll
      for (int pt = 0; pt < PARTS; ++pt) o.a[k][pt] = *(const uintx4 *)((k ? AFm1 : AFm) + off + pt * 512);
  };

  BlockTile tg = block_tile<P, PARTS, JOINT>(pl, rows, item, mellin_x), next_tg = tg;
  if (my_tiles <= 0) return;
  int n_ents = build_tile(tg, 0, nullptr), next_ents = n_ents;
  __syncthreads();
  issue(tg, tg.c_first, 0, 0);
  int c0 = tg.c_first, j0 = 0, buf = 0, ti = 0;
  int se = 0;                                          // the stage's first entry (of this tile's)
  unsigned af_c = (unsigned)(c0 * taps * PARTS * 512);
  const int2 *my_ents = ents + 2 * wk + half;          // this half-wave's entries (of parity 0)
  int2 e0 = my_ents[0], e1 = my_ents[2 * WK];
  fetch_a(e0, af_c, A0);
  fetch_a(e1, af_c, A1);
  if constexpr (AD == 4) {
    fetch_a(my_ents[4], af_c, A2);
    fetch_a(my_ents[6], af_c, A3);
  }
  wait_and_barrier<0>();

  for (bool first = true;;) {
    {
      unsigned zero;                                   // a zero the compiler cannot see through: plan fields are loaded anew per stage
      asm volatile("s_mov_b32 %0, 0" : "=s"(zero));
      plp = (ConstBlockPlan *)((const __attribute__((address_space(4))) char *)__builtin_amdgcn_kernarg_segment_ptr() + zero);
    }
    if (first) {
      if constexpr (LOW)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) low[i][t][r] = 0.f;
      // position -> virtual position of its (first filter row, first column) tap; accumulators start from the bias
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        int local = (wn * NT + t) * 32 + l32;
        if (local >= tg.count) local = 0;
        const int row = udiv(tg.q0 + local, pl.noy, pl.mg_noy), oy = tg.q0 + local - row * pl.noy;
        lane_vpos[t] = (((mellin_x ? 1 : pl.ax) * (row - tg.row_lo)) * pl.RS + pl.ay * oy) * UB;
        lane_q[t] = (mellin_x ? rows[JOINT ? udiv(row, pl.batch, pl.mg_batch) : row].x : row) * pl.noy + oy;
      }
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          float4 bv = *(const float4 *)(Bs + (wm * MT + i) * 32 + g4 * 8 + half * 4);
          if ((WK > 1 && wk > 0) || tg.slice > 0) bv = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            acc[i][t][4 * g4 + 0] = bv.x; acc[i][t][4 * g4 + 1] = bv.y;
            acc[i][t][4 * g4 + 2] = bv.z; acc[i][t][4 * g4 + 3] = bv.w;
          }
        }
    }
    const char *Xb = bufs + buf * pl.buf_bytes;
    auto fetch_b = [&](const int2 &e, SignalOps &o) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int pt = 0; pt < PARTS; ++pt) o.b[t][pt] = *(const uintx4 *)(Xb + (lane_vpos[t] + e.x) + pt * 16);
    };
    fetch_b(e0, B0);
    // ---- the stage after this one: its loads are issued under this stage's steps, its first fragments in the last two
    const int halves = stage_halves((mellin_x ? min(pl.F, tg.nv - j0) : tg.nv) * pl.nfy * tg.G);
    const int steps = halves / (2 * WK);
    int nj0 = mellin_x ? j0 + pl.F : tg.nv, nc0 = c0, n_se = se + halves;
    if (nj0 >= tg.nv) { nj0 = 0; nc0 = c0 + tg.G; n_se = 0; }
    const bool last = nc0 >= tg.c_end;
    const bool more = !last || ti + 1 < my_tiles;
    const int2 *ep = my_ents + (ti & 1) * pl.ents + se;
    if (last) {
      nc0 = 0;
      nj0 = 0;
      if (more) {
        // another tile: its tables (every load of this tile has been issued, every wavefront is past the barrier)
        next_tg = block_tile<P, PARTS, JOINT>(pl, rows, (int)blockIdx.x + (ti + 1) * (int)gridDim.x, mellin_x);
        next_ents = build_tile(next_tg, (ti + 1) & 1, ents + (ti & 1) * pl.ents + n_ents);
        lds_barrier();
        nc0 = next_tg.c_first;
        issue(next_tg, nc0, 0, buf ^ 1);
      }
    } else {
      issue(tg, nc0, nj0, buf ^ 1);
    }
    const unsigned n_af = (unsigned)(nc0 * taps * PARTS * 512);
    // A step: the next step's signal operands are requested before its multiplies and the fragments of the step
    // AD further on behind them (pinned: the scheduler moves reads next to their use).  Nothing here depends on which
    // step it is, so that every wait counts exactly what is younger: the last pair's last signal reads are of no use,
    // and its fragment fetches are the next stage's.
    auto multiply = [&](const Operands &a, const SignalOps &b) {
      if constexpr (LOW) block_multiply_low<MT, NT>(acc, low, a.a, b.b);
      else block_multiply<MT, NT, PARTS>(acc, a.a, b.b);
    };
    if constexpr (AD == 4) {
      // (entries: e1 of the step after this one, ahead the offset of the fragments that are requested next)
      unsigned ahead = (unsigned)ep[8].y;
      e1 = ep[2];
      int at = 0;
      auto step = [&](Operands &a, const SignalOps &b, SignalOps &next) {
        fetch_b(e1, next);
        e0 = e1;
        e1.x = ep[4].x;
        const unsigned further = (unsigned)ep[10].y;
        __builtin_amdgcn_sched_barrier(0);
        multiply(a, b);
        __builtin_amdgcn_sched_barrier(0);
        fetch_a(make_int2(0, (int)ahead), at + 4 < steps ? af_c : n_af, a);
        ahead = further;
        ep += 2;
        ++at;
      };
      while (at + 3 < steps) {
        step(A0, B0, B1);
        step(A1, B1, B0);
        step(A2, B0, B1);
        step(A3, B1, B0);
      }
      // (the fragments of the next stage's first steps move to their places)
      if (steps & 2) {
        step(A0, B0, B1);
        step(A1, B1, B0);
        const Operands a0 = A0, a1 = A1;
        A0 = A2; A1 = A3; A2 = a0; A3 = a1;
      }
      if (steps & 1) {
        step(A0, B0, B1);
        const Operands a0 = A0;
        A0 = A1; A1 = A2; A2 = A3; A3 = a0;
      }
    } else {
      int2 e2 = ep[4 * WK];
      for (int i = 0; i + 1 < steps; i += 2) {
        fetch_b(e1, B1);
        const int2 e3 = ep[6 * WK];
        __builtin_amdgcn_sched_barrier(0);
        multiply(A0, B0);
        __builtin_amdgcn_sched_barrier(0);
        fetch_a(e2, i + 2 < steps ? af_c : n_af, A0);
        fetch_b(e2, B0);
        const int2 e4 = ep[8 * WK];
        __builtin_amdgcn_sched_barrier(0);
        multiply(A1, B1);
        __builtin_amdgcn_sched_barrier(0);
        fetch_a(e3, i + 3 < steps ? af_c : n_af, A1);
        e0 = e2;
        e1 = e3;
        e2 = e4;
        ep += 4 * WK;
      }
      if (steps & 1) {
        // one step left, whose operands are in A0 and B0; A1 holds the next stage's first fragments where its second's belong
        multiply(A0, B0);
        e0 = e1;
        e1 = e2;
        fetch_a(e0, n_af, A0);
        fetch_a(e1, n_af, A1);
      }
    }
    // every wavefront's loads for the next stage have landed (the newest in flight are the fragments of AD steps),
    // and every wavefront is done with this stage's buffer
    wait_and_barrier<kALoads>();
    first = last;
    if (last) {
      // ---- the tile is finished
      if constexpr (LOW)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            acc[i][t] += low[i][t];
            asm volatile("" : "+v"(acc[i][t]));        // (here, not next to their uses: `low` ends here)
          }
      if constexpr (WK > 1) {
        // sums of the wavefronts, in their order (one tile per workgroup: the buffers are free)
        float *red = (float *)bufs;
#pragma unroll
        for (int k = 0; k < MT; ++k)
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
              *(float4 *)(red + (((wk * MT * NT + k * NT + t) * 4 + r4) * 64 + lane) * 4) =
                  make_float4(acc[k][t][4 * r4], acc[k][t][4 * r4 + 1], acc[k][t][4 * r4 + 2], acc[k][t][4 * r4 + 3]);
        __syncthreads();
      }
      const bool whole = tg.slot < 0, relu = pl.relu && whole;
      const int m0 = m_tile * M_T + wm * MT * 32;
      // A gradient's mask, and the sums of its channels over the tile's positions
      const unsigned unit_row = (unsigned)(pl.out_q + 1) * UB;              // bytes of a channel group of a blocked output
      const unsigned mask_row = UNPOOLED ? (unsigned)(pl.Q + 1) * UB : unit_row;
      const i64 image_bytes = (i64)pl.out_groups * unit_row, mask_bytes = (i64)pl.out_groups * mask_row;
      // joint: the images of the lane's positions
      int lane_n[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        lane_n[t] = 0;
        if constexpr (JOINT) {
          const int local = (wn * NT + t) * 32 + l32, pair = udiv(tg.q0 + (local < tg.count ? local : 0), pl.noy, pl.mg_noy);
          lane_n[t] = pair - udiv(pair, pl.batch, pl.mg_batch) * pl.batch;
        }
      }
      const int images = JOINT ? pl.batch : 1, all_images = (int)image_bytes * images;
      __amdgpu_buffer_rsrc_t mask_rsrc, which_rsrc;
      if constexpr (GRAD) mask_rsrc = wave_buffer(mask + tg.n * mask_bytes, (int)mask_bytes * images);
      const int which_row = 8 * (POOLED ? pl.out_q : pl.Q), which_bytes = pl.out_groups * which_row;
      if constexpr (POOLED || UNPOOLED) which_rsrc = wave_buffer(which + (i64)tg.n * which_bytes, which ? which_bytes * images : 0);
      // the lane's quarter unit in its group, in the output and in the mask (none: past any end)
      int unit_at[NT], mask_at[NT];
      const bool odd_cols = UNPOOLED && (pl.out_cols & 1);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const bool there = (wn * NT + t) * 32 + l32 < tg.count;
        int unit = lane_q[t];
        if constexpr (POOLED) unit >>= 1;              // (an even number of columns)
        if constexpr (UNPOOLED) unit = 2 * unit + (odd_cols ? udiv(unit, pl.noy, pl.mg_noy) : 0);
        unit_at[t] = there ? lane_n[t] * (int)image_bytes + unit * UB + half * 8 : (int)0x80000000u;
        mask_at[t] = !UNPOOLED ? unit_at[t] : there ? lane_n[t] * (int)mask_bytes + lane_q[t] * UB + half * 8 : (int)0x80000000u;
      }
      auto load_mask = [&](int group, int at) -> uintx2 {
        return __builtin_amdgcn_raw_buffer_load_b64(mask_rsrc, at < 0 ? at : at + (int)(group * mask_row), 0, 0);   // (none: zeros)
      };
      // GRAD_POOLED: the four bytes of a lane's quarter unit as masks over its values, for the pair's second value
      auto load_which = [&](int group, int t) -> unsigned {
        const int at = lane_n[t] * which_bytes + lane_q[t] * 8 + half * 4 + group * which_row;
        return __builtin_amdgcn_raw_buffer_load_b32(which_rsrc, mask_at[t] < 0 ? mask_at[t] : at, 0, 0);
      };
      auto second_mask = [](unsigned w) {
        const unsigned bytes = (w << 8) - w;           // 0 or 255 each
        return uintx2{__builtin_amdgcn_perm(0, bytes, 0x01010000), __builtin_amdgcn_perm(0, bytes, 0x03030202)};
      };
      // the unit behind a row's last pair where there is an odd column, which took no part: zeros
      auto odd_at = [&](int t, int to) { return to >= 0 && lane_q[t] - udiv(lane_q[t], pl.noy, pl.mg_noy) * pl.noy == pl.noy - 1 ? to + 2 * UB : (int)0x80000000u; };
      // OUT_POOLED: of two values a lane, the pair's that the lane keeps -- with its neighbour, an even lane that of the first,
      // an odd lane that of the second -- and whether its second value is the larger
      auto pool = [&](float a, float b, bool &second) {
        if constexpr (F16) { a = (float)(_Float16)a; b = (float)(_Float16)b; }         // (the stored values are compared)
        const bool odd = lane & 1;
        const float keep = odd ? b : a, send = odd ? a : b;
        const float got = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(send), 0xb1, 0xf, 0xf, true));
        const float one = odd ? got : keep, two = odd ? keep : got;
        second = two > one;                            // (behind a ReLU: no NaN)
        return second ? two : one;
      };
      auto pool4 = [&](const float4 &a, const float4 &b, unsigned &seconds) {
        bool s0, s1, s2, s3;
        const float4 v = make_float4(pool(a.x, b.x, s0), pool(a.y, b.y, s1), pool(a.z, b.z, s2), pool(a.w, b.w, s3));
        seconds = (s0 ? 1u : 0u) | (s1 ? 0x100u : 0u) | (s2 ? 0x10000u : 0u) | (s3 ? 0x1000000u : 0u);
        return v;
      };
      auto masked = [&](float4 v, uintx2 x) {
        auto keep = [](float f, unsigned sixteen) { return (short)sixteen > 0 ? f : 0.f; };
        return make_float4(keep(v.x, x[0]), keep(v.y, x[0] >> 16), keep(v.z, x[1]), keep(v.w, x[1] >> 16));
      };
      auto put_sums = [&](const float (&s)[16], int k, int slot) {
        const float total = lane_sums(s, lane);
        const int r = (lane >> 1) & 15, m = m0 + k * 32 + (r >> 2) * 8 + half * 4 + (r & 3);
        if (!(lane & 1) && m < pl.M) chan_sums[(i64)m * pl.chan_slots + slot] = total;
      };
      const int first_slot = (tg.id * (WK > 1 ? NT : WN));

      // ---- stores of the tensor as it lies.  The descriptor ends with the block's last channel, so rows past it and
      // lanes without a position (an offset past any end) are dropped by its range check.  A slice's sums are fp32, in
      // the order of the tile.
      const bool as_half = F16 && !BLOCKED && whole;
      const int ES = as_half ? 2 : 4, h_m = wave_value((whole ? (int)pl.h_m : P) * ES);
      char *const base = wave_value(whole ? (char *)Hv + ((i64)tg.n * pl.h_n + (i64)m0 * (int)pl.h_m) * ES
                                          : (char *)(sums + (((i64)tg.slot * pl.m_tiles + m_tile) * M_T + wm * MT * 32) * P));
      const int base_bytes = wave_value(max(0, min(MT * 32, pl.M - m0)) * h_m + (whole && JOINT ? (pl.batch - 1) * (int)pl.h_n * ES : 0));
      const __amdgpu_buffer_rsrc_t rsrc = BLOCKED && whole ? wave_buffer((char *)Hv + tg.n * image_bytes, all_images) : wave_buffer(base, base_bytes);
      int at[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int local = (wn * NT + t) * 32 + l32;
        at[t] = local < tg.count ? (whole ? lane_n[t] * (int)pl.h_n + lane_q[t] : local) * ES : (int)0x80000000u;
      }
      auto store_one = [&](float v, int to) {
        if (as_half) __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(short, (_Float16)v), rsrc, to, 0, 0);
        else __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rsrc, to, 0, 0);
      };
      auto relu4 = [&](float4 v) { return !GRAD && relu ? make_float4(fmaxf(v.x, 0.f), fmaxf(v.y, 0.f), fmaxf(v.z, 0.f), fmaxf(v.w, 0.f)) : v; };
      auto store_four = [&](float4 v, int to) {        // four channels of the lane's position
        store_one(v.x, to);
        store_one(v.y, to + h_m);
        store_one(v.z, to + 2 * h_m);
        store_one(v.w, to + 3 * h_m);
      };
      const int row0 = half * 4 * h_m;
      if constexpr (WK > 1) {
        // the tile's 32 x 32 blocks are dealt to the wavefronts
        const float *red = (const float *)bufs;
        for (int kt = wk; kt < MT * NT; kt += WK) {
          const int k = kt / NT, t = kt - k * NT;
          const int unit = NT > 1 && t ? unit_at[NT - 1] : unit_at[0], m_at = NT > 1 && t ? mask_at[NT - 1] : mask_at[0];
          int to = (NT > 1 && t ? at[NT - 1] : at[0]) + row0 + k * 32 * h_m;
          float s[16];
#pragma unroll
          for (int r4 = 0; r4 < 4; ++r4) {
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int w = 0; w < WK; ++w) {
              const float4 p = *(const float4 *)(red + (((w * MT * NT + kt) * 4 + r4) * 64 + lane) * 4);
              v.x += p.x; v.y += p.y; v.z += p.z; v.w += p.w;
            }
            v = relu4(v);
            const int group = m0 / 8 + k * 4 + r4;
            if constexpr (GRAD) {
              if (whole) {
                v = masked(v, load_mask(group, m_at));
                s[4 * r4] = v.x; s[4 * r4 + 1] = v.y; s[4 * r4 + 2] = v.z; s[4 * r4 + 3] = v.w;
              }
            }
            if (BLOCKED && whole) {
              unsigned w[PARTS][2], seconds = 0;
              if constexpr (POOLED) v = pool4(v, v, seconds);
              cut_four<F16>(v, w);
              const int o = unit < 0 || (POOLED && (lane & 1)) ? (int)0x80000000u : unit + (int)(group * unit_row);
              if constexpr (POOLED) __builtin_amdgcn_raw_buffer_store_b32(seconds, which_rsrc, o < 0 ? o : group * which_row + (unit - half * 8) / (2 * PARTS) + half * 4, 0, 0);
              uintx2 m2 = {0, 0};
              if constexpr (UNPOOLED) m2 = second_mask(load_which(group, NT > 1 && t ? NT - 1 : 0));
#pragma unroll
              for (int pt = 0; pt < PARTS; ++pt) {
                const uintx2 x = {w[pt][0], w[pt][1]};
                __builtin_amdgcn_raw_buffer_store_b64(x & ~m2, rsrc, o < 0 ? o : o + pt * 16, 0, 0);
                if constexpr (UNPOOLED) __builtin_amdgcn_raw_buffer_store_b64(x & m2, rsrc, o < 0 ? o : o + UB + pt * 16, 0, 0);
              }
              if (odd_cols) {
                const int z = odd_at(NT > 1 && t ? NT - 1 : 0, o);
#pragma unroll
                for (int pt = 0; pt < PARTS; ++pt) __builtin_amdgcn_raw_buffer_store_b64(uintx2{0, 0}, rsrc, z < 0 ? z : z + pt * 16, 0, 0);
              }
            } else {
              store_four(v, to);
            }
            to += 8 * h_m;                             // (registers 4 g .. 4 g + 3 are rows 8 g + 4 half ..)
          }
          if constexpr (GRAD)
            if (whole) put_sums(s, k, first_slot + t);
        }
      } else {
        if constexpr (GRAD) {
          if (whole) {
            // The masks of kAhead groups of channels are requested before the first is used, in registers that are free
            // here (fp32: of `low`; half: of the signal's operands); read where they were used, each of the tile's 16 or
            // 32 waits took a trip to memory: 28000 of 90000 cycles of a tile of 64 x 512 half values.
            constexpr int kGroups = MT * 4, kAhead = F16 ? (8 / NT < kGroups ? 8 / NT : kGroups) : kGroups;
            uintx2 mask_of[kAhead][NT];
            auto request = [&](int i) {
#pragma unroll
              for (int t = 0; t < NT; ++t) mask_of[i % kAhead][t] = load_mask(m0 / 8 + i, mask_at[t]);
            };
#pragma unroll
            for (int i = 0; i < kAhead; ++i) request(i);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < MT; ++k) {
              float s[16];
#pragma unroll
              for (int g4 = 0; g4 < 4; ++g4) {
                float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                  const float4 v = masked(make_float4(acc[k][t][4 * g4], acc[k][t][4 * g4 + 1], acc[k][t][4 * g4 + 2], acc[k][t][4 * g4 + 3]),
                                          mask_of[(k * 4 + g4) % kAhead][t]);
                  acc[k][t][4 * g4] = v.x; acc[k][t][4 * g4 + 1] = v.y; acc[k][t][4 * g4 + 2] = v.z; acc[k][t][4 * g4 + 3] = v.w;
                  sum.x += v.x; sum.y += v.y; sum.z += v.z; sum.w += v.w;
                }
                s[4 * g4] = sum.x; s[4 * g4 + 1] = sum.y; s[4 * g4 + 2] = sum.z; s[4 * g4 + 3] = sum.w;
                if (k * 4 + g4 + kAhead < kGroups) request(k * 4 + g4 + kAhead);
              }
              put_sums(s, k, first_slot + wn);
            }
          }
        }
        if constexpr (!GRAD)
          if (relu)
#pragma unroll
            for (int k = 0; k < MT; ++k)
#pragma unroll
              for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[k][t][r] = fmaxf(acc[k][t][r], 0.f);
        // Tensors as they lie, and slices: a value at a time, 32 positions of a channel side by side.  (Four positions a lane,
        // by transposes over four lanes, are a quarter of the stores but no fewer bytes or lines: stores alone, 64 channels x
        // 256 positions a workgroup, fp32 18.7 us in singles and 20.7 in fours, half 13.0 and 26.8 where channels have an odd
        // number of positions.)
        auto store_all = [&](auto store) {
#pragma unroll
          for (int k = 0; k < MT; ++k)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const int row = k * 32 + (r >> 2) * 8 + (r & 3);                   // (and four further on in the upper half)
              const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc(base + row * h_m, 0, max(0, base_bytes - row * h_m), 0x00020000);
#pragma unroll
              for (int t = 0; t < NT; ++t) store(acc[k][t][r], to, at[t] + row0);
            }
        };
        if (BLOCKED && whole) {
          // the halves of a wavefront exchange quarters, so that a lane stores whole units: the lower one groups 0 and 2
          // of a tile's four, the upper one groups 1 and 3
          // (pooled: of two blocks of 32 positions the even lanes store the maxima of one, the odd lanes those of the other)
          constexpr int NS = POOLED ? (NT + 1) / 2 : NT;
          int to[NS], which_at[NS];
#pragma unroll
          for (int t = 0; t < NS; ++t) {
            const bool odd = lane & 1;
            int u = POOLED ? (odd ? (2 * t + 1 < NT ? unit_at[POOLED && 2 * t + 1 < NT ? 2 * t + 1 : 0] : (int)0x80000000u) : unit_at[POOLED ? 2 * t : 0]) : unit_at[t];
            to[t] = u < 0 ? u : u - half * 8 + (int)((m0 / 8 + half) * unit_row);
            which_at[t] = u < 0 ? u : (u - half * 8) / (2 * PARTS) + (m0 / 8 + half) * which_row;
          }
#pragma unroll
          for (int k = 0; k < MT; ++k) {
            unsigned seconds_of[UNPOOLED ? 4 : 1][UNPOOLED ? NT : 1];
            if constexpr (UNPOOLED) {
#pragma unroll
              for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int t = 0; t < NT; ++t) seconds_of[i][t] = load_which(m0 / 8 + k * 4 + i, t);
              __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int p2 = 0; p2 < 4; p2 += 2) {
#pragma unroll
              for (int t = 0; t < NS; ++t) {
                unsigned lo[PARTS][2], hi[PARTS][2], lo2 = 0, hi2 = 0;
                auto four = [&](int tile, int r) { return make_float4(acc[k][tile][r], acc[k][tile][r + 1], acc[k][tile][r + 2], acc[k][tile][r + 3]); };
                if constexpr (POOLED) {
                  const int other = 2 * t + 1 < NT ? 2 * t + 1 : 2 * t;
                  cut_four<F16>(pool4(four(2 * t, 4 * p2), four(other, 4 * p2), lo2), lo);
                  cut_four<F16>(pool4(four(2 * t, 4 * p2 + 4), four(other, 4 * p2 + 4), hi2), hi);
                  const auto s2 = __builtin_amdgcn_permlane32_swap(lo2, hi2, false, false);
                  __builtin_amdgcn_raw_buffer_store_b64(uintx2{s2[0], s2[1]}, which_rsrc, which_at[t], 0, 0);
                  if (which_at[t] >= 0) which_at[t] += 2 * which_row;
                } else {
                  cut_four<F16>(four(t, 4 * p2), lo);
                  cut_four<F16>(four(t, 4 * p2 + 4), hi);
                }
                uintx2 lo_m = {0, 0}, hi_m = {0, 0};
                if constexpr (UNPOOLED) { lo_m = second_mask(seconds_of[p2][t]); hi_m = second_mask(seconds_of[p2 + 1][t]); }
                auto put = [&](int pt, uintx2 a, uintx2 b, int o) {
                  const auto s0 = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);
                  const auto s1 = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
                  __builtin_amdgcn_raw_buffer_store_b128(uintx4{s0[0], s1[0], s0[1], s1[1]}, rsrc, o < 0 ? o : o + pt * 16, 0, 0);
                };
#pragma unroll
                for (int pt = 0; pt < PARTS; ++pt) {
                  const uintx2 a = {lo[pt][0], lo[pt][1]}, b = {hi[pt][0], hi[pt][1]};
                  put(pt, a & ~lo_m, b & ~hi_m, to[t]);
                  if constexpr (UNPOOLED) put(pt, a & lo_m, b & hi_m, to[t] < 0 ? to[t] : to[t] + UB);
                }
                if (odd_cols) {
                  const int z = odd_at(t, to[t]);
#pragma unroll
                  for (int pt = 0; pt < PARTS; ++pt) __builtin_amdgcn_raw_buffer_store_b128(uintx4{0, 0, 0, 0}, rsrc, z < 0 ? z : z + pt * 16, 0, 0);
                }
                if (to[t] >= 0) to[t] += (int)(2 * unit_row);
                __builtin_amdgcn_sched_barrier(0);     // (one block's registers at a time)
              }
            }
          }
        } else if (as_half) {
          store_all([](float v, const __amdgpu_buffer_rsrc_t &to, int at) {
            __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(short, (_Float16)v), to, at, 0, 0);
          });
        } else {
          store_all([](float v, const __amdgpu_buffer_rsrc_t &to, int at) { __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), to, at, 0, 0); });
        }
      }
      if constexpr (BLOCKED)
        if constexpr (JOINT) {
          // the units of zeros behind the images, which are dealt to the tiles
          const int tiles = max(pl.whole, 1), lo = (int)((i64)tg.id * pl.batch / tiles), hi = whole ? (int)((i64)(tg.id + 1) * pl.batch / tiles) : lo;
          for (int i = tid; i < (hi - lo) * (M_T / 8); i += kThreads) {
            const int n = lo + i / (M_T / 8), group = m_tile * (M_T / 8) + i % (M_T / 8);
            uintx4 *z = (uintx4 *)((char *)Hv + n * image_bytes + (i64)group * unit_row + (i64)pl.out_q * UB);
            const uintx4 zero = {0, 0, 0, 0};
#pragma unroll
            for (int pt = 0; pt < PARTS; ++pt) z[pt] = zero;
          }
        } else if (whole && tg.q0 + tg.count == pl.Q && tid < M_T / 8 && m_tile * (M_T / 8) + tid < pl.out_groups) {
          // the units of zeros behind an image's last positions
          uintx4 *z = (uintx4 *)((char *)Hv + tg.n * image_bytes + (i64)(m_tile * (M_T / 8) + tid) * unit_row + (i64)pl.out_q * UB);
          const uintx4 zero = {0, 0, 0, 0};
#pragma unroll
          for (int pt = 0; pt < PARTS; ++pt) z[pt] = zero;
        }
      if (!more) break;
      ++ti;
      tg = next_tg;
      n_ents = next_ents;
    }
    c0 = nc0;
    j0 = nj0;
    buf ^= 1;
    se = n_se;
    af_c = n_af;
  }
#undef pl
}

template <int MT, int NT, int WM, int WK, bool F16, int OUT, bool JOINT>
hipError_t launch_joint(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream) {
  auto kern = block_gemm_kernel<MT, NT, WM, WK, F16, OUT, JOINT>;
  static std::atomic<int> lds_allowed{0};
  hipError_t e = allow_large_lds((const void *)kern, pl.lds_bytes, lds_allowed);
  if (e != hipSuccess) return e;
  dim3 grid((unsigned)pl.grid_x, (unsigned)pl.m_tiles);
  if (WK > 1 && (pl.m_tiles == 2 || pl.m_tiles == 4 || pl.m_tiles == 8) && pl.filter_bytes >= (size_t)1 << 20)   // by XCD: see the kernel
    grid = dim3((unsigned)((pl.grid_x + 8 / pl.m_tiles - 1) / (8 / pl.m_tiles) * 8));
  hipLaunchKernelGGL(kern, grid, dim3(kThreads), pl.lds_bytes, stream, pl,
                     (const char *)a.signal, (const char *)a.frag, a.bias, a.out, a.sums, (const char *)a.mask, a.chan_sums, (unsigned char *)a.which);
  return hipGetLastError();
}

template <int MT, int NT, int WM, int WK, bool F16, int OUT>
hipError_t launch_instance(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream) {
  if constexpr (OUT != OUT_POOLED)                     // (no joint tiles of those: make_block_plan)
    if (pl.joint) return launch_joint<MT, NT, WM, WK, F16, OUT, true>(pl, a, stream);
  return launch_joint<MT, NT, WM, WK, F16, OUT, false>(pl, a, stream);
}

template <int OUT>
hipError_t launch_shape(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream) {
#define MELLIN_BLOCK_CASE(MT_, NT_, WM_, WK_)                                                                \
  if (pl.mt == MT_ && pl.nt == NT_ && pl.wm == WM_ && pl.wk == WK_) {                                        \
    if (pl.f16) return launch_instance<MT_, NT_, WM_, WK_, true, OUT>(pl, a, stream);                        \
    return launch_instance<MT_, NT_, WM_, WK_, false, OUT>(pl, a, stream);                                   \
  }
  if (pl.f16 && pl.nt == 4) {
    if (pl.wm == 2) return launch_instance<2, 4, 2, 1, true, OUT>(pl, a, stream);
    if (pl.mt == 2) return launch_instance<2, 4, 1, 1, true, OUT>(pl, a, stream);
    return launch_instance<1, 4, 1, 1, true, OUT>(pl, a, stream);
  }
  if (pl.f16 && pl.nt == 2 && pl.wk == 4)
    return pl.mt == 2 ? launch_instance<2, 2, 1, 4, true, OUT>(pl, a, stream) : launch_instance<1, 2, 1, 4, true, OUT>(pl, a, stream);
  if (!pl.f16 && pl.wm == 2)
    return pl.mt == 2 ? launch_instance<2, 2, 2, 1, false, OUT>(pl, a, stream) : launch_instance<1, 2, 2, 1, false, OUT>(pl, a, stream);
  if (pl.f16 && pl.mt == 2 && pl.nt == 1 && pl.wk == 1) return launch_instance<2, 1, 1, 1, true, OUT>(pl, a, stream);
  MELLIN_BLOCK_CASE(2, 2, 1, 1)
  MELLIN_BLOCK_CASE(1, 2, 1, 1)
  MELLIN_BLOCK_CASE(1, 1, 1, 1)
  MELLIN_BLOCK_CASE(2, 1, 1, 4)
  MELLIN_BLOCK_CASE(1, 1, 1, 4)
#undef MELLIN_BLOCK_CASE
  return hipErrorInvalidValue;
}

}  // namespace

}  // namespace mellin
