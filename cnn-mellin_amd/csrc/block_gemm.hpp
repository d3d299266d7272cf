// Channel-blocked forms of a layer's passes, for layers with many channels: operands are first
// laid out with eight channels of a position side by side (16 bytes: what a lane feeds one matrix
// instruction), cut into their bf16 parts once per element, and the matrix kernels then read
// ready-made operands (block_pack.hip, block_gemm.hip, block_wgrad.hip).
#pragma once

#include "mellin_common.hpp"

namespace mellin {

constexpr int kBlockClasses = 32;                  // residue classes of a Mellin axis a plan can hold
constexpr int kBlockFilterRows = 16;

// A blocked tensor of `channels` channels and `plane` positions per image:
//   [image][group of eight channels][plane + 1][part][8 channels]
// with three bf16 parts (fp32 tensors) or one f16 part (half tensors); channels past the last are
// zeros, and so is the unit past the plane's last position (the source of padding).
inline size_t blocked_bytes(i64 batch, i64 channels, i64 plane, bool f16) {
  return (size_t)batch * (size_t)((channels + 7) / 8) * (size_t)(plane + 1) * (f16 ? 16 : 48);
}

// A class of output rows: every `stride`-th row from `first` on, with the filter rows of `mask`.
struct BlockClass { int first, start; unsigned mask; };     // start: the class's first row in the order of the classes

// Channel groups to a stage (see BlockPlan::stage), and what divides by them and by a filter row's halves of steps (udiv).
struct BlockStage { int G; unsigned mg_G, mg_per_row; };

struct BlockPlan {
  int f16;
  int wide;                        // f16: filter and bias are float (rounded to half where they are read)
  int batch, M, CG;                // images, output channels, groups of eight contracted channels
  int nfx, nfy;                    // filter rows; filter columns (those that have taps)
  int nox, noy, Q;                 // output extent
  int ngx, ngy, plane;             // signal extent
  // x axis.  Mellin kinds: tap_index(); linear kinds: (ax ox + bx fx + cx) / ux
  int kind_x, sx, dx, px, ux, ax, bx, cx, bx_min, bx_span;
  unsigned mg_p1;                  // floor(2^32 / (px + 1)) (see udiv)
  int ay, by, cy, uy, by_min;      // y axis: (ay oy + by fy + cy) / uy
  int RS;                          // units per virtual row
  int F, G;                        // filter rows and channel groups of a stage
  BlockStage stage[kBlockFilterRows];                        // of a whole tile with one, two, .. F (and more) filter rows
  int tab_units;                   // positions of a tile's source table
  int ents;                        // operand offsets of a tile's steps
  int group_bytes, buf_bytes;      // LDS of one group of a stage, of a stage
  // tiles: (position tile, image), the images of a position tile side by side.  The last `rest` of them, which would
  // leave workgroups without one, are dealt out in `slices` of the contracted channels, whose sums go to the workspace
  int whole, rest, slices;
  int out_groups, chan_slots;      // groups of eight output channels; partial sums of a channel over the positions
  int pool, out_q, out_cols;       // pairs of columns: 1 stored as their maxima, 2 a gradient of such; positions and columns of what is stored
  unsigned mg_batch, mg_noy, mg_full;      // floor(2^32 / d) (see udiv)
  i64 h_n, h_m;
  int relu, half_out;
  int n_classes, cls_stride;
  BlockClass cls[kBlockClasses];
  // filter (block_pack.hip)
  i64 f_m, f_c;
  int f_pitch, f_off;
  // launch
  int mt, nt, wm, wk, m_tiles, grid_x;
  size_t lds_bytes;
  size_t rows_off, filter_bytes;   // the packed filter: fragments, then (Mellin axes) the output rows in the order of their classes
  size_t slice_bytes;              // workspace of the slices' sums
  // `joint`: a tile's positions run over the images of an output row (row, image, column), not over the rows of an image;
  // tile_batch and tile_q: images that are numbered apart (1) and positions that tiles are cut from (all there are), else
  // batch and Q
  int joint, tile_batch, tile_q;
};

// Whether the kernel requests filter fragments four steps ahead and not two (see there); a stage then has four steps or more.
constexpr bool deep_fragments(bool f16, int wk) { return f16 && wk == 1; }

// Frequency pooling behind the layer: a forward pass of an even number of columns (`pr` leaves an odd last one out) stores the
// maxima of pairs of them; an input gradient of `pr`, whose output is that of the maxima, is stored as that of the `cols`
// columns they were taken from (an odd last one of them: zeros).
struct BlockPool { int kind, cols; };  // kind: 0 no pooling, 1 forward, 2 input gradient

// False: the kernel does not apply.  gradient: of an input (a forward pass has no joint tiles).  `like`, for a pooled forward pass
// without an odd last column: the plan of the same layer without the pooling, whose order of sums is kept (false as well where
// that cannot be).
bool make_block_plan(const SepConv &pr, bool f16, bool gradient, const BlockPool &pool, const BlockPlan *like, BlockPlan &pl);
// A plan without pooling as that of the same pass beside it (a forward pass: of an even number of columns): tiles and sums are
// the same.  False: the tensor in front of the pooling is too large for it.
bool pool_block_plan(const BlockPool &pool, BlockPlan &pl);
// out = [relu](bias + sum) from a blocked signal and packed filter; bias (fp32 / half, or null), relu as the plan says.
// With `grad`, the input gradient of a layer behind a ReLU: zero where `mask`, the blocked output of that ReLU, is not
// positive; its sums over the positions go to chan_sums ([channel][pl.chan_slots]: partial sums for launch_block_finish).
// Of tiles in slices (pl.rest > 0) the sums go to `sums`, and launch_block_finish does all that.
struct BlockGemmArgs {
  const void *signal, *frag, *bias;
  void *out;
  float *sums;
  bool blocked, grad;              // out: blocked
  const void *mask;
  float *chan_sums;
  void *which;                     // of pooled pairs, eight bytes a unit: 1 where the second is the larger (forward: null where nobody asks)
};
hipError_t launch_block_gemm(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream);
hipError_t launch_out_blocked(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream);
hipError_t launch_grad_plain(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream);
hipError_t launch_grad_blocked(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream);
hipError_t launch_out_pooled(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream);
hipError_t launch_grad_pooled(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream);

// The rows of one filter row in the weight gradient: output rows ox0 + i step and input rows gx0 + i gstep for
// i < count; its share of the launch: `slices` workgroups from slice0 on.
struct BlockWgradRow { int ox0, step, gx0, gstep, count, slice0, slices; unsigned mg_count; };

struct BlockWgradPlan {
  int f16;
  int batch, M, C, MG, CG;         // images, channels of grad_out and input, their groups of eight
  int q_out, plane, noy, ngy;
  int nfx, nfy, f_pitch, f_off;    // filter columns f_off .. f_off + nfy - 1 have taps
  int ay, by, cy, uy, by_span;     // y axis: (ay oy + by fy + cy) / uy
  int nw, mt, nt, wm, ctb;         // wavefronts, tiles of each, how many lie along the output channels, 32-channel tiles of the input in a block
  int m_blocks, c_blocks, mgt, cgt;
  int VP, zero_unit;               // units of a channel group's input in a stage, the first that is always zero
  int slices;
  unsigned mg_noy;                 // reciprocals, as udiv() takes them
  BlockWgradRow row[kBlockFilterRows];
  size_t lds_bytes, ws_bytes;
};

// `fwd`: the forward pass's problem (x axis Mellin or linear correlation, y linear correlation).
bool make_block_wgrad_plan(const SepConv &fwd, bool f16, BlockWgradPlan &pl);
// Partial blocks of the weight gradient (ws_bytes at `partial`) from blocked tensors.
hipError_t launch_block_wgrad(const BlockWgradPlan &pl, const void *grad_out, const void *input, float *partial,
                              hipStream_t stream);

// A tensor to lay out: x (batch, channels, plane), fp32 or half -> blocked.  With `relu_out` (the layer's output) values
// whose output is not positive are zeros (the backward of the fused ReLU).  With `partial`: per-channel sums of what was
// written, block by block, for launch_block_finish (pack_partial_count(): floats).
struct PackSignal {
  const void *x, *relu_out;
  char *blocked;
  float *partial;
  int batch, channels, plane;
};
size_t pack_partial_count(i64 batch, i64 channels, i64 plane);
// A filter to pack for `pl`, and on Mellin axes the output rows in the order of their classes: f (fp32 or half; wide: fp32
// where the tensors are half) of `channels` contracted channels -> filter_bytes at `frag`.  `copy`: the filter's
// `copy_count` floats, rounded to half.
struct PackFilterHead {
  const void *f;
  char *frag;
  void *copy;
  i64 copy_count, f_m, f_c;
  size_t rows_off;
  int channels, wide, M, CG, nfx, nfy, f_pitch, f_off, tiles;          // (tiles of 32 channels)
  int kind_x, nox, ngx, sx, dx, px, ux;
  unsigned mg_p1;
  int n_classes, cls_stride;
};
struct PackFilter : PackFilterHead { BlockClass cls[kBlockClasses]; };
PackFilter pack_filter(const BlockPlan &pl, int channels, const void *f, void *frag, void *copy, i64 copy_count);
// Everything a pass reads, in one launch (more of them for more filters or classes than a launch's arguments hold): up to two
// tensors (null: not there) and filters.
hipError_t launch_block_pack(bool f16, const PackSignal *a, const PackSignal *b, const PackFilter *filters, int n_filters,
                             hipStream_t stream);

// Maximum over pairs of neighbouring columns of a blocked tensor (batch, channels, rows, cols), as pool_pairs: y is blocked
// with cols / 2 columns; `which` (eight bytes a unit of y): 1 where the second was taken.
hipError_t launch_block_pool(bool f16, const void *x, i64 batch, i64 channels, i64 rows, i64 cols, void *y, void *which, hipStream_t stream);

// The sums that end passes, in one launch.
constexpr int kFinishJobs = 16;
struct WeightSums {                // a weight gradient from its partial blocks
  const float *partial;
  void *grad;
  int M, C, nfx, nfy, f_pitch, f_off, ctb, m_t, m_blocks, c_blocks;    // (m_t: output channels of a block)
  int tap_chunk, parts;            // taps of a block of threads; parts that the slices are added in
  unsigned blocks, zero_blocks;    // blocks of threads; of those for columns without a tap
  unsigned short slice0[kBlockFilterRows], slices[kBlockFilterRows];
};
struct BiasSums {                  // a bias gradient: `count` partial sums of each of `channels`
  const float *partial;
  void *grad;
  i64 count;
  unsigned channels;
};
struct BlockFinish {
  int n_weights, n_biases;
  WeightSums weight[kFinishJobs];
  BiasSums bias[kFinishJobs];
  const BlockPlan *slices;         // what a block_gemm called with `args` made of tiles in slices (null: none)
  BlockGemmArgs args;
  void add_weight(const BlockWgradPlan &pl, const void *partial, void *grad);
  void add_bias(const void *partial, i64 count, i64 channels, void *grad) {
    bias[n_biases++] = BiasSums{(const float *)partial, grad, count, (unsigned)channels};
  }
};
// (wide: the gradients are float where the tensors are half)
hipError_t launch_block_finish(bool f16, bool wide, const BlockFinish &job, hipStream_t stream);

}  // namespace mellin
