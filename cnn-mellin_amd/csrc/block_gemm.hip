// Plans of the channel-blocked matrix kernel (block_gemm_kernel.hpp): tile shape, stages and turns of a launch, and the
// launches that write a layer's output as it lies.  The kernel's other endings are in block_gemm_out.hip and
// block_gemm_grad_*.hip (a translation unit each, for the time they take to compile).
#include <algorithm>
#include <cmath>

#include "block_gemm_kernel.hpp"
#include "tap_runs.hpp"

namespace mellin {

namespace {

// Residue classes of a Mellin axis (mellin_common.hpp: tap relations), those with the same filter
// rows next to each other.
void plan_classes(const Axis &x, BlockPlan &pl) {
  auto gcd = [](i64 a, i64 b) { while (b) { const i64 t = a % b; a = b; b = t; } return a; };
  i64 L = 1;
  if (x.kind == AX_MCORR) L = x.p + 1;
  else if (x.kind == AX_MCONV)
    for (i64 f = 0; f < x.nf && L <= kBlockClasses; ++f) {
      const i64 m = (f + x.d) / gcd(f + x.d, x.p + 1);
      L = L / gcd(L, m) * m;
    }
  pl.n_classes = 1;
  pl.cls_stride = 1;
  pl.cls[0] = BlockClass{0, 0, (1u << x.nf) - 1};
  if (L < 2 || L > kBlockClasses) return;
  struct Item { unsigned mask; int first; } items[kBlockClasses];
  int n = 0;
  for (i64 r = 0; r < L; ++r) {
    const i64 first = ((r - x.s) % L + L) % L;
    if (first >= x.nh) continue;
    unsigned mask = 0;
    for (i64 f = 0; f < x.nf; ++f) {
      const bool has = x.kind == AX_MCORR ? (r * (f + x.d)) % (x.p + 1) == 0 : r % ((f + x.d) / gcd(f + x.d, x.p + 1)) == 0;
      if (has) mask |= 1u << f;
    }
    items[n++] = Item{mask, (int)first};
  }
  std::sort(items, items + n, [](const Item &a, const Item &b) {
    const int ca = __builtin_popcount(a.mask), cb = __builtin_popcount(b.mask);
    return ca != cb ? ca > cb : (a.mask != b.mask ? a.mask < b.mask : a.first < b.first);
  });
  int start = 0;
  for (int i = 0; i < n; ++i) {
    pl.cls[i] = BlockClass{items[i].first, start, items[i].mask};
    start += (int)((x.nh - items[i].first + L - 1) / L);
  }
  pl.n_classes = n;
  pl.cls_stride = (int)L;
}

}  // namespace

bool make_block_plan(const SepConv &pr, bool f16, bool gradient, const BlockPool &pool, const BlockPlan *like, BlockPlan &pl) {
  const Axis &X = pr.x, &Y = pr.y;
  const i64 lim = (i64)1 << 30;
  if (pr.accumulate || pr.batch < 1 || pr.c_out < 1 || pr.c_in < 1 || X.nf < 1 || Y.nf < 1 || X.nf > kBlockFilterRows) return false;
  if (Y.kind != AX_LCORR && Y.kind != AX_LCONV) return false;
  const i64 plane = X.ng * Y.ng, Q = X.nh * Y.nh, out_q = pool.kind == 1 ? Q / 2 : pool.kind == 2 ? X.nh * pool.cols : Q;
  if (pool.kind == 1 && Y.nh % 2) return false;        // (and a gradient's `cols` are 2 nh or 2 nh + 1)
  if (plane < 1 || Q < 1 || plane >= (i64)1 << 22 || Q >= (i64)1 << 22) return false;
  if (pr.batch > 65535 || pr.c_in > 8 * 65535 || pr.c_out * Q >= lim / 2 || Q >= (i64)1 << 20 ||
      (pr.c_out + 7) / 8 * (std::max(Q, out_q) + 1) * 48 >= (i64)1 << 31)
    return false;                                      // (32-bit byte offsets)
  if (X.s > 4096 || X.d > 4096 || X.u > 4096 || X.p > 4096 || X.p < -lim || Y.s > 64 || Y.d > 4096 || Y.u > 64 || Y.p > lim || Y.p < -lim)
    return false;
  pl.f16 = f16;
  pl.wide = 0;
  pl.pool = pool.kind; pl.out_q = (int)out_q; pl.out_cols = pool.cols;
  pl.out_groups = (int)((pr.c_out + 7) / 8);
  pl.batch = (int)pr.batch; pl.M = (int)pr.c_out; pl.CG = (int)((pr.c_in + 7) / 8);
  pl.nox = (int)X.nh; pl.noy = (int)Y.nh; pl.Q = (int)Q;
  pl.ngx = (int)X.ng; pl.ngy = (int)Y.ng; pl.plane = (int)plane;
  pl.h_n = pr.h_n; pl.h_m = pr.h_m; pl.f_m = pr.f_m; pl.f_c = pr.f_c;
  pl.relu = pr.relu; pl.half_out = pr.out_half;
  // filter columns with a tap inside the signal for some output column (the rest meet padding only)
  i64 fy_lo = 0, fy_hi = Y.nf - 1;
  if (Y.u == 1) {
    const i64 span = Y.s * (Y.nh - 1);
    const i64 lo = Y.kind == AX_LCORR ? -floor_div(-(Y.p - span), Y.d) : -floor_div(-(Y.p - (Y.ng - 1)), Y.d);
    const i64 hi = Y.kind == AX_LCORR ? floor_div(Y.ng - 1 + Y.p, Y.d) : floor_div(Y.p + span, Y.d);
    if (std::max<i64>(lo, 0) <= std::min<i64>(hi, Y.nf - 1)) { fy_lo = std::max<i64>(lo, 0); fy_hi = std::min<i64>(hi, Y.nf - 1); }
  }
  pl.nfx = (int)X.nf; pl.nfy = (int)(fy_hi - fy_lo + 1);
  pl.f_pitch = (int)Y.nf; pl.f_off = (int)fy_lo;
  if (pl.nfy > 64) return false;
  // A pooled output's sums keep the order of the unpooled one's, which decides what its ReLU lets through (see can_join), and
  // are those of the layer called by itself bit for bit: the same channel groups and filter columns to a stage, the same
  // slices.  An even number of columns makes the same tiles of them (pool_block_plan; one utterance of a ten-layer Mellin stack,
  // whose wavefronts share tiles: 212 -> 207 us with two of its three poolings inside the products).  An odd last column, as
  // here, is in no tile, so these hold other
  // positions than without the pooling, and the order must not depend on what a tile holds: not on its being one of those in
  // slices, nor, on Mellin axes, on the filter rows of its other output rows -- they shift the pairs that share a step where a
  // row's taps and groups are odd in number, and the steps that wavefronts share.
  if (like && (like->nfy != pl.nfy || like->f_off != pl.f_off || (like->whole && like->rest) ||
               ((X.kind == AX_MCORR || X.kind == AX_MCONV) && (like->wk > 1 || like->nfy * like->G % 2))))
    return false;
  const i64 py = Y.p - Y.d * fy_lo;
  pl.ay = (int)Y.s; pl.by = Y.kind == AX_LCORR ? (int)Y.d : -(int)Y.d; pl.cy = Y.kind == AX_LCORR ? -(int)py : (int)py;
  pl.uy = (int)Y.u;
  const i64 by_ext = (i64)pl.by * (pl.nfy - 1);
  pl.by_min = (int)std::min<i64>(by_ext, 0);
  const i64 RS = (i64)pl.ay * (pl.noy - 1) + (by_ext < 0 ? -by_ext : by_ext) + 1;
  if (RS > 4096) return false;
  pl.RS = (int)RS;
  const bool mellin = X.kind == AX_MCORR || X.kind == AX_MCONV;
  pl.kind_x = X.kind; pl.sx = (int)X.s; pl.dx = (int)X.d; pl.px = (int)X.p; pl.ux = (int)X.u;
  pl.mg_p1 = X.p <= 0 ? 0xFFFFFFFFu : (unsigned)(0x100000000ull / (unsigned)(X.p + 1));
  pl.ax = pl.bx = pl.cx = pl.bx_min = pl.bx_span = 0;
  if (mellin) {
    const i64 hmax = X.nh + X.s, fmax = X.nf + X.d;
    if (hmax * fmax >= lim || (X.p + 1) * hmax >= lim || (X.ng + X.u) * std::max(fmax, X.p + 1) >= lim) return false;
    plan_classes(X, pl);
  } else {
    pl.ax = (int)X.s; pl.bx = X.kind == AX_LCORR ? (int)X.d : -(int)X.d; pl.cx = X.kind == AX_LCORR ? -(int)X.p : (int)X.p;
    const i64 ext = (i64)pl.bx * (pl.nfx - 1);
    pl.bx_min = (int)std::min<i64>(ext, 0);
    pl.bx_span = (int)(ext < 0 ? -ext : ext);
    pl.n_classes = 1; pl.cls_stride = 1; pl.cls[0] = BlockClass{0, 0, 0};
  }
  const int parts = f16 ? 1 : 3;
  pl.mt = pr.c_out > 32 ? 2 : 1;
  pl.wm = 1;

  // Tile shapes: tiles of 32 positions of a wavefront, wavefronts along the channels, wavefronts that share a tile.
  constexpr int kShapes = 7;
  static const int shapes[kShapes][3] = {{4, 2, 1}, {4, 1, 1}, {2, 2, 1}, {2, 1, 1}, {1, 1, 1}, {2, 1, 4}, {1, 1, 4}};
  // A tile shape's stage: the channel groups and filter rows that fit twice into the LDS that a
  // workgroup may take, two workgroups to a CU
  struct Stage { i64 rows; int F, G; };
  Stage stages[2][kShapes] = {};
  int groups[8], n_groups = 0;                         // the channel groups of a stage that divide all, most first
  for (int G = std::min(pl.CG, 8); G >= 1; --G)
    if (pl.CG % G == 0 && (!like || G == like->G)) groups[n_groups++] = G;
  i64 room = 79 * 1024;                                // LDS of a workgroup
  auto shape = [&](int at) {
    const int nt = shapes[at][0], wm = shapes[at][1], wk = shapes[at][2];
    const int P = (kWaves / wk / wm) * nt * 32, M_T = wm * pl.mt * 32;
    const i64 RT = std::min<i64>(pl.joint ? (i64)pl.nox * pl.batch : pl.nox, (P - 1 + pl.noy - 1) / pl.noy + 1);
    const i64 vrows = mellin ? RT : (i64)pl.ax * (RT - 1) + pl.bx_span + 1;
    const i64 tab = ((mellin ? vrows * pl.nfx : vrows) * pl.RS + 64 + 64 + 3) & ~(i64)3;
    const i64 row_src = mellin ? 4 * RT * pl.nfx : 0;
    const bool deep = deep_fragments(f16, wk);
    auto pad = [&](int halves) { return std::max((halves + 2 * wk - 1) & -(2 * wk), (deep ? 8 : 4) * wk); };      // (wk: 1 or 4)
    Stage &st = stages[pl.mt - 1][at];                 // (joint tiles mostly have as many rows as those of an image)
    if (st.rows != RT) {
      st = Stage{RT, 0, 0};
      int best_halves = 0, best_all = 1;               // the best rate so far, as a fraction
      for (int F = mellin ? pl.nfx : 1; F >= 1; --F) {
        const int rows = mellin ? F : pl.nfx, subsets = mellin ? (pl.nfx + F - 1) / F : 1;
        const i64 gb = (vrows * (mellin ? F : 1) * pl.RS * parts + 63) / 64 * 1024, fixed = 4 * tab + row_src + M_T * 4;
        if (2 * gb + fixed > room) continue;
        for (int k = 0; k < n_groups; ++k) {
          const int G = groups[k], halves = rows * pl.nfy * G, all = pad(halves);
          if (2 * gb * G + fixed + 16 * (i64)(subsets * all + (deep ? 12 : 8) * wk) > room) continue;
          // what a stage's steps fill of their whole pairs, against what a stage costs on top (its barrier and first reads)
          if (halves * best_all > best_halves * (all + 2 * wk)) { best_halves = halves; best_all = all + 2 * wk; st.F = F; st.G = G; }
        }
      }
    }
    const int best_f = st.F, best_g = st.G;
    if (!best_f) return false;
    const i64 units = vrows * (mellin ? best_f : 1) * pl.RS;
    pl.F = mellin ? best_f : pl.nfx;
    pl.G = best_g;
    pl.tab_units = (int)tab;
    pl.ents = (mellin ? (pl.nfx + pl.F - 1) / pl.F : 1) * pad(pl.F * pl.nfy * best_g) + (deep ? 12 : 8) * wk;
    pl.group_bytes = (int)((units * parts + 63) / 64 * 1024);
    pl.buf_bytes = pl.group_bytes * best_g;
    pl.nt = nt; pl.wm = wm; pl.wk = wk;
    if ((i64)((pl.tile_q + P - 1) / P) * pl.tile_batch >= (i64)1 << 26) return false;
    if (pl.joint && pl.M % M_T) return false;          // (channels past the last would be the next image's)
    size_t bytes = 2 * (size_t)pl.buf_bytes;
    if (wk > 1) bytes = std::max(bytes, (size_t)wk * pl.mt * nt * 4096);
    if (wk > 1) pl.buf_bytes = (int)(bytes / 2);
    bytes += 4 * (size_t)tab + 16 * (size_t)pl.ents + row_src + M_T * 4;
    pl.lds_bytes = bytes;
    pl.m_tiles = (int)((pr.c_out + M_T - 1) / M_T);
    return bytes <= room;
  };
  auto magic = [](i64 d) { return d <= 1 ? 0xFFFFFFFFu : (unsigned)(0x100000000ull / (unsigned)d); };
  pl.mg_batch = magic(pl.batch); pl.mg_noy = magic(pl.noy);
  auto set_joint = [&](int joint) {
    pl.joint = joint;
    pl.tile_batch = joint ? 1 : pl.batch;
    pl.tile_q = joint ? pl.nox * pl.batch * pl.noy : pl.Q;
  };
  // Mellin axes: which filter rows have a tap inside the signal, for runs of output rows in the order of the classes (axes of
  // more rows, of which a tile's share a class: those of the class)
  static_assert(TapRuns::kFilterRows == kBlockFilterRows, "");
  TapRuns runs;
  const bool masks = mellin && pl.nox <= TapRuns::kRows;
  double class_rows = 0;
  if (mellin) {
    const TapAxis axis = {X.kind == AX_MCORR, pl.nfx, pl.ngx, pl.sx, pl.dx, pl.px + 1, pl.ux};
    for (int k = 0; k < pl.n_classes; ++k) {
      const int end = k + 1 < pl.n_classes ? pl.cls[k + 1].start : pl.nox;
      class_rows += __builtin_popcount(pl.cls[k].mask) * (double)(end - pl.cls[k].start) / pl.nox;
      if (masks) runs.add_class(axis, pl.cls[k].first, pl.cls_stride, end - pl.cls[k].start);
    }
  }
  // What a tile of P positions stages: filter rows, and stages of them, on average.  (Counted over the tile's rows together:
  // with the average of single rows small images of many classes got tiles that stage nearly every filter row; windows of
  // ten frames 1989 -> 1968 us a step, a ten-layer Mellin stack of 24 to 192 channels on two utterances 1175 -> 1117 us.)
  // Tiles of P positions are counted once for all shapes.
  struct Tiles { int joint, of[TapRuns::kFilterRows + 1]; } tiles_by_p[5] = {{-1, {}}, {-1, {}}, {-1, {}}, {-1, {}}, {-1, {}}};
  // (F: filter rows of a stage)
  auto tile_rows = [&](int P, int F, double &filter_rows, double &subsets) {
    filter_rows = mellin ? std::max(1.0, class_rows) : pl.nfx;
    subsets = mellin ? std::ceil(filter_rows / F) : 1;
    if (!masks) return;
    Tiles &count = tiles_by_p[__builtin_ctz((unsigned)P) - 5];            // (32 to 512)
    if (count.joint != pl.joint) {
      count = Tiles{pl.joint, {}};
      runs.count_tiles(P, pl.joint ? pl.batch * pl.noy : pl.noy, count.of);
    }
    int rows = 0, stages = 0, tiles = 0;
    for (int n = 1; n <= pl.nfx; ++n) {
      rows += n * count.of[n];
      stages += (n + F - 1) / F * count.of[n];
      tiles += count.of[n];
    }
    filter_rows = (double)rows / tiles;
    subsets = (double)stages / tiles;
  };

  // The launch of a tile shape, in cycles.  Workgroups take tiles in turn, two to a CU (512 at a time).  What does not fill
  // a last turn -- for few tiles: all of them -- can be cut into slices of the contracted channels, which another kernel
  // adds up.  Measured on this chip, and rounded:
  //   a step's matrix instructions at 55-80 % of their rate (larger tiles: the higher; 128 channels x 128 positions of two by
  //   two wavefronts measure that of 64 x 512), shared by a CU's workgroups;
  //   -- all but wavefronts that share a tile, two workgroups of which in a single turn take 1.5 of one's time: one's
  //   fragments come too late for its next step (256 -> 256 channels, 4 x 4 taps, one utterance of 337 x 5, in two slices: 35
  //   -> 24 us and 5 for the sums; taken everywhere 46 drawn passes change, and take 1.04 of their time, 0.80 to 1.45; 1.2 for
  //   1.5: seven, 1.01);
  //   a stage at least 4000 (the latency of its loads);
  //   per tile 5000 for its tables (9000 where wavefronts share it in fp32: nothing runs under them) and its output at 9
  //   bytes a cycle; 9000 for a launch's start, as much for the kernel that adds the slices, and 2400 bytes a cycle for
  //   their sums.
  // Half tiles that wavefronts share cost 5000 as well: what the others pay on top is the wait for every short step's
  // fragments, which the steps' rate leaves out.  Of 3000 passes of half layers and stacks drawn over 1 to 32 images of 100 to
  // 780 rows, 1183 take other plans with 9000; 276 of those take 0.86 of the time with 5000 in the geometric mean (0.53 to
  // 1.20, twelve of them more than 1.03).  In fp32 it decides 361 of 3000, for either side: 205 of them 0.66 to 1.29.
  const int slots = 512;
  struct Launch { int M_T, P, m_tiles, per_m; i64 total; double rate, tile, output; };
  auto launch_of = [&](int nt, int wm, int wk) {
    Launch l;
    l.M_T = wm * pl.mt * 32; l.P = kWaves / wk / wm * nt * 32;
    l.m_tiles = ((int)pr.c_out + l.M_T - 1) / l.M_T;
    l.per_m = std::max(1, slots / l.m_tiles);
    l.total = (i64)((pl.tile_q + l.P - 1) / l.P) * pl.tile_batch;
    l.rate = pl.mt * nt * wm >= 8 ? 0.8 : pl.mt * nt >= 4 ? 0.65 : 0.55;
    l.tile = wk > 1 && !f16 ? 9000 : 5000;
    l.output = (double)l.M_T * l.P * (f16 ? 2 : 4) / 9;
    return l;
  };
  // Whether a shape costs `wanted` and more whatever its stages and slices are: full turns of whole steps without gaps.
  // (Choosing among the shapes is host time that every new size pays: a ten-layer Mellin stack on 32 x 700 frames took
  // 1.15 ms to plan where tiles were counted one by one for every shape and none was passed over, and takes 0.035.)
  auto hopeless = [&](const int *sh, double wanted) {
    const int nt = sh[0], wk = sh[2];
    const Launch l = launch_of(nt, sh[1], wk);
    double filter_rows, subsets;
    tile_rows(l.P, pl.nfx, filter_rows, subsets);
    const double steps = filter_rows * pl.nfy * pl.CG / (2 * wk) * pl.mt * nt * (f16 ? 1 : 6) * 32 / l.rate;
    const double least = 9000 + (double)l.total / l.per_m * (steps * (wk > 1 ? 1.5 : 2) + l.tile + l.output);
    return least >= wanted * (1 + 1e-9);
  };
  // (wanted, or 0: what costs as much is not taken)
  auto cost = [&](double wanted) {
    const Launch l = launch_of(pl.nt, pl.wm, pl.wk);
    const int M_T = l.M_T, P = l.P, total = (int)l.total, per_m = l.per_m, c_stages = pl.CG / pl.G;      // (shape(): less than 2^26 tiles)
    double filter_rows, subsets;
    tile_rows(P, pl.F, filter_rows, subsets);
    const double rows = filter_rows / subsets, tile = l.tile, output = l.output;
    const double steps = std::ceil(rows * pl.nfy * pl.G / (2 * pl.wk)) * pl.mt * pl.nt * (f16 ? 1 : 6) * 32 / l.rate;
    auto turns_cost = [&](int items, double stages) {
      const int full = items / per_m, left = items - full * per_m;
      auto turn = [&](int n) { return stages * std::max(4000.0, steps * (n * pl.m_tiles > slots / 2 ? pl.wk > 1 && full == 0 ? 1.5 : 2 : 1)) + tile + output; };
      return full * turn(per_m) + (left ? turn(left) : 0);
    };
    double best = 9000 + turns_cost(total, c_stages * subsets);
    pl.slices = like ? like->slices : 1;
    int rest = !like || !like->rest ? 0 : total;
    for (int all = 0; all < (like ? 0 : 2); ++all) {
      const int r = all ? total : total % per_m;
      if (r == 0 || (all && total >= 2 * per_m) || (pl.wk > 1 && !all)) continue;
      const double whole = 9000 + turns_cost(total - r, c_stages * subsets);
      const double least = whole + subsets * std::max(4000.0, steps) + tile + output + 9000;      // (a slice is a stage or more)
      if (least >= 0.95 * best || (wanted > 0 && best >= wanted && least >= wanted * (1 + 1e-9))) continue;
      for (int s = 2; s <= std::min(c_stages, 16); ++s) {
        const double bytes = (double)r * s * pl.m_tiles * M_T * P * 8;
        const double c = whole + turns_cost(r * s, (c_stages + s - 1) / s * subsets) + 9000 + bytes / 2400;
        if (c < 0.95 * best) { best = c; pl.slices = s; rest = r; }
      }
    }
    pl.rest = rest;
    pl.whole = total - rest;
    pl.chan_slots = total * (pl.wk > 1 ? pl.nt : kWaves / pl.wm);
    const int items = pl.whole + pl.rest * pl.slices;
    pl.grid_x = pl.wk > 1 ? items : std::min(per_m, items);      // (wavefronts that share a tile's steps take one tile)
    pl.slice_bytes = (size_t)pl.rest * pl.slices * pl.m_tiles * (size_t)(M_T * P) * 4;
    return best;
  };
  // Wavefronts that share a tile have 32 positions of it in fp32: 64 leave no registers for a gradient's ending beside the
  // separate sums, and were slower as they were (windows of ten frames 2111 -> 1998 us a step, one utterance decoded 246 ->
  // 233 us).  Half has the registers, and its shorter steps are better shared (1-D layer, 41 -> 128 channels: 15.1 us
  // without the 64 positions, 10.7 with them).
  // fp32, two wavefronts along the channels: 128 channels x 128 positions instead of 64 x 256 stage half the signal for as
  // many products, and a stage has twice the steps (128 -> 256 channels, 3 x 3, 32 x 256 x 41: 1075 -> 905 us).  77 passes of
  // stacks and layers drawn over 1 to 32 images take it: with more workgroups than CUs 1.15 times as fast in the geometric mean
  // (0.99 to 1.46), with less, which leave nothing on a CU to run beside a workgroup's waits, 0.95 (0.73 to 1.18): not those.
  // Joint tiles (Mellin axes): on small images a tile has rows of every class, and multiplies the filter rows of all of them;
  // an output row of several images has the filter rows of that row alone, and no image ends inside a tile.  96 passes of
  // windows of 5 to 20 frames and of deep layers take them: 1.36 times as fast in the geometric mean (up to 2.6; 0.92 to 1.05
  // where the model gains less than a tenth, which is why it has to).  Windows of ten frames, 64 channels: input gradients
  // 319 -> 181 us.  Channels that end inside a tile are left out (their rows would be the next image's in the stores), and
  // offsets into all images have 32 bits.
  // Input gradients only.  A stage's filter rows decide the order of the sums, and the signs of a forward pass's outputs
  // decide what their ReLU lets through: a value within its rounding error of zero passes a whole gradient on in one order
  // and none in another.  On those windows up to five flags of 74 million are not those of 64 bits, and log_eps's gradient,
  // one sum that nearly cancels, moves by up to 2e-2, where 3e-6 is its error against 64 bits at given flags.  Forward passes
  // therefore keep the tiles of an image (joint ones: the training step 1364 -> 1205 us).
  const i64 unit_bytes = 16 * parts, most = (i64)1 << 31;
  const bool can_join = gradient && mellin && masks && pl.batch > 1 && Q * pl.batch < lim && (i64)pl.batch * pl.CG * (plane + 1) * unit_bytes < most &&
                        (i64)pl.batch * pl.out_groups * (std::max(Q, out_q) + 1) * unit_bytes < most && (i64)pl.batch * pl.M * Q * 4 < most &&
                        pl.h_n == (i64)pl.M * Q;
  // Tiles of 32 channels are tried as well: where those of 64 leave half of the last one empty (65 to 96 channels, 129 to 160,
  // ..) they are taken like any other (28 passes of 400 drawn layers, 0.92 of the time in the geometric mean, 0.82 to 0.99),
  // elsewhere if the model gains a seventh (8 passes on few workgroups, 0.95, 0.91 to 1.00; with any gain 150, 0.97, 0.70 to 1.20).
  const int mt = pl.mt;
  const double narrow = (pr.c_out + 31) / 32 % 2 == 1 ? 1 : 0.85;
  BlockPlan best_plan;
  double best_cost = 0;
  for (int joint = 0; joint <= (can_join ? 1 : 0); ++joint) {
    double limit = joint && best_cost > 0 ? 0.9 * best_cost : 0;
    set_joint(joint);
    for (pl.mt = mt; pl.mt >= 1; --pl.mt)
      for (int k = 0; k < kShapes; ++k) {
        const int *const sh = shapes[k];
        if (pl.mt < mt && sh[1] == 2) continue;
        if (like && (like->mt * like->wm != pl.mt * sh[1] || kWaves / like->wm * like->nt != kWaves / sh[1] * sh[0] || sh[2] != like->wk)) continue;
        if (f16 ? sh[0] == 2 && sh[1] == 2 : sh[0] == 4 || (sh[0] == 2 && sh[2] == 4)) continue;
        if (sh[1] == 2 && pr.c_out <= 96) continue;      // (two wavefronts along the channels: most of 128)
        const double wanted = (pl.mt < mt ? narrow : 1) * limit;
        // (joint tiles often have no stage that fits, and take longer to count)
        if (limit > 0 && !joint && hopeless(sh, wanted)) continue;
        if (!shape(k) || (limit > 0 && joint && hopeless(sh, wanted))) continue;
        const double c = cost(wanted);
        if (!f16 && sh[1] == 2 && ((i64)pl.whole + (i64)pl.rest * pl.slices) * pl.m_tiles <= slots / 2) continue;
        if (limit == 0 || c < wanted) { limit = best_cost = c; best_plan = pl; }
      }
  }
  if (best_cost == 0) return false;
  pl = best_plan;
  // Wavefronts that share a tile, more workgroups than two a CU: stages that leave room for a third, where it has registers,
  // if they are not much smaller for it (or half on linear axes, whose steps are short).  Input gradient of 41 -> 128
  // channels, 8 taps, 32 x 780, p = 3, 800 workgroups: 29.5 -> 24.6 us.  Of 40 drawn passes of more than 512 workgroups 13 take
  // it, 0.80 to 0.98 of their time; those with smaller stages 0.97 to 1.26.  Input gradients only: a stage decides which
  // wavefront adds what (see can_join).
  if (gradient && pl.wk > 1 && ((i64)pl.whole + (i64)pl.rest * pl.slices) * pl.m_tiles > slots) {
    const int at = pl.nt == 2 ? 5 : 6, fg = pl.F * pl.G, g = pl.G;
    room = 53 * 1024;
    stages[pl.mt - 1][at].rows = -1;
    const bool fits = shape(at), large = (pl.G == g && 2 * pl.F * pl.G >= fg) || (2 * pl.G >= g && 5 * pl.F * pl.G >= 3 * fg);
    const bool dealt = pl.rest == 0 || pl.slices <= pl.CG / pl.G;        // (a slice is a stage or more)
    if (!fits || !dealt || !(large || (f16 && !mellin))) pl = best_plan;
  }
  if (!f16 && pl.mt == 2 && pl.nt == 1 && pl.wk == 1) {
    // fp32, 64 channels x 128 positions: two by two wavefronts of 32 channels x 64 positions.  Four side by side take each
    // filter fragment from L1 four times, 64 bytes a cycle and CU, which is all that it gives; two by two take half of that and
    // twice the signal's operands out of LDS, also 64 of its 128 (64 -> 64 channels, 5 x 3 taps on 1177 x 10 x 41: 195 -> 178
    // us; on 5 x 41: 180 -> 167).  Tile, stage and order of sums are the same.
    pl.mt = 1; pl.nt = 2; pl.wm = 2;
    pl.chan_slots = (pl.whole + pl.rest) * (kWaves / pl.wm);
  }
  const i64 per_row = (i64)pl.nfy * pl.G, pairs = 2 * pl.wk;
  // Whole tiles with fewer filter rows than a stage holds have stages of more channel groups, as many as its LDS has room for: a
  // stage of one row of three, two groups and three columns is three steps, shorter than the trip of the next one's loads (128 <-
  // 256 channels, 3 x 3 taps, p = 2, 32 x 256 x 41, half: 182 -> 165 us; fp32, whose steps are six times as long: 96 channels, 6 x 3 taps, p = 2, 640 -> 629
  // us a step).  Input gradients only: in a forward pass the order of a value's sums would depend on the tile that it lies
  // in, and that order decides what the ReLUs let through (see can_join, `like`); in half it gained a twentieth there.
  const i64 tile_rows_most = std::min<i64>(pl.joint ? (i64)pl.nox * pl.batch : pl.nox, (kWaves / pl.wk / pl.wm * pl.nt * 32 + pl.noy - 2) / pl.noy + 1);
  for (int n = 1; n <= pl.F; ++n) {
    int G = pl.G;
    if (mellin && gradient)
      for (int k = n_groups - 1; k >= 0; --k)              // (fewest first)
        if (groups[k] > G && n * groups[k] <= pl.F * pl.G &&
            groups[k] * ((n * tile_rows_most * pl.RS * parts + 63) / 64 * 1024) <= pl.buf_bytes)
          G = groups[k];
    pl.stage[n - 1] = BlockStage{G, magic(G), magic((i64)pl.nfy * G)};
  }
  pl.mg_full = magic(std::max<i64>((pl.F * per_row + pairs - 1) / pairs * pairs, (deep_fragments(f16, pl.wk) ? 4 : 2) * pairs));
  pl.rows_off = (size_t)pl.m_tiles * pl.wm * pl.mt * ((size_t)pl.CG * pl.nfx * pl.nfy + 1) * parts * 512;
  if (pl.rows_off >= (size_t)lim) return false;
  pl.filter_bytes = pl.rows_off + (mellin ? 8 * (size_t)pl.nox : 0);
  return true;
}

bool pool_block_plan(const BlockPool &pool, BlockPlan &pl) {
  const i64 out_q = pool.kind == 1 ? pl.Q / 2 : (i64)pl.nox * pool.cols, most = (i64)1 << 31;
  if (pl.out_groups * (out_q + 1) * 48 >= most) return false;    // (32-bit byte offsets, as make_block_plan)
  if (pl.joint && pl.batch * pl.out_groups * (out_q + 1) * (pl.f16 ? 16 : 48) >= most) return false;
  pl.pool = pool.kind;
  pl.out_q = (int)out_q;
  pl.out_cols = pool.cols;
  return true;
}

hipError_t launch_block_gemm(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream) {
  if (pl.pool) return a.grad ? launch_grad_pooled(pl, a, stream) : launch_out_pooled(pl, a, stream);
  if (a.grad) return a.blocked ? launch_grad_blocked(pl, a, stream) : launch_grad_plain(pl, a, stream);
  return a.blocked ? launch_out_blocked(pl, a, stream) : launch_shape<OUT_PLAIN>(pl, a, stream);
}

}  // namespace mellin
