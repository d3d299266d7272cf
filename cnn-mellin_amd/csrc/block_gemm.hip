// Plans of the channel-blocked matrix kernel (block_gemm_kernel.hpp): tile shape, stages and turns of a launch, and the
// launches that write a layer's output as it lies.  The kernel's other endings are in block_gemm_out.hip and
// block_gemm_grad_*.hip (a translation unit each, for the time they take to compile).
#include <algorithm>
#include <cmath>

#include "block_gemm_kernel.hpp"

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

bool make_block_plan(const SepConv &pr, bool f16, bool gradient, BlockPlan &pl) {
  const Axis &X = pr.x, &Y = pr.y;
  const i64 lim = (i64)1 << 30;
  if (pr.accumulate || pr.batch < 1 || pr.c_out < 1 || pr.c_in < 1 || X.nf < 1 || Y.nf < 1 || X.nf > kBlockFilterRows) return false;
  if (Y.kind != AX_LCORR && Y.kind != AX_LCONV) return false;
  const i64 plane = X.ng * Y.ng, Q = X.nh * Y.nh;
  if (plane < 1 || Q < 1 || plane >= (i64)1 << 22 || Q >= (i64)1 << 22) return false;
  if (pr.batch > 65535 || pr.c_in > 8 * 65535 || pr.c_out * Q >= lim / 2 || Q >= (i64)1 << 20 ||
      (pr.c_out + 7) / 8 * (Q + 1) * 48 >= (i64)1 << 31)
    return false;                                      // (32-bit byte offsets)
  if (X.s > 4096 || X.d > 4096 || X.u > 4096 || X.p > 4096 || X.p < -lim || Y.s > 64 || Y.d > 4096 || Y.u > 64 || Y.p > lim || Y.p < -lim)
    return false;
  pl.f16 = f16;
  pl.wide = 0;
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

  // A tile shape's stage: the channel groups and filter rows that fit twice into the LDS that a
  // workgroup may take, two workgroups to a CU
  auto shape = [&](int nt, int wm, int wk) {
    const int P = (kWaves / wk / wm) * nt * 32, M_T = wm * pl.mt * 32;
    const i64 RT = std::min<i64>(pl.joint ? (i64)pl.nox * pl.batch : pl.nox, (P - 1 + pl.noy - 1) / pl.noy + 1);
    const i64 vrows = mellin ? RT : (i64)pl.ax * (RT - 1) + pl.bx_span + 1;
    const i64 tab = ((mellin ? vrows * pl.nfx : vrows) * pl.RS + 64 + 64 + 3) & ~(i64)3;
    const i64 row_src = mellin ? 4 * RT * pl.nfx : 0;
    auto pad = [&](i64 halves) { return std::max<i64>((halves + 2 * wk - 1) / (2 * wk) * (2 * wk), 4 * wk); };
    int best_f = 0, best_g = 0;
    double best = 0;
    for (int F = mellin ? pl.nfx : 1; F >= 1; --F) {
      const int rows = mellin ? F : pl.nfx;
      const i64 units = vrows * (mellin ? F : 1) * pl.RS;
      const i64 gb = (units * parts + 63) / 64 * 1024;
      for (int G = std::min(pl.CG, 8); G >= 1; --G) {
        if (pl.CG % G) continue;
        const i64 ents = (mellin ? (pl.nfx + F - 1) / F : 1) * pad((i64)rows * pl.nfy * G) + 8 * wk;
        const i64 bytes = 2 * gb * G + 4 * tab + 16 * ents + row_src + M_T * 4;
        if (bytes > 79 * 1024) continue;
        // what a stage's steps fill of their whole pairs, against what a stage costs on top (its barrier and first reads)
        const i64 halves = (i64)rows * pl.nfy * G;
        const double rate = (double)halves / (double)(pad(halves) + 2 * wk);
        if (rate > best) { best = rate; best_f = F; best_g = G; }
      }
    }
    if (!best_f) return false;
    const i64 units = vrows * (mellin ? best_f : 1) * pl.RS;
    pl.F = mellin ? best_f : pl.nfx;
    pl.G = best_g;
    pl.tab_units = (int)tab;
    pl.ents = (int)((mellin ? (pl.nfx + pl.F - 1) / pl.F : 1) * pad((i64)pl.F * pl.nfy * best_g) + 8 * wk);
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
    return bytes <= 79 * 1024;
  };
  auto magic = [](i64 d) { return d <= 1 ? 0xFFFFFFFFu : (unsigned)(0x100000000ull / (unsigned)d); };
  pl.mg_batch = magic(pl.batch); pl.mg_noy = magic(pl.noy);
  auto set_joint = [&](int joint) {
    pl.joint = joint;
    pl.tile_batch = joint ? 1 : pl.batch;
    pl.tile_q = joint ? pl.nox * pl.batch * pl.noy : pl.Q;
  };
  // Mellin axes: which filter rows have a tap inside the signal, per output row in the order of the classes (axes of
  // more rows, of which a tile's share a class: those of the class)
  constexpr int kMaskRows = 4096;
  unsigned row_mask[kMaskRows];
  const bool masks = mellin && pl.nox <= kMaskRows;
  double class_rows = 0;
  if (mellin)
    for (int k = 0; k < pl.n_classes; ++k) {
      const int end = k + 1 < pl.n_classes ? pl.cls[k + 1].start : pl.nox;
      class_rows += __builtin_popcount(pl.cls[k].mask) * (double)(end - pl.cls[k].start) / pl.nox;
      for (int at = pl.cls[k].start; masks && at < end; ++at) {
        const unsigned h = (unsigned)(pl.cls[k].first + (at - pl.cls[k].start) * pl.cls_stride + pl.sx), p1 = (unsigned)pl.px + 1;
        unsigned mask = 0;
        for (int f = 0; f < pl.nfx; ++f) {
          const unsigned fd = (unsigned)(f + pl.dx), num = X.kind == AX_MCORR ? h * fd : h * p1, den = X.kind == AX_MCORR ? p1 : fd;
          const unsigned q = num / den;
          if (q * den == num && q >= (unsigned)pl.ux && q - (unsigned)pl.ux < (unsigned)pl.ngx) mask |= 1u << f;
        }
        row_mask[at] = mask;
      }
    }
  // What a tile of P positions stages: filter rows, and stages of them, on average.  (Counted over the tile's rows together:
  // with the average of single rows small images of many classes got tiles that stage nearly every filter row; windows of
  // ten frames 1989 -> 1968 us a step, a ten-layer Mellin stack of 24 to 192 channels on two utterances 1175 -> 1117 us.)
  auto tile_rows = [&](int P, double &filter_rows, double &subsets) {
    filter_rows = mellin ? std::max(1.0, class_rows) : pl.nfx;
    subsets = mellin ? std::ceil(filter_rows / pl.F) : 1;
    if (!masks) return;
    i64 rows = 0, stages = 0, tiles = 0;
    const i64 per_row = pl.joint ? (i64)pl.batch * pl.noy : pl.noy, all = pl.tile_q;
    // (rows of many tiles: as if each began one)
    for (i64 q0 = 0; q0 < all; q0 = per_row >= 8 * P ? q0 + per_row : q0 + P, ++tiles) {
      const i64 last = per_row >= 8 * P ? q0 / per_row : (std::min<i64>(q0 + P, all) - 1) / per_row;
      unsigned mask = 0;
      for (i64 r = q0 / per_row; r <= last; ++r) mask |= row_mask[r];
      const int n = std::max(1, __builtin_popcount(mask));
      rows += n;
      stages += (n + pl.F - 1) / pl.F;
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
  const i64 slots = 512;
  auto cost = [&]() {
    const int M_T = pl.wm * pl.mt * 32, P = kWaves / pl.wk / pl.wm * pl.nt * 32;
    const i64 total = (i64)((pl.tile_q + P - 1) / P) * pl.tile_batch, per_m = std::max<i64>(1, slots / pl.m_tiles), c_stages = pl.CG / pl.G;
    double filter_rows, subsets;
    tile_rows(P, filter_rows, subsets);
    const double rows = filter_rows / subsets;
    const double rate = pl.mt * pl.nt * pl.wm >= 8 ? 0.8 : pl.mt * pl.nt >= 4 ? 0.65 : 0.55;
    const double steps = std::ceil(rows * pl.nfy * pl.G / (2 * pl.wk)) * pl.mt * pl.nt * (f16 ? 1 : 6) * 32 / rate;
    const double output = (double)M_T * P * (f16 ? 2 : 4) / 9;
    const double tile = pl.wk > 1 && !f16 ? 9000 : 5000;
    auto turns_cost = [&](i64 items, double stages) {
      const i64 full = items / per_m, left = items - full * per_m;
      auto turn = [&](i64 n) { return stages * std::max(4000.0, steps * (n * pl.m_tiles > slots / 2 ? pl.wk > 1 && full == 0 ? 1.5 : 2 : 1)) + tile + output; };
      return full * turn(per_m) + (left ? turn(left) : 0);
    };
    double best = 9000 + turns_cost(total, c_stages * subsets);
    pl.slices = 1;
    i64 rest = 0;
    for (int all = 0; all < 2; ++all) {
      const i64 r = all ? total : total % per_m;
      if (r == 0 || (all && total >= 2 * per_m) || (pl.wk > 1 && !all)) continue;
      for (i64 s = 2; s <= std::min<i64>(c_stages, 16); ++s) {
        const double bytes = (double)r * s * pl.m_tiles * M_T * P * 8;
        const double c = 9000 + turns_cost(total - r, c_stages * subsets) + turns_cost(r * s, std::ceil((double)c_stages / s) * subsets) +
                         9000 + bytes / 2400;
        if (c < 0.95 * best) { best = c; pl.slices = (int)s; rest = r; }
      }
    }
    pl.rest = (int)rest;
    pl.whole = (int)(total - rest);
    pl.chan_slots = (int)total * (pl.wk > 1 ? pl.nt : kWaves / pl.wm);
    const i64 items = (i64)pl.whole + (i64)pl.rest * pl.slices;
    pl.grid_x = (int)(pl.wk > 1 ? items : std::min<i64>(per_m, items));      // (wavefronts that share a tile's steps take one tile)
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
  static const int shapes[][3] = {{4, 2, 1}, {4, 1, 1}, {2, 2, 1}, {2, 1, 1}, {1, 1, 1}, {2, 1, 4}, {1, 1, 4}};   // nt, wm, wk
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
                        (i64)pl.batch * pl.out_groups * (Q + 1) * unit_bytes < most && (i64)pl.batch * pl.M * Q * 4 < most &&
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
      for (const auto &sh : shapes) {
        if (pl.mt < mt && sh[1] == 2) continue;
        if (f16 ? sh[0] == 2 && sh[1] == 2 : sh[0] == 4 || (sh[0] == 2 && sh[2] == 4)) continue;
        if (sh[1] == 2 && pr.c_out <= 96) continue;      // (two wavefronts along the channels: most of 128)
        if (!shape(sh[0], sh[1], sh[2])) continue;
        const double c = cost();
        if (!f16 && sh[1] == 2 && ((i64)pl.whole + (i64)pl.rest * pl.slices) * pl.m_tiles <= slots / 2) continue;
        if (limit == 0 || c < (pl.mt < mt ? narrow : 1) * limit) { limit = best_cost = c; best_plan = pl; }
      }
  }
  if (best_cost == 0) return false;
  pl = best_plan;
  const i64 per_row = (i64)pl.nfy * pl.G, pairs = 2 * pl.wk;
  pl.mg_per_row = magic(per_row); pl.mg_G = magic(pl.G);
  pl.mg_full = magic(std::max<i64>((pl.F * per_row + pairs - 1) / pairs * pairs, 2 * pairs));
  pl.rows_off = (size_t)pl.m_tiles * pl.wm * pl.mt * ((size_t)pl.CG * pl.nfx * pl.nfy + 1) * parts * 512;
  if (pl.rows_off >= (size_t)lim) return false;
  pl.filter_bytes = pl.rows_off + (mellin ? 8 * (size_t)pl.nox : 0);
  return true;
}

hipError_t launch_block_gemm(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream) {
  if (a.grad) return a.blocked ? launch_grad_blocked(pl, a, stream) : launch_grad_plain(pl, a, stream);
  return a.blocked ? launch_out_blocked(pl, a, stream) : launch_shape<OUT_PLAIN>(pl, a, stream);
}

}  // namespace mellin
