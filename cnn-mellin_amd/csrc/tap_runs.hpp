// Which filter rows have a tap inside the signal, over the output rows of a Mellin axis, and how many of them the tiles of a
// blocked pass meet: what its plan is chosen by (block_gemm.hip).  Plain host code.
//
// The plan of a new size is host time that its first call pays: rows are taken in runs with the same taps and tiles are counted
// by the run.  Row by row and tile by tile, for every tile shape, a ten-layer Mellin stack on 32 x 700 frames took 1150 us of
// host time before its first step; with runs, counted once per number of positions, 35.
#pragma once

#include <algorithm>

namespace mellin {

// h = output row + s, f = filter row + d: the input row + u is h f / p1 (corr) or h p1 / f, where that is whole
struct TapAxis { bool corr; int nf, ng, s, d, p1, u; };

class TapRuns {
 public:
  static constexpr int kRows = 4096, kFilterRows = 16;
  struct Run { int end; unsigned mask; };              // rows up to `end` (from the run before), bits of filter rows

  // The next `count` rows: output rows first, first + stride, ...  (products of rows and filter rows below 2^31)
  void add_class(const TapAxis &x, int first, int stride, int count) {
    // the input rows of a filter row's taps step evenly, so it has taps for one run [lo, hi) of a residue class's rows
    int lo[kFilterRows], hi[kFilterRows], cut[2 * kFilterRows + 1], cuts = 0;
    const int h = first + x.s;
    bool even = true;
    for (int f = 0; f < x.nf && even; ++f) {
      const int up = x.corr ? f + x.d : x.p1, den = x.corr ? x.p1 : f + x.d, num = h * up, step = stride * up / den;
      even = step * den == stride * up;
      lo[f] = hi[f] = 0;
      if (!even || num % den) continue;
      const int at = num / den - x.u;                  // the first row's input row
      lo[f] = at >= 0 ? 0 : std::min((step - 1 - at) / step, count);
      hi[f] = at >= x.ng ? 0 : std::min((x.ng - 1 - at) / step + 1, count);
      if (lo[f] >= hi[f]) { lo[f] = hi[f] = 0; continue; }
      if (lo[f] > 0) cut[cuts++] = lo[f];
      if (hi[f] < count) cut[cuts++] = hi[f];
    }
    const int start = n_ ? runs_[n_ - 1].end : 0;
    if (even) {
      cut[cuts++] = count;
      std::sort(cut, cut + cuts);
      for (int c = 0, from = 0; c < cuts; from = cut[c++]) {
        if (cut[c] == from) continue;
        unsigned mask = 0;
        for (int f = 0; f < x.nf; ++f)
          if (from >= lo[f] && from < hi[f]) mask |= 1u << f;
        add(start + cut[c], mask);
      }
      return;
    }
    // rows of several residue classes (more than a plan holds): filter row by filter row, every `every`th row has its tap
    unsigned short row_mask[kRows];
    std::fill(row_mask, row_mask + count, 0);
    for (int f = 0; f < x.nf; ++f) {
      const int up = x.corr ? f + x.d : x.p1, den = x.corr ? x.p1 : f + x.d;
      int a = up * stride, b = den;
      while (b) { const int t = a % b; a = b; b = t; }
      const int every = den / a, step = up * stride / a;
      for (int r = 0; r < std::min(every, count); ++r) {
        if ((h + r * stride) * up % den) continue;
        for (int row = r, at = (h + r * stride) * up / den - x.u; row < count && at < x.ng; row += every, at += step)
          if (at >= 0) row_mask[row] |= 1u << f;
        break;
      }
    }
    for (int row = 0; row < count; ++row) add(start + row + 1, row_mask[row]);
  }

  // of[n] += tiles of P positions whose rows (per_row positions each) meet n filter rows, at least one.  Rows of many tiles are
  // counted as if each began one.
  void count_tiles(int P, int per_row, int *of) const {
    auto put = [&](unsigned mask, int n) { of[std::max(1, __builtin_popcount(mask))] += n; };
    if (per_row >= 8 * P) {
      for (int r = 0; r < n_; ++r) put(runs_[r].mask, runs_[r].end - (r ? runs_[r - 1].end : 0));
      return;
    }
    const int all = n_ ? runs_[n_ - 1].end * per_row : 0;
    for (int q = 0, r = 0; q < all;) {
      while (runs_[r].end * per_row <= q) ++r;
      const int inside = (runs_[r].end * per_row - q) / P;
      if (inside) { put(runs_[r].mask, inside); q += inside * P; continue; }
      unsigned mask = runs_[r].mask;
      for (int k = r, last = std::min(q + P, all); runs_[k].end * per_row < last;) mask |= runs_[++k].mask;
      put(mask, 1);
      q += P;
    }
  }

 private:
  void add(int end, unsigned mask) {
    if (n_ && runs_[n_ - 1].mask == mask) runs_[n_ - 1].end = end;
    else runs_[n_++] = Run{end, mask};
  }
  Run runs_[kRows];
  int n_ = 0;
};

}  // namespace mellin
