"""The counting behind the blocked kernels' plans (csrc/tap_runs.hpp), compiled for the host, against the same counted row by row
and tile by tile."""
import ctypes
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "tap_runs.hpp"
using namespace mellin;
// the axis's residue classes, one behind the other (n_classes = 1: rows of all residues)
extern "C" void count(const int *axis, int n_classes, const int *first, int stride, const int *rows, int P, int per_row, int *of) {
  TapRuns runs;
  for (int k = 0; k < n_classes; ++k)
    runs.add_class(TapAxis{axis[0] != 0, axis[1], axis[2], axis[3], axis[4], axis[5], axis[6]}, first[k], stride, rows[k]);
  runs.count_tiles(P, per_row, of);
}
"""


@pytest.fixture(scope="module")
def count(tmp_path_factory):
    at = tmp_path_factory.mktemp("tap_runs")
    (at / "runs.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror",
                           "-I" + os.path.join(ROOT, "cnn-mellin_amd", "csrc"), str(at / "runs.cpp"), "-o", str(at / "runs.so")])
    fn = ctypes.CDLL(str(at / "runs.so")).count
    fn.restype = None

    def call(axis, classes, stride, P, per_row):
        ints = lambda v: (ctypes.c_int * len(v))(*v)
        of = (ctypes.c_int * 17)()
        fn(ints(axis), len(classes), ints([c[0] for c in classes]), stride, ints([c[1] for c in classes]), P, per_row, of)
        return list(of)
    return call


def _count(axis, classes, stride, P, per_row):
    corr, nf, ng, s, d, p1, u = axis
    masks = []
    for first, rows in classes:
        for i in range(rows):
            h, mask = first + i * stride + s, 0
            for f in range(nf):
                num, den = (h * (f + d), p1) if corr else (h * p1, f + d)
                if num % den == 0 and u <= num // den < u + ng:
                    mask |= 1 << f
            masks.append(mask)
    of = [0] * 17
    if per_row >= 8 * P:
        for m in masks:
            of[max(1, bin(m).count("1"))] += 1
        return of
    total = len(masks) * per_row
    for q in range(0, total, P):
        mask = 0
        for m in masks[q // per_row:(min(q + P, total) - 1) // per_row + 1]:
            mask |= m
        of[max(1, bin(mask).count("1"))] += 1
    return of


@pytest.mark.parametrize("corr", [1, 0], ids=["corr", "conv"])
@pytest.mark.parametrize("whole", [False, True], ids=["classes", "mixed"])
def test_tiles_by_runs_are_those_row_by_row(count, corr, whole):
    rng = random.Random(100 + 2 * corr + whole)
    for _ in range(300):
        nf, ng, s, d, p1, u = rng.randint(1, 16), rng.randint(1, 200), rng.randint(1, 4), rng.randint(1, 12), rng.randint(1, 9), rng.randint(1, 5)
        nh = rng.choice((1, 2, rng.randint(1, 60), rng.randint(1, 400)))
        period = p1
        if not corr:
            period = 1
            for f in range(nf):
                a, b = f + d, p1
                while b:
                    a, b = b, a % b
                m = (f + d) // a
                a, b = period, m
                while b:
                    a, b = b, a % b
                period = period // a * m
        if whole or period > 32:
            classes, stride = [(0, nh)], 1
        else:
            order = rng.sample(range(period), period)
            classes, stride = [(r, len(range(r, nh, period))) for r in order if r < nh], period
        axis, P = (corr, nf, ng, s, d, p1, u), rng.choice((32, 64, 128, 256, 512))
        per_row = rng.choice((1, 5, 41, 33, rng.randint(1, 300), 8 * P, 8 * P - 1, 3 * P))
        assert count(axis, classes, stride, P, per_row) == _count(axis, classes, stride, P, per_row), (axis, classes, stride, P, per_row)
