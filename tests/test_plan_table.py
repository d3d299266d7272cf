"""The table that keeps the layers' plans by their sizes (csrc/plan_table.hpp), compiled for the host."""
import ctypes
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PLACES, WORDS = 64, 18
SOURCE = """
#include "plan_table.hpp"
static mellin::PlanTable<int64_t, %d, %d> table;
extern "C" int64_t look_up(const int64_t *words, int64_t value) {
  int64_t key[%d];
  memcpy(key, words, sizeof key);
  int64_t &at = table.at(key), before = at;
  at = value;
  return before;
}
""" % (PLACES, WORDS, WORDS)


@pytest.fixture
def look_up(tmp_path):
    (tmp_path / "table.cpp").write_text(SOURCE)
    lib = str(tmp_path / "table.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "cnn-mellin_amd", "csrc"),
                           str(tmp_path / "table.cpp"), "-o", lib])
    fn = ctypes.CDLL(lib).look_up
    fn.restype, fn.argtypes = ctypes.c_int64, [ctypes.POINTER(ctypes.c_int64), ctypes.c_int64]
    return lambda key, value: fn((ctypes.c_int64 * WORDS)(*key), value)


def _sizes(n, seed):
    """Distinct layers of ordinary sizes, as the library's look-ups name them."""
    rng, keys = random.Random(seed), set()
    while len(keys) < n:
        c, t = rng.choice((16, 32, 64, 128, 256)), rng.randint(10, 780)
        keys.add((rng.choice((1, 2, 5, 6)), rng.randint(1, 32), c, c, 4, 4, t, 41, t, 41) + (1,) * 4 + (1, 1, 1, 1))
    return sorted(keys)


@pytest.mark.parametrize("n", [1, 10, PLACES])
def test_every_size_is_found_again(look_up, n):
    keys = _sizes(n, 11 + n)
    assert [look_up(k, i + 1) for i, k in enumerate(keys)] == [0] * n
    for _ in range(2):
        assert [look_up(k, i + 1) for i, k in enumerate(keys)] == [i + 1 for i in range(n)]


def test_more_sizes_than_places_never_give_another_size_its_plan(look_up):
    keys = _sizes(3 * PLACES, 5)
    for _ in range(4):
        for i, k in enumerate(keys):
            assert look_up(k, i + 1) in (0, i + 1)
            assert look_up(k, i + 1) == i + 1
