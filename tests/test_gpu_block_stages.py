"""Stages of the channel-blocked matrix kernel: how many channel groups and steps one has, from tile to tile of a launch; output
and gradients against the float64 checker."""
import ctypes

import numpy as np
import pytest

import _mellin_hip as hip
import mconv
from _gpu import assert_close, to_gpu
from oracle import oracle

CASES = [
    # (op, n, c_in, c_out, nf, ng, s, d, p, r)
    # input gradients on Mellin axes whose rows have one, two or all filter rows: stages of the plan's groups, of two, three and
    # four times as many, of a number that the groups leave no room for (5 and 7 groups have no divisor), tiles of several
    # classes, tiles over the images of a row, tiles in slices of the contracted channels
    ("mcorr", 6, 64, 128, (3, 3), (64, 41), (1, 1), (2, 1), (2, 1), (2, 1)),
    ("mcorr", 4, 48, 96, (6, 3), (100, 40), (1, 1), (1, 1), (2, 1), (2, 1)),
    ("mcorr", 3, 32, 40, (4, 2), (70, 21), (1, 1), (1, 1), (3, 0), (5, 0)),
    ("mcorr", 3, 32, 56, (5, 1), (130, 7), (1, 1), (1, 1), (1, 0), (40, 0)),
    ("mcorr", 90, 32, 64, (4, 3), (9, 20), (1, 1), (1, 1), (1, 1), (3, 1)),
    ("mcorr", 1, 32, 128, (7, 1), (300, 1), (1, 1), (1, 1), (2, 0), (0, 0)),
    ("mcorr", 1, 64, 256, (4, 4), (60, 5), (1, 1), (1, 1), (1, 1), (30, 2)),
    ("mcorr", 1, 40, 64, (6, 1), (145, 10), (1, 1), (2, 1), (0, 0), (3, 0)),
    ("mcorr", 6, 32, 64, (8, 1), (160, 20), (1, 1), (1, 1), (0, 0), (0, 0)),
    # stages of one, two, three, four, five, six and seven steps: half tiles request fragments four steps ahead, and one stage
    # (one tile, or several, or many of a workgroup) reads into the next
    ("lcorr", 20, 16, 64, (2, 1), (200, 20), (1, 1), (1, 1), (0, 0), (0, 0)),
    ("lcorr", 20, 16, 64, (2, 2), (200, 20), (1, 1), (1, 1), (0, 0), (0, 0)),
    ("lcorr", 20, 16, 64, (3, 1), (200, 20), (1, 1), (1, 1), (1, 0), (1, 0)),
    ("lcorr", 20, 24, 64, (3, 1), (200, 20), (1, 1), (1, 1), (1, 0), (1, 0)),
    ("lcorr", 20, 40, 40, (2, 1), (200, 20), (1, 1), (1, 1), (0, 0), (0, 0)),
    ("lcorr", 70, 16, 128, (3, 2), (90, 20), (1, 1), (1, 1), (1, 0), (1, 0)),
    ("lcorr", 20, 56, 104, (2, 1), (200, 20), (1, 1), (1, 1), (0, 0), (0, 0)),
    ("mcorr", 30, 24, 72, (3, 1), (150, 20), (1, 1), (1, 1), (2, 0), (60, 0)),
    # input gradients by wavefronts that share a tile, stages that leave room for a third workgroup on a CU (float; half)
    ("mcorr", 16, 41, 128, (6, 1), (1201, 1), (1, 1), (1, 1), (2, 0), (0, 0)),
    ("lcorr", 7, 24, 110, (4, 4), (130, 41), (1, 1), (1, 1), (1, 1), (1, 1)),
]


def plan(case, elem_bytes, gradient):
    """The pass's plan, its stages' channel groups by the filter rows of a tile, and a workgroup's LDS bytes."""
    op, n, c_in, c_out, nf, ng, s, d, p, r = case
    kind, valid = (hip.AX_MCORR, mconv.mcorr_valid_size) if op == "mcorr" else (hip.AX_LCORR, mconv.lcorr_valid_size)
    nh = valid(nf[0], ng[0], s[0], d[0], p[0]) + r[0], mconv.lcorr_valid_size(nf[1], ng[1], s[1], d[1], p[1]) + r[1]
    dims, words, stages = hip._dims(n, c_in, c_out, nf, ng, nh, s, d, p, (1, 1)), (ctypes.c_int * 10)(), (ctypes.c_int * 17)()
    assert hip.lib.mellin_layer_plan(kind, elem_bytes, gradient, *dims, words)
    assert hip.lib.mellin_layer_stages(kind, elem_bytes, gradient, *dims, stages)
    return dict(zip("mt nt wm wk joint F G whole rest slices".split(), words)), list(stages[:16]), stages[16]


def test_cases_have_the_stages_that_they_are_there_for():
    larger, kinds = CASES[:9], set()
    for elem_bytes in (4, 2):
        ratios = set()
        for case in larger:
            pl, groups, _ = plan(case, elem_bytes, 1)
            assert all(g == pl["G"] for g in groups[pl["F"] - 1:])
            if pl["whole"]:
                ratios |= {g / pl["G"] for g in groups}
                kinds |= {"joint"} if pl["joint"] and groups[0] > pl["G"] else set()
                kinds |= {"no divisor"} if pl["G"] in (5, 7) else set()
            kinds |= {"slices"} if pl["rest"] and pl["wk"] > 1 and groups[0] > pl["G"] else set()
            assert set(plan(case, elem_bytes, 0)[1]) == {plan(case, elem_bytes, 0)[0]["G"]}      # (forward passes: one size)
        assert ratios >= ({1, 2, 3, 4} if elem_bytes == 4 else {1, 1.5, 4})
    assert kinds == {"joint", "no divisor", "slices"}
    steps = set()
    for case in CASES[9:17]:
        for gradient in (0, 1):
            pl = plan(case, 2, gradient)[0]
            if pl["wk"] == 1:
                steps.add(-(-pl["F"] * case[4][1] * pl["G"] // 2))
    assert steps >= set(range(1, 8))
    for case, elem_bytes in zip(CASES[17:], (4, 2)):
        pl, _, lds = plan(case, elem_bytes, 1)
        m_tiles = -(-case[2] // (32 * pl["mt"] * pl["wm"]))
        assert pl["wk"] > 1 and (pl["whole"] + pl["rest"] * pl["slices"]) * m_tiles > 512 and lds <= 53 * 1024


@pytest.mark.gpu
@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_stages_match_checker(case, half):
    op, n, c_in, c_out, nf, ng, s, d, p, r = case
    rng = np.random.default_rng(7700 + CASES.index(case))
    kind = np.float16 if half else np.float32
    x = rng.standard_normal((n, c_in) + ng).astype(kind)
    w = (rng.standard_normal((c_out, c_in) + nf) * (c_in * nf[0] * nf[1]) ** -0.5).astype(kind)
    b = rng.standard_normal(c_out).astype(kind)
    fwd = oracle.mcorrlcorr if op == "mcorr" else oracle.lcorrlcorr
    bwd = oracle.mcorrlcorr_backward if op == "mcorr" else oracle.lcorrlcorr_backward
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    exp = fwd(x64, w64, b.astype(np.float64), s, d, p, (1, 1), r)
    go = rng.standard_normal(exp.shape).astype(kind)
    egi, egw, _ = bwd(x64, w64, go.astype(np.float64), s, d, p, (1, 1))
    xg, wg, bg = (to_gpu(a).requires_grad_() for a in (x, w, b))
    out = (mconv._ext_mcorrlcorr if op == "mcorr" else mconv._ext_lcorrlcorr)(xg, wg, bg, s, d, p, (1, 1), r)
    assert hip.last_variant() == ("mfma-f16-blocks" if half else "mfma-blocks")
    out.backward(to_gpu(go))
    taps, positions = nf[0] * nf[1], n * exp.shape[2] * exp.shape[3]
    for got, ref, fan, what in ((out, exp, c_in * taps, "out"), (xg.grad, egi, c_out * taps, "grad_input"),
                                (wg.grad, egw, positions, "grad_weight")):
        if half:                                       # one rounding of a result whose sum has an error of its own
            err = np.abs(got.detach().double().cpu().numpy() - ref)
            assert np.all(err <= 2.0 ** -10 * np.abs(ref) + 2e-5 * fan ** 0.5), what
        else:
            assert_close(got, ref, fan, what)
