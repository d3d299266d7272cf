"""Tile shapes of the channel-blocked matrix kernel that the layers of test_gpu_blocks.py are too small for: all three
gradients and the output against the float64 checker."""
import numpy as np
import pytest
import torch

import _mellin_hip as hip
import mconv
from _gpu import assert_close, to_gpu
from oracle import oracle
from test_block_plans import plan

pytestmark = pytest.mark.gpu

CASES = [
    # (op, n, c_in, c_out, nf, ng, s, d, p, r)
    # fp32, two wavefronts along the channels (more than 96 channels, more workgroups than CUs): a second tile of two
    # channels, a first one that ends inside a tile of 32, last position tiles of a few rows; forward and input gradient
    ("lcorr", 34, 24, 130, (3, 3), (20, 41), (1, 1), (1, 1), (1, 1), (1, 1)),
    ("mcorr", 9, 24, 100, (4, 3), (90, 41), (1, 1), (1, 1), (1, 1), (45, 1)),
    ("lcorr", 34, 130, 24, (3, 3), (20, 41), (1, 1), (1, 1), (1, 1), (1, 1)),
    ("mcorr", 9, 100, 24, (4, 3), (90, 41), (1, 1), (1, 1), (1, 1), (45, 1)),
    # small images on Mellin axes, whose input gradients' tiles take an output row of several images: more tiles than
    # workgroups, wavefronts sharing a tile, slices of the contracted channels, images ending inside tiles, rows of one column
    ("mcorr", 200, 64, 64, (5, 3), (10, 41), (1, 1), (1, 1), (2, 1), (4, 1)),
    ("mcorr", 1177, 64, 64, (5, 3), (5, 41), (1, 1), (6, 1), (2, 1), (0, 1)),
    ("mcorr", 300, 32, 96, (3, 3), (5, 40), (1, 1), (1, 1), (1, 1), (2, 1)),
    ("mcorr", 300, 32, 128, (3, 3), (5, 40), (1, 1), (1, 1), (1, 1), (2, 1)),
    ("mcorr", 400, 40, 32, (5, 3), (7, 13), (1, 1), (1, 1), (2, 1), (3, 1)),
    ("mcorr", 900, 32, 32, (5, 1), (11, 1), (1, 1), (2, 1), (2, 0), (2, 0)),
    ("mcorr", 9, 128, 128, (4, 4), (12, 10), (1, 1), (1, 1), (1, 1), (6, 2)),
    ("mcorr", 4, 32, 96, (5, 3), (7, 3), (1, 1), (1, 1), (0, 1), (2, 1)),
    ("mcorr", 300, 96, 256, (5, 2), (7, 3), (1, 1), (1, 1), (2, 1), (2, 1)),
    ("mcorr", 300, 32, 64, (4, 4), (12, 20), (1, 1), (1, 1), (1, 1), (4, 1)),
    ("mcorr", 60, 128, 128, (5, 2), (7, 20), (1, 1), (1, 1), (0, 1), (2, 1)),
]
#: what a case is there for: (case, element bytes, input gradient, words of its plan)
REACHED = [
    (0, 4, 0, dict(wm=2)), (1, 4, 0, dict(wm=2)), (2, 4, 1, dict(wm=2)), (3, 4, 1, dict(wm=2)),
    (4, 4, 1, dict(joint=1, wk=1)), (4, 2, 1, dict(joint=1, wk=1)), (5, 4, 1, dict(joint=1, wk=1)), (5, 2, 1, dict(joint=1, nt=4)),
    (6, 4, 1, dict(joint=1)), (6, 2, 1, dict(joint=1)), (7, 4, 1, dict(joint=1, whole=0, slices=2)), (7, 2, 1, dict(joint=1)),
    (9, 4, 1, dict(joint=1, wk=4)), (9, 2, 1, dict(joint=1, wk=4)), (10, 2, 1, dict(joint=1, wk=4)),
    (11, 4, 1, dict(joint=1, wk=4, whole=0)), (12, 2, 1, dict(joint=1, whole=0)), (13, 4, 1, dict(joint=1, whole=512, slices=4)),
    (14, 4, 1, dict(joint=1, wm=2, whole=0)),
]


def dims_of(case):
    op, n, c_in, c_out, nf, ng, s, d, p, r = case
    valid = mconv.mcorr_valid_size if op == "mcorr" else mconv.lcorr_valid_size
    return [n, c_in, c_out, *nf, *ng, valid(nf[0], ng[0], s[0], d[0], p[0]) + r[0],
            mconv.lcorr_valid_size(nf[1], ng[1], s[1], d[1], p[1]) + r[1], *s, *d, *p, 1, 1]


@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_tile_shapes_match_checker(case, half):
    op, n, c_in, c_out, nf, ng, s, d, p, r = case
    rng = np.random.default_rng(7300 + CASES.index(case))
    for which, elem_bytes, gradient, words in REACHED:
        if which == CASES.index(case) and elem_bytes == (2 if half else 4):
            got = plan(hip.AX_MCORR if op == "mcorr" else hip.AX_LCORR, elem_bytes, gradient, dims_of(case))
            assert words.items() <= got.items(), got
    kind = np.float16 if half else np.float32
    x = rng.standard_normal((n, c_in) + ng).astype(kind)
    w = (rng.standard_normal((c_out, c_in) + nf) * (c_in * nf[0] * nf[1]) ** -0.5).astype(kind)
    b = rng.standard_normal(c_out).astype(kind)
    fwd = oracle.mcorrlcorr if op == "mcorr" else oracle.lcorrlcorr
    bwd = oracle.mcorrlcorr_backward if op == "mcorr" else oracle.lcorrlcorr_backward
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    exp = fwd(x64, w64, b.astype(np.float64), s, d, p, (1, 1), r)
    go = rng.standard_normal(exp.shape).astype(kind)
    egi, egw, egb = bwd(x64, w64, go.astype(np.float64), s, d, p, (1, 1))
    if egb is None:
        egb = go.astype(np.float64).sum((0, 2, 3))
    xg, wg, bg = (to_gpu(a).requires_grad_() for a in (x, w, b))
    out = (mconv._ext_mcorrlcorr if op == "mcorr" else mconv._ext_lcorrlcorr)(xg, wg, bg, s, d, p, (1, 1), r)
    assert hip.last_variant() == ("mfma-f16-blocks" if half else "mfma-blocks")
    out.backward(to_gpu(go))
    taps, positions = nf[0] * nf[1], n * exp.shape[2] * exp.shape[3]
    for got, ref, fan, what in ((out, exp, c_in * taps, "out"), (xg.grad, egi, c_out * taps, "grad_input"),
                                (wg.grad, egw, positions, "grad_weight"), (bg.grad, egb, positions, "grad_bias")):
        if half:                                       # one rounding of a result whose sum has an error of its own
            err = np.abs(got.detach().double().cpu().numpy() - ref)
            assert np.all(err <= 2.0 ** -10 * np.abs(ref) + 2e-5 * fan ** 0.5), what
        else:
            assert_close(got, ref, fan, what)


#: tiles of channels of filters of a megabyte and more, whose workgroups share XCDs
DEALT = {(256, 128): 2, (256, 256): 4, (64, 512): 8, (128, 500): 8}


@pytest.mark.parametrize("case", [
    # several tiles of channels dealt to the XCDs (two, four and eight of them: DEALT), position tiles that do not divide evenly;
    # two workgroups a CU by slices; sixteen tiles and fifteen, which are not
    ("mcorr", 1, 256, 128, (4, 4), (61, 5), (1, 1), (1, 1), (1, 1), (31, 2)),
    ("mcorr", 1, 256, 256, (4, 4), (337, 5), (1, 1), (1, 1), (1, 1), (169, 2)),
    ("lcorr", 1, 128, 512, (3, 3), (30, 9), (1, 1), (1, 1), (1, 1), (1, 1)),
    ("lcorr", 1, 128, 450, (3, 3), (7, 5), (1, 1), (1, 1), (1, 1), (1, 1)),
    # tiles of 32 channels for an odd number of them
    ("lcorr", 2, 64, 67, (4, 4), (60, 40), (1, 1), (1, 1), (1, 1), (1, 1)),
    ("mcorr", 1, 96, 160, (3, 3), (50, 20), (1, 1), (1, 1), (1, 1), (25, 1)),
    ("lcorr", 24, 48, 90, (3, 3), (60, 40), (1, 1), (1, 1), (1, 1), (1, 1)),
    # eight tiles of 64 channels, whole and in slices, the last of them not full
    ("mcorr", 1, 64, 512, (5, 3), (61, 20), (1, 1), (1, 1), (2, 1), (30, 1)),
    ("mcorr", 1, 128, 500, (4, 4), (30, 9), (1, 1), (1, 1), (1, 1), (15, 2)),
], ids=str)
def test_channel_tiles_match_checker(case):
    op, n, c_in, c_out, nf, ng, s, d, p, r = case
    words = plan(hip.AX_MCORR if op == "mcorr" else hip.AX_LCORR, 4, 0, dims_of(case))
    tiles = -(-c_out // (32 * words["mt"] * words["wm"]))
    if (c_in, c_out) in DEALT:
        assert words["wk"] == 4 and tiles == DEALT[c_in, c_out] and 6 * 32 * tiles * words["mt"] * c_in * nf[0] * nf[1] >= 1 << 20, words
    else:
        assert words["mt"] == 1, words
    rng = np.random.default_rng(7400 + c_out)
    x = rng.standard_normal((n, c_in) + ng).astype(np.float32)
    w = (rng.standard_normal((c_out, c_in) + nf) * (c_in * nf[0] * nf[1]) ** -0.5).astype(np.float32)
    fwd = oracle.mcorrlcorr if op == "mcorr" else oracle.lcorrlcorr
    exp = fwd(x.astype(np.float64), w.astype(np.float64), None, s, d, p, (1, 1), r)
    out = (mconv._ext_mcorrlcorr if op == "mcorr" else mconv._ext_lcorrlcorr)(to_gpu(x), to_gpu(w), None, s, d, p, (1, 1), r)
    assert hip.last_variant() == "mfma-blocks"
    assert_close(out, exp, c_in * nf[0] * nf[1], "out")
