"""Tile shapes of the channel-blocked matrix kernel that the layers of test_gpu_blocks.py are too small for: all three
gradients and the output against the float64 checker."""
import numpy as np
import pytest
import torch

import _mellin_hip as hip
import mconv
from _gpu import assert_close, to_gpu
from oracle import oracle

pytestmark = pytest.mark.gpu

CASES = [
    # (op, n, c_in, c_out, nf, ng, s, d, p, r)
    # fp32, two wavefronts along the channels (more than 96 channels, more workgroups than CUs): a second tile of two
    # channels, a first one that ends inside a tile of 32, last position tiles of a few rows; forward and input gradient
    ("lcorr", 34, 24, 130, (3, 3), (20, 41), (1, 1), (1, 1), (1, 1), (1, 1)),
    ("mcorr", 9, 24, 100, (4, 3), (90, 41), (1, 1), (1, 1), (1, 1), (45, 1)),
    ("lcorr", 34, 130, 24, (3, 3), (20, 41), (1, 1), (1, 1), (1, 1), (1, 1)),
    ("mcorr", 9, 100, 24, (4, 3), (90, 41), (1, 1), (1, 1), (1, 1), (45, 1)),
    # small images on Mellin axes, whose tiles take an output row of several images: more tiles than workgroups, wavefronts
    # sharing a tile, slices of the contracted channels (the last), images ending inside tiles, rows of one column
    ("mcorr", 200, 64, 64, (5, 3), (10, 41), (1, 1), (1, 1), (2, 1), (4, 1)),
    ("mcorr", 1177, 64, 64, (5, 3), (5, 41), (1, 1), (6, 1), (2, 1), (0, 1)),
    ("mcorr", 300, 32, 96, (3, 3), (5, 40), (1, 1), (1, 1), (1, 1), (2, 1)),
    ("mcorr", 300, 32, 128, (3, 3), (5, 40), (1, 1), (1, 1), (1, 1), (2, 1)),
    ("mcorr", 400, 40, 32, (5, 3), (7, 13), (1, 1), (1, 1), (2, 1), (3, 1)),
    ("mcorr", 900, 32, 32, (5, 1), (11, 1), (1, 1), (2, 1), (2, 0), (2, 0)),
    ("mcorr", 9, 128, 128, (4, 4), (12, 10), (1, 1), (1, 1), (1, 1), (6, 2)),
]


@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_tile_shapes_match_checker(case, half):
    op, n, c_in, c_out, nf, ng, s, d, p, r = case
    rng = np.random.default_rng(7300 + CASES.index(case))
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


@pytest.mark.parametrize("case", [
    # several tiles of channels dealt to the XCDs: two, four and eight of them, position tiles that do not divide evenly; two
    # workgroups a CU by slices
    ("mcorr", 1, 256, 128, (4, 4), (61, 5), (1, 1), (1, 1), (1, 1), (31, 2)),
    ("mcorr", 1, 256, 256, (4, 4), (337, 5), (1, 1), (1, 1), (1, 1), (169, 2)),
    ("lcorr", 1, 128, 512, (3, 3), (30, 9), (1, 1), (1, 1), (1, 1), (1, 1)),
    ("lcorr", 1, 128, 450, (3, 3), (7, 5), (1, 1), (1, 1), (1, 1), (1, 1)),
    # tiles of 32 channels for an odd number of them
    ("lcorr", 2, 64, 67, (4, 4), (60, 40), (1, 1), (1, 1), (1, 1), (1, 1)),
    ("mcorr", 1, 96, 160, (3, 3), (50, 20), (1, 1), (1, 1), (1, 1), (25, 1)),
    ("lcorr", 24, 48, 90, (3, 3), (60, 40), (1, 1), (1, 1), (1, 1), (1, 1)),
], ids=str)
def test_channel_tiles_match_checker(case):
    op, n, c_in, c_out, nf, ng, s, d, p, r = case
    rng = np.random.default_rng(7400 + c_out)
    x = rng.standard_normal((n, c_in) + ng).astype(np.float32)
    w = (rng.standard_normal((c_out, c_in) + nf) * (c_in * nf[0] * nf[1]) ** -0.5).astype(np.float32)
    fwd = oracle.mcorrlcorr if op == "mcorr" else oracle.lcorrlcorr
    exp = fwd(x.astype(np.float64), w.astype(np.float64), None, s, d, p, (1, 1), r)
    out = (mconv._ext_mcorrlcorr if op == "mcorr" else mconv._ext_lcorrlcorr)(to_gpu(x), to_gpu(w), None, s, d, p, (1, 1), r)
    assert hip.last_variant() == "mfma-blocks"
    assert_close(out, exp, c_in * nf[0] * nf[1], "out")
