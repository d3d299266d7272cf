"""The channel-blocked weight gradient's walk over images, rows and columns (its carries from stage to stage), and slices for
more than two workgroups a CU: against the float64 checker."""
import numpy as np
import pytest
import torch

import _mellin_hip as hip
import mconv
from _gpu import assert_close, to_gpu
from oracle import oracle

pytestmark = pytest.mark.gpu

CASES = [
    # (op, n, c_in, c_out, nf, ng, s, d, p, u, r); a stage is 32 positions in fp32, 64 in half
    ("lcorr", 70, 16, 32, (2, 1), (4, 1), (1, 1), (1, 1), (1, 0), (1, 1), (1, 0)),    # a stage of several images, one column
    ("lcorr", 41, 24, 40, (2, 3), (2, 5), (2, 1), (1, 1), (0, 1), (1, 1), (0, 1)),    # one row an image
    ("lcorr", 5, 16, 32, (3, 3), (9, 32), (1, 1), (1, 1), (1, 1), (1, 1), (1, 1)),    # rows of a stage and of half a stage
    ("lcorr", 3, 16, 32, (3, 3), (7, 64), (1, 1), (1, 1), (1, 1), (1, 1), (1, 1)),
    ("lcorr", 3, 32, 64, (2, 4), (11, 33), (1, 1), (1, 2), (0, 3), (1, 1), (0, 0)),
    ("lcorr", 3, 32, 33, (2, 4), (11, 65), (2, 1), (1, 1), (0, 1), (1, 1), (0, 0)),
    ("lcorr", 6, 16, 32, (3, 1), (8, 50), (1, 3), (1, 1), (1, 0), (1, 1), (1, 0)),    # strides past the filter's reach
    ("lcorr", 6, 16, 32, (3, 2), (8, 60), (1, 5), (1, 1), (1, 0), (1, 1), (1, 0)),
    ("lcorr", 4, 16, 32, (3, 3), (8, 21), (1, 1), (1, 1), (1, 1), (1, 2), (1, 2)),    # upsampled columns
    ("mcorr", 9, 32, 32, (5, 3), (12, 13), (1, 1), (1, 1), (2, 1), (1, 1), (5, 1)),   # filter rows of different counts
    ("mcorr", 150, 24, 40, (5, 3), (3, 7), (1, 1), (1, 1), (2, 1), (1, 1), (1, 1)),
    ("lcorr", 8, 32, 32, (4, 4), (200, 41), (1, 1), (1, 1), (1, 1), (1, 1), (1, 1)),  # four workgroups a CU
    ("mcorr", 8, 32, 64, (4, 4), (300, 41), (1, 1), (1, 1), (1, 1), (1, 1), (150, 1)),
]


@pytest.mark.parametrize("half", [False, True], ids=["f32", "f16"])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_weight_gradient_matches_checker(case, half):
    op, n, c_in, c_out, nf, ng, s, d, p, u, r = case
    rng = np.random.default_rng(8800 + CASES.index(case))
    kind = np.float16 if half else np.float32
    x = rng.standard_normal((n, c_in) + ng).astype(kind)
    w = (rng.standard_normal((c_out, c_in) + nf) * (c_in * nf[0] * nf[1]) ** -0.5).astype(kind)
    xg, wg = to_gpu(x), to_gpu(w).requires_grad_()
    out = (mconv._ext_mcorrlcorr if op == "mcorr" else mconv._ext_lcorrlcorr)(xg, wg, None, s, d, p, u, r)
    go = rng.standard_normal(tuple(out.shape)).astype(kind)
    bwd = oracle.mcorrlcorr_backward if op == "mcorr" else oracle.lcorrlcorr_backward
    ref = bwd(x.astype(np.float64), w.astype(np.float64), go.astype(np.float64), s, d, p, u)[1]
    out.backward(to_gpu(go))
    assert hip.last_variant() == ("mfma-f16-blocks" if half else "mfma-blocks")
    positions = n * out.shape[2] * out.shape[3]
    if half:                                           # one rounding of a result whose sum has an error of its own
        err = np.abs(wg.grad.double().cpu().numpy() - ref)
        assert np.all(err <= 2.0 ** -10 * np.abs(ref) + 2e-5 * positions ** 0.5)
    else:
        assert_close(wg.grad, ref, positions, "grad_weight")
