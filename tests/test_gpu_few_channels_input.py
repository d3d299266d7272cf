"""Input gradients of layers with few input channels that go through the channel-blocked kernels because nothing else suits
them -- more than 128 output channels, filters of a few taps, one column, half precision on linear axes -- against the float64
checker, with the weight and bias gradients that other kernels make in the same call."""
import numpy as np
import pytest
import torch

import _mellin_hip as hip
import mconv
from _gpu import assert_close, to_gpu
from oracle import oracle

pytestmark = pytest.mark.gpu

CASES = [
    # (op, n, c_in, c_out, nf, ng, s, d, p, r, half)
    ("lcorr", 3, 1, 171, (3, 4), (112, 41), (1, 1), (1, 1), (0, 1), (0, 1), False),   # more than 128 output channels
    ("mcorr", 2, 3, 146, (4, 3), (150, 41), (1, 1), (1, 1), (3, 1), (0, 1), False),
    ("lcorr", 3, 5, 110, (3, 2), (300, 41), (1, 1), (2, 1), (0, 0), (0, 0), False),   # six taps of a tile's 32 rows
    ("lcorr", 9, 6, 16, (3, 3), (324, 38), (1, 1), (1, 1), (2, 0), (2, 0), False),    # taps in no whole eights
    ("lcorr", 4, 3, 9, (5, 3), (177, 41), (2, 1), (1, 1), (1, 0), (1, 0), False),
    ("mcorr", 28, 3, 156, (14, 1), (203, 1), (1, 1), (1, 1), (0, 0), (0, 0), False),  # one column
    ("lcorr", 24, 7, 86, (9, 1), (193, 1), (1, 1), (1, 1), (3, 0), (3, 0), False),
    ("lcorr", 5, 1, 45, (3, 4), (553, 41), (1, 1), (1, 1), (0, 1), (0, 1), True),     # half, linear
    ("lcorr", 4, 5, 46, (4, 3), (439, 41), (1, 1), (1, 1), (0, 0), (0, 0), True),
    ("lcorr", 3, 3, 170, (7, 2), (297, 41), (2, 1), (2, 1), (2, 0), (2, 0), True),
]


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_input_gradients_of_few_channels_match_checker(case):
    op, n, c_in, c_out, nf, ng, s, d, p, r, half = case
    rng = np.random.default_rng(8200 + CASES.index(case))
    kind = np.float16 if half else np.float32
    x = rng.standard_normal((n, c_in) + ng).astype(kind)
    w = (rng.standard_normal((c_out, c_in) + nf) * (c_out * nf[0] * nf[1]) ** -0.5).astype(kind)
    xg, wg, bg = to_gpu(x).requires_grad_(), to_gpu(w).requires_grad_(), torch.zeros(c_out, device="cuda", dtype=torch.float16 if half else torch.float32, requires_grad=True)
    out = (mconv._ext_mcorrlcorr if op == "mcorr" else mconv._ext_lcorrlcorr)(xg, wg, bg, s, d, p, (1, 1), r)
    go = rng.standard_normal(tuple(out.shape)).astype(kind)
    out.backward(to_gpu(go))
    assert hip.last_variant() == ("mfma-f16-blocks" if half else "mfma-blocks")
    bwd = oracle.mcorrlcorr_backward if op == "mcorr" else oracle.lcorrlcorr_backward
    go64 = go.astype(np.float64)
    egi, egw, _ = bwd(x.astype(np.float64), w.astype(np.float64), go64, s, d, p, (1, 1))
    taps, positions = nf[0] * nf[1], n * out.shape[2] * out.shape[3]
    for got, ref, fan, what in ((xg.grad, egi, c_out * taps, "grad_input"), (wg.grad, egw, positions, "grad_weight"),
                                (bg.grad, go64.sum((0, 2, 3)), positions, "grad_bias")):
        if half:
            err = np.abs(got.detach().double().cpu().numpy() - ref)
            assert np.all(err <= 2.0 ** -10 * np.abs(ref) + 2e-5 * fan ** 0.5), what
        else:
            assert_close(got, ref, fan, what)
