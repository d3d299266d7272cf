"""Bias gradients of float layers with few input channels, which their weight gradient's kernels add up beside it, against
float64 sums: rows around whole groups of eight outputs, odd rows, channels around whole tiles of 32, several column blocks,
units of a part of their rows, and layers that keep the launch of its own (rows past the filter's support)."""
import numpy as np
import pytest
import torch

import _mellin_hip as hip
import mconv
from _gpu import assert_close, to_gpu
from oracle import oracle
from test_block_plans import BIAS_BESIDE_WEIGHT, BIAS_OWN, WANT_BIAS, WANT_WEIGHT, bias_route

pytestmark = pytest.mark.gpu

CASES = [
    # (op, n, c_in, c_out, nf, ng, p, r); the first eight are long enough for the kernels of few channels
    ("lcorr", 6, 3, 64, (8, 4), (300, 41), (0, 0), (0, 0)),          # rows of 38: the last group shares two with the one before
    ("lcorr", 5, 3, 70, (8, 4), (400, 19), (0, 0), (0, 0)),          # whole groups of eight; a third tile of six channels
    ("lcorr", 7, 1, 97, (3, 3), (333, 40), (1, 1), (1, 1)),
    ("lcorr", 9, 5, 33, (5, 3), (210, 11), (0, 0), (0, 0)),          # rows of nine: seven shared; J = 75
    ("lcorr", 4, 14, 40, (5, 4), (207, 43), (2, 1), (2, 2)),         # J = 280: three column blocks, of which the first adds up
    ("mcorr", 9, 3, 64, (8, 4), (301, 41), (0, 0), (0, 0)),
    ("mcorr", 5, 7, 50, (6, 2), (400, 20), (1, 0), (0, 0)),          # odd rows of 19
    ("mcorr", 6, 2, 129, (3, 3), (200, 41), (0, 1), (0, 1)),
    ("mcorr", 4, 3, 64, (4, 4), (200, 41), (1, 1), (100, 1)),        # more rows than whole filters reach
    ("mcorr", 4, 3, 64, (4, 4), (200, 41), (1, 1), (350, 1)),        # rows past the support: a launch of its own
]
#: where a bias gradient wanted with the weight gradient is made
ROUTES = 9 * [BIAS_BESIDE_WEIGHT] + [BIAS_OWN]


@pytest.mark.parametrize("offset", [0.0, 3.0], ids=["centred", "offset"])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_bias_gradient_beside_the_weight_gradient(case, offset):
    op, n, c_in, c_out, nf, ng, p, r = case
    rng = np.random.default_rng(4100 + CASES.index(case))
    x = rng.standard_normal((n, c_in) + ng).astype(np.float32)
    w = rng.standard_normal((c_out, c_in) + nf).astype(np.float32)
    xg, wg, bg = to_gpu(x), to_gpu(w).requires_grad_(), torch.zeros(c_out, device="cuda", requires_grad=True)
    out = (mconv._ext_mcorrlcorr if op == "mcorr" else mconv._ext_lcorrlcorr)(xg, wg, bg, (1, 1), (1, 1), p, (1, 1), r)
    assert bias_route(hip.AX_MCORR if op == "mcorr" else hip.AX_LCORR, 4, WANT_WEIGHT | WANT_BIAS,
                      [n, c_in, c_out, *nf, *ng, *out.shape[2:], 1, 1, 1, 1, *p, 1, 1]) == ROUTES[CASES.index(case)]
    go = (rng.standard_normal(tuple(out.shape)) + offset).astype(np.float32)
    out.backward(to_gpu(go))
    go64 = go.astype(np.float64)
    bwd = oracle.mcorrlcorr_backward if op == "mcorr" else oracle.lcorrlcorr_backward
    egw = bwd(x.astype(np.float64), w.astype(np.float64), go64, (1, 1), (1, 1), p, (1, 1))[1]
    positions = n * out.shape[2] * out.shape[3]
    assert_close(wg.grad, egw, positions, "grad_weight")
    # a lane adds some hundred values in turn, then sums of lanes, wavefronts and workgroups follow: 2^-24 a step of what has
    # been added so far, of 300 steps at most
    err = np.abs(bg.grad.double().cpu().numpy() - go64.sum((0, 2, 3)))
    assert np.all(err <= 300 * 2.0 ** -24 * np.abs(go64).sum((0, 2, 3))), err.max()


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_weight_gradient_has_the_same_bits_without_a_bias(case):
    """A weight gradient without a bias is a kernel of its own, without the sums, on the same tiles."""
    op, n, c_in, c_out, nf, ng, p, r = case
    torch.manual_seed(4200 + CASES.index(case))
    x, w = torch.randn(n, c_in, *ng, device="cuda"), torch.randn(c_out, c_in, *nf, device="cuda", requires_grad=True)
    b = torch.zeros(c_out, device="cuda", requires_grad=True)
    layer = mconv._ext_mcorrlcorr if op == "mcorr" else mconv._ext_lcorrlcorr
    outs = [layer(x, w, bias, (1, 1), (1, 1), p, (1, 1), r) for bias in (b, None)]
    go = torch.randn_like(outs[0])
    assert torch.equal(torch.autograd.grad(outs[0], (w, b), go)[0], torch.autograd.grad(outs[1], w, go)[0])
