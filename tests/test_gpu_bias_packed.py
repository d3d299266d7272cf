"""Bias gradients of layers with few channels whose input gradient is the blocked kernels': added up by the pass that blocks
grad_out."""
import numpy as np
import pytest
import torch

import _mellin_hip as hip
import mconv
from _gpu import assert_close, to_gpu
from test_block_plans import BIAS_PACKED, WANT_BIAS, WANT_INPUT, WANT_RELU, WANT_WEIGHT, bias_route

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["f32", "f16", "amp"])
@pytest.mark.parametrize("relu", [False, True], ids=["plain", "relu"])
@pytest.mark.parametrize("shape", [(4, 1, 125, 774), (3, 2, 17, 61), (1, 5, 40, 300)], ids=str)
def test_bias_gradient_beside_blocked_input_gradient(shape, relu, kind):
    n, c_in, c_out, t = shape
    rng = np.random.default_rng(9300 + c_out)
    size = np.float16 if kind == "f16" else np.float32
    x = rng.standard_normal((n, c_in, t)).astype(size)
    w = (rng.standard_normal((c_out, c_in, 8)) * (8 * c_in) ** -0.5).astype(size)
    b = rng.standard_normal(c_out).astype(size)
    xg, wg, bg = (to_gpu(a).requires_grad_() for a in (x, w, b))
    with torch.autocast("cuda", torch.float16, enabled=kind == "amp"):
        out = mconv._ext_mcorr1d(xg, wg, bg, 1, 2, 1, 1, 0, "relu" if relu else None)
    assert bias_route(hip.AX_MCORR, 4 if kind == "f32" else 2, WANT_INPUT | WANT_WEIGHT | WANT_BIAS | (WANT_RELU if relu else 0),
                      [n, c_in, c_out, 8, 1, t, 1, out.shape[2], 1, 1, 1, 2, 1, 1, 0, 1, 1]) == BIAS_PACKED
    go = to_gpu(rng.standard_normal(tuple(out.shape)).astype(np.float16 if out.dtype == torch.float16 else np.float32))
    out.backward(go)
    g = go.double().cpu().numpy() * ((out.detach() > 0).cpu().numpy() if relu else 1)
    ref = g.sum((0, 2))
    if kind == "f32":
        assert_close(bg.grad, ref, g.shape[0] * g.shape[2], "grad_bias")
    else:                                              # one rounding of a sum that has an error of its own
        err = np.abs(bg.grad.double().cpu().numpy() - ref)
        assert np.all(err <= 2.0 ** -10 * np.abs(ref) + 2e-5 * (g.shape[0] * g.shape[2]) ** 0.5)
