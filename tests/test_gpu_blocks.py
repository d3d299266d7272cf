"""The channel-blocked kernels behind the layers (forward, input gradient, weight gradient, bias
gradient with the backward of a fused ReLU) against the float64 checker, at the sizes where they
can go wrong: channel counts around whole groups of eight and tiles of 32, last tiles and stages of
positions, stages of an odd number of halves, subsets of filter rows on a Mellin axis, few tiles
(wavefronts sharing a tile's steps), stages that run across images."""
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
    ("lcorr", 1, 16, 1, (3, 3), (5, 4), (1, 1), (1, 1), (1, 1), (1, 1)),            # one output channel, 20 positions
    ("lcorr", 3, 17, 33, (3, 3), (19, 13), (1, 1), (2, 1), (2, 1), (2, 1)),         # 27 halves; one channel past a group, one past a tile
    ("mcorr", 2, 24, 65, (5, 3), (60, 7), (1, 1), (1, 1), (2, 1), (20, 1)),         # three classes, rows past the support
    ("mcorr", 2, 64, 32, (4, 4), (90, 41), (1, 1), (1, 1), (1, 1), (45, 1)),        # two subsets of filter rows in a stage's LDS
    ("mcorr", 5, 41, 70, (16, 1), (97, 1), (2, 1), (1, 1), (3, 0), (5, 0)),         # 1-D, sixteen filter rows, stride
    ("lcorr", 4, 40, 128, (2, 4), (33, 64), (1, 2), (1, 2), (1, 3), (0, 2)),        # y stride and dilation; 128 channels (two wavefronts along them)
    ("lcorr", 2, 130, 100, (1, 1), (9, 8), (1, 1), (1, 1), (0, 0), (0, 0)),         # one tap, 17 groups
    ("mcorr", 70, 16, 36, (3, 2), (10, 3), (1, 1), (2, 1), (1, 0), (2, 0)),         # small images: stages run across several
    ("lcorr", 2, 48, 34, (3, 4), (25, 2), (1, 1), (1, 1), (1, 1), (1, 1)),          # filter columns without a tap
    ("lcorr", 40, 32, 96, (4, 4), (48, 20), (1, 1), (1, 1), (1, 1), (2, 2)),        # enough tiles for the widest tile shapes
]


@pytest.mark.parametrize("kinds", [(np.float32, np.float32), (np.float16, np.float16), (np.float16, np.float32)], ids=["f32", "f16", "amp"])
@pytest.mark.parametrize("relu", [False, True], ids=["plain", "relu"])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_blocked_layers_match_checker(case, kinds, relu):
    op, n, c_in, c_out, nf, ng, s, d, p, r = case
    rng = np.random.default_rng(5100 + CASES.index(case))
    kind, param_kind = kinds                           # tensors; parameters (float ones under autocast: rounded to half)
    half = kind is np.float16
    x = rng.standard_normal((n, c_in) + ng).astype(kind)
    w = (rng.standard_normal((c_out, c_in) + nf) * (c_in * nf[0] * nf[1]) ** -0.5).astype(kind)
    b = rng.standard_normal(c_out).astype(kind)
    fwd = oracle.mcorrlcorr if op == "mcorr" else oracle.lcorrlcorr
    bwd = oracle.mcorrlcorr_backward if op == "mcorr" else oracle.lcorrlcorr_backward
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    exp = fwd(x64, w64, b.astype(np.float64), s, d, p, (1, 1), r)
    nh = exp.shape[2:]
    go = rng.standard_normal(exp.shape).astype(kind)
    xg, wg, bg = (to_gpu(a).requires_grad_() for a in (x, w.astype(param_kind), b.astype(param_kind)))
    call = mconv._ext_mcorrlcorr if op == "mcorr" else mconv._ext_lcorrlcorr
    with torch.autocast("cuda", torch.float16, enabled=kind is not param_kind):
        out = call(xg, wg, bg, s, d, p, (1, 1), r, activation="relu" if relu else None)
    assert hip.last_variant() == ("mfma-f16-blocks" if half else "mfma-blocks")
    out.backward(to_gpu(go))
    assert hip.last_variant() == ("mfma-f16-blocks" if half else "mfma-blocks")
    masked = go.astype(np.float64)
    if relu:
        exp = np.maximum(exp, 0)
        masked = masked * (out.detach().float().cpu().numpy() > 0)       # the mask the layer itself applied
    egi, egw, egb = bwd(x64, w64, masked, s, d, p, (1, 1))
    if egb is None:
        egb = masked.sum((0, 2, 3))
    for got, ref, fan, what in ((out, exp, c_in * nf[0] * nf[1], "out"), (xg.grad, egi, c_out * nf[0] * nf[1], "grad_input"),
                                (wg.grad, egw, n * nh[0] * nh[1], "grad_weight"), (bg.grad, egb, n * nh[0] * nh[1], "grad_bias")):
        if half:
            err = np.abs(got.detach().double().cpu().numpy() - ref)
            assert np.all(err <= 2.0 ** -10 * np.abs(ref) + 2e-5 * fan ** 0.5), what
        else:
            assert_close(got, ref, fan, what)


@pytest.mark.parametrize("case", [(2, 64, 32, (4, 4), (70, 21)), (2, 64, 64, (4, 4), (70, 21)), (24, 32, 96, (3, 3), (40, 20))],
                         ids=["32 channels", "64 channels", "many tiles"])
def test_long_float_sums_are_rounded_once_in_sixteen_products(case):
    """The small products of the bf16 parts have sums of their own, so a sum of n products is rounded n / 16 times, each time
    by 2^-24 / sqrt(3) at most in the mean square, of a partial sum that grows with the root of the products: 2^-24 sqrt(n / 96)
    in the 2-norm, doubled for the partial sums that are added behind it, and 2^-23 for the products themselves."""
    n, c_in, c_out, nf, ng = case
    rng = np.random.default_rng(91)
    x = rng.standard_normal((n, c_in) + ng).astype(np.float32)
    w = rng.standard_normal((c_out, c_in) + nf).astype(np.float32)
    exp = oracle.lcorrlcorr(x.astype(np.float64), w.astype(np.float64), None, (1, 1), (1, 1), (1, 1), (1, 1), (1, 1))
    go = rng.standard_normal(exp.shape).astype(np.float32)
    egi, egw, _ = oracle.lcorrlcorr_backward(x.astype(np.float64), w.astype(np.float64), go.astype(np.float64), (1, 1), (1, 1), (1, 1), (1, 1))
    xg, wg = to_gpu(x).requires_grad_(), to_gpu(w).requires_grad_()
    out = mconv._ext_lcorrlcorr(xg, wg, None, (1, 1), (1, 1), (1, 1), (1, 1), (1, 1))
    assert hip.last_variant() == "mfma-blocks"
    out.backward(to_gpu(go))
    taps = nf[0] * nf[1]
    for got, ref, terms in ((out, exp, c_in * taps), (xg.grad, egi, c_out * taps), (wg.grad, egw, n * exp.shape[2] * exp.shape[3])):
        err = np.linalg.norm(got.detach().double().cpu().numpy() - ref) / np.linalg.norm(ref)
        assert err <= 2.0 ** -24 * (2 * (terms / 96) ** 0.5 + 2), (err, terms)


def test_blocked_passes_repeat_bit_for_bit_and_replay_in_a_graph():
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(3, 24, 50, 21, device="cuda", generator=gen)
    w = torch.randn(40, 24, 4, 4, device="cuda", generator=gen) * 0.05
    dims = hip._dims(3, 24, 40, (4, 4), (50, 21), (50, 21), (1, 1), (1, 1), (1, 1), (1, 1))
    go = torch.randn(3, 40, 50, 21, device="cuda", generator=gen)
    want = 1 | 2 | 4
    nf = hip.lib.mellin_layer_forward_workspace(hip.AX_MCORR, 4, *dims)
    nb = hip.lib.mellin_layer_backward_workspace(hip.AX_MCORR, 4, want, *dims)
    ws = torch.empty(max(nf, nb), dtype=torch.uint8, device="cuda")
    out, gi, gw, gb = torch.empty_like(go), torch.empty_like(x), torch.empty_like(w), torch.empty(40, device="cuda")

    def both():
        st = hip._stream(x.device)
        hip._check(hip.lib.mellin_layer_forward(hip.AX_MCORR, 4, 0, hip._dp(x), hip._dp(w), None, *dims, hip._dp(out), None, hip._dp(ws), nf, st))
        hip._check(hip.lib.mellin_layer_backward(hip.AX_MCORR, 4, want, hip._dp(x), hip._dp(w), hip._dp(go), None, *dims, hip._dp(gi),
                                                 hip._dp(gw), hip._dp(gb), hip._dp(ws), nb, st))
    both()
    eager = [t.clone() for t in (out, gi, gw, gb)]
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        both()
        with torch.cuda.graph(graph, stream=stream):
            both()
    for _ in range(3):
        for t in (out, gi, gw, gb):
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, t) for a, t in zip(eager, (out, gi, gw, gb)))
        both()


@pytest.mark.parametrize("op,half,relu", [("lcorr", False, True), ("mcorr", True, False)], ids=["f32", "amp"])
def test_layers_whose_blocked_tensors_would_be_huge_go_through_them_in_parts(op, half, relu):
    """Results of images of every part, and both sides of a part's end, as those of the images alone; the gradients of the
    parameters as those of a call that wants nothing else."""
    size = 2 if half else 4
    image = 2 * (1024 * 41 + 1) * (16 if half else 48)           # blocked bytes of an image of 16 channels
    n = 2 * ((4 << 30) // image) + 1                             # three parts
    per = -(-n // 3)
    gen = torch.Generator(device="cuda").manual_seed(9)
    dtype = torch.float16 if half else torch.float32
    x = torch.empty(n, 16, 1024, 41, device="cuda", dtype=dtype).normal_(generator=gen).requires_grad_()
    w = (torch.randn(16, 16, 3, 3, device="cuda", generator=gen) / 12).requires_grad_()
    b = torch.randn(16, device="cuda", generator=gen).requires_grad_()
    call = mconv._ext_mcorrlcorr if op == "mcorr" else mconv._ext_lcorrlcorr
    r = (512, 1) if op == "mcorr" else (1, 1)

    def passes(x):
        with torch.autocast("cuda", torch.float16, enabled=half):
            return call(x, w, b, (1, 1), (1, 1), (1, 1), (1, 1), r, activation="relu" if relu else None)

    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    out = passes(x)
    torch.cuda.synchronize()
    assert torch.cuda.max_memory_allocated() - before <= out.numel() * size + (5 << 30)
    assert hip.last_variant() == ("mfma-f16-blocks" if half else "mfma-blocks")
    go = torch.empty_like(out).normal_(std=0.1, generator=gen)   # (parameters' gradients in half stay finite)
    gi, gw, gb = torch.autograd.grad(out, (x, w, b), go, retain_graph=True)
    assert all(torch.equal(g, alone) for g, alone in zip((gw, gb), torch.autograd.grad(out, (w, b), go)))
    tol = 1e-3 if half else 1e-6
    for i in (0, per - 1, per, 2 * per - 1, 2 * per, n - 1):
        xi = x[i:i + 1].detach().clone().requires_grad_()
        oi = passes(xi)
        gii, = torch.autograd.grad(oi, xi, go[i:i + 1])
        assert float((oi - out[i:i + 1]).detach().double().norm() / oi.detach().double().norm()) <= tol
        # (another order of summation may pass a value within its rounding error of the ReLU's kink: 1.7e-3 of the gradient)
        assert float((gii - gi[i:i + 1]).double().norm() / gii.double().norm()) <= (5e-3 if relu else tol)


def test_layer_entry_points_refuse_what_they_cannot_do():
    dims = hip._dims(2, 16, 8, (3, 3), (9, 9), (7, 7), (1, 1), (1, 1), (0, 0), (1, 1))
    x, w, out = torch.zeros(2, 16, 9, 9, device="cuda"), torch.zeros(8, 16, 3, 3, device="cuda"), torch.zeros(2, 8, 7, 7, device="cuda")
    need = hip.lib.mellin_layer_forward_workspace(hip.AX_LCORR, 4, *dims)
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    call = hip.lib.mellin_layer_forward
    assert call(hip.AX_LCORR, 8, 0, hip._dp(x), hip._dp(w), None, *dims, hip._dp(out), None, hip._dp(ws), need, None) == 1
    assert call(hip.AX_LCORR, 4, 0, hip._dp(x), hip._dp(w), None, *dims, hip._dp(out), None, hip._dp(ws), need - 1, None) == 3
    assert call(hip.AX_LCORR, 4, 7, hip._dp(x), hip._dp(w), None, *dims, hip._dp(out), None, hip._dp(ws), need, None) == 1
    assert call(hip.AX_LCORR, 4, 0, None, hip._dp(w), None, *dims, hip._dp(out), None, hip._dp(ws), need, None) == 1
    back = hip.lib.mellin_layer_backward
    assert back(hip.AX_LCORR, 4, hip_want_input := 1, hip._dp(x), hip._dp(w), hip._dp(out), None, *dims, None, None, None, None, 0, None) == 1
    nb = hip.lib.mellin_layer_backward_workspace(hip.AX_LCORR, 4, hip_want_input, *dims)
    assert back(hip.AX_LCORR, 4, hip_want_input, hip._dp(x), hip._dp(w), hip._dp(out), None, *dims, hip._dp(x), None, None, hip._dp(ws), nb - 1, None) == 3
