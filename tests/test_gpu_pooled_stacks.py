"""Stack layers with pooling behind them, whose kernels store the maxima of pairs of columns themselves, and the input gradients
that are stored as those of the unpooled values, in every form that their endings take -- blocks of positions in ones, twos and
fours, channels that end inside a tile, wavefronts that share a tile or lie along the channels, slices of the contracted
channels, odd and even columns -- against the same layers called one by one: outputs bit for bit (the sums keep their order, and
equal halves the first of a pair), gradients within the bounds of tests/test_gpu_joint_stacks.py."""
import ctypes

import pytest
import torch

import _mellin_hip as hip
from conv_stack import ConvStack, ConvStackParams
from test_block_plans import WORDS, stack_dims

pytestmark = pytest.mark.gpu

CASES = [
    # (element bytes, Mellin, layers, kernel, channels, schedule, channel_factor, time_factor, batch, frames, bins), the pooled
    # layer's plan (2: its kernel pools)
    ((2, False, 4, (2, 1), 16, 2, 1, 2, 20, 100, 33), 2, dict(mt=1, nt=1, wk=1)),
    ((2, False, 3, (2, 1), 16, 3, 2, 2, 60, 10, 33), 2, dict(mt=1, nt=2, wk=4)),
    ((2, False, 4, (2, 1), 16, 3, 1, 2, 60, 400, 6), 2, dict(mt=1, nt=4)),
    ((2, False, 4, (5, 2), 128, 2, 1, 2, 1, 10, 41), 2, dict(mt=2, nt=1, wk=4, whole=0)),
    ((2, False, 3, (3, 1), 70, 2, 2, 2, 60, 200, 6), 2, dict(mt=2, nt=4, wm=2)),
    ((4, False, 3, (2, 1), 70, 2, 1, 2, 1, 100, 6), 2, dict(mt=1, nt=1, wk=1, whole=0)),
    ((4, False, 3, (4, 4), 20, 3, 1, 2, 1, 5, 5), 2, dict(mt=1, nt=1, wk=4)),
    ((4, False, 4, (2, 1), 70, 2, 1, 2, 9, 60, 41), 2, dict(mt=1, nt=2, whole=0)),
    ((4, False, 4, (5, 3), 64, 2, 1, 2, 1, 5, 20), 2, dict(mt=2, nt=1, wk=4, whole=0)),
    ((4, False, 4, (2, 1), 48, 3, 2, 1, 20, 100, 33), 2, dict(mt=2, nt=2)),
    ((4, False, 4, (2, 1), 70, 2, 2, 2, 60, 100, 6), 2, dict(mt=2, nt=2, wm=2)),
    ((2, True, 3, (2, 1), 16, 3, 2, 2, 20, 100, 41), 2, dict(mt=1, nt=2)),
    ((2, True, 3, (3, 1), 48, 3, 1, 2, 20, 100, 33), 2, dict(mt=2, nt=2)),
    ((4, True, 3, (4, 4), 70, 2, 1, 2, 1, 10, 10), 2, dict(mt=1, nt=1, whole=0)),
    ((4, True, 4, (4, 2), 20, 2, 2, 1, 60, 200, 7), 2, dict(mt=2, nt=2)),
    ((4, True, 4, (2, 1), 64, 2, 2, 1, 20, 100, 20), 2, dict(mt=2, nt=2, wm=2)),
    # an even number of columns: the same tiles, whatever the order of their sums depends on
    ((4, True, 3, (5, 3), 32, 3, 1, 2, 60, 60, 10), 2, dict(wk=1)),
    ((4, True, 4, (5, 1), 20, 3, 1, 2, 2, 5, 6), 2, dict(wk=4)),
    ((2, True, 3, (4, 4), 40, 3, 1, 1, 1, 70, 20), 2, dict(wk=4)),
    ((4, True, 3, (4, 4), 128, 3, 1, 1, 1, 337, 10), 2, dict(wk=4, whole=0)),
    ((4, True, 4, (5, 3), 64, 3, 1, 2, 300, 10, 20), 2, dict(mt=1, nt=2, wm=2)),
    # an odd one, and an order of the sums that would depend on what a tile holds: a pass of its own
    ((4, True, 3, (5, 3), 32, 3, 1, 2, 60, 60, 11), 1, dict(wk=1)),
    ((4, True, 4, (5, 1), 20, 3, 1, 2, 2, 5, 7), 1, dict(wk=4)),
    ((4, False, 4, (3, 4), 70, 2, 1, 1, 60, 100, 5), 1, dict(whole=170, rest=10)),
]


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_pooled_layers_match_layer_by_layer(case):
    (elem_bytes, mellin, layers, kernel, channels, schedule, cf, tf, batch, frames, bins), route, tiles = case
    params = ConvStackParams(layers=layers, mellin=mellin, kernel_time=kernel[0], kernel_freq=kernel[1], initial_channels=channels,
                             factor_schedule=schedule, channel_factor=cf, time_factor=tf, in_channels=1, freq_pool_after=(2,))
    words = (ctypes.c_int * len(WORDS))()
    dims = list(stack_dims(batch, frames, bins, params))[1]
    assert hip.lib.mellin_layer_plan(hip.AX_MCORR if mellin else hip.AX_LCORR, elem_bytes, 2, *dims, words) == route
    plan = dict(zip(WORDS, words))
    assert {k: plan[k] for k in tiles} == tiles, plan
    torch.manual_seed(9800 + CASES.index(case))
    stack = ConvStack(frames, bins, params).cuda()
    with torch.no_grad():
        for conv in stack.convs:
            conv.weight.uniform_(-1, 1).mul_((6 / conv.weight[0].numel()) ** 0.5)
            conv.bias.uniform_(-0.1, 0.1)
    x = torch.randn(batch, 1, frames, bins, device="cuda", requires_grad=True)
    leaves = list(stack.parameters()) + [x]
    results, grad = [], None
    for one_call in (True, False):
        hooks = [] if one_call else [conv.register_forward_hook(lambda *a: None) for conv in stack.convs]
        with torch.autocast("cuda", torch.float16, enabled=elem_bytes == 2):
            with torch.no_grad():
                served = stack(x)
            out = stack(x)
        assert ("StackBackward" in out.grad_fn.name()) == one_call
        assert torch.equal(served, out)
        grad = torch.randn_like(out) if grad is None else grad
        results.append([out.detach()] + list(torch.autograd.grad(out, leaves, grad)))
        for h in hooks:
            h.remove()
    assert torch.equal(results[0][0], results[1][0])
    for got, want in zip(*results):
        rel = float((got.double() - want.double()).norm() / want.double().norm())
        assert rel <= (2e-3 if elem_bytes == 2 else 2e-6), rel
