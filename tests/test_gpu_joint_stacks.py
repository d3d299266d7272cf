"""Input gradients inside a stack whose tiles run over the images of an output row, in every form their ending takes there --
masked, blocked, with the channels' sums, or blocked alone above a pooling; whole tiles, tiles in slices of the contracted
channels, both; wavefronts that share a tile, wavefronts along the channels -- against the same layers called one by one, whose
gradients are plain tensors."""
import pytest
import torch

import _mellin_hip as hip
from conv_stack import ConvStack, ConvStackParams
from test_block_plans import plan, stack_dims

pytestmark = pytest.mark.gpu

WHOLE, SLICES = (True, False), (False, True)
CASES = [
    # (element bytes, (wavefronts along the channels, that share a tile), (whole tiles, in slices), the layer (its input gradient),
    #  layers, kernel, channels, schedule, channel_factor, time_factor, batch, frames, bins, pooled behind the layer)
    (4, (1, 1), WHOLE, 2, 4, (5, 3), 32, 3, 1, 1, 60, 60, 5, None),
    (4, (1, 1), SLICES, 2, 4, (5, 3), 96, 4, 1, 1, 2, 5, 5, None),
    (4, (1, 1), (True, True), 2, 4, (3, 4), 96, 2, 2, 1, 60, 10, 20, None),
    (4, (1, 4), WHOLE, 2, 4, (4, 4), 64, 3, 1, 2, 2, 10, 5, None),
    (4, (1, 4), SLICES, 2, 4, (3, 4), 64, 3, 2, 2, 4, 5, 3, None),
    (4, (2, 1), WHOLE, 3, 4, (3, 3), 128, 3, 2, 1, 60, 120, 3, None),
    (4, (2, 1), SLICES, 2, 3, (5, 2), 128, 2, 2, 1, 300, 5, 3, None),
    (4, (2, 1), (True, True), 3, 4, (4, 1), 64, 2, 2, 1, 300, 60, 5, None),
    (2, (1, 1), WHOLE, 3, 4, (4, 3), 32, 4, 1, 2, 60, 120, 5, None),
    (2, (1, 1), SLICES, 3, 4, (5, 3), 128, 2, 2, 1, 150, 5, 10, None),
    (2, (1, 1), (True, True), 3, 4, (5, 4), 96, 2, 2, 1, 150, 60, 5, None),
    (2, (1, 4), WHOLE, 2, 3, (5, 4), 64, 3, 2, 1, 4, 5, 10, None),
    (2, (1, 4), SLICES, 3, 4, (5, 3), 128, 2, 2, 1, 9, 5, 10, None),
    (2, (2, 1), WHOLE, 2, 4, (4, 1), 64, 2, 2, 1, 300, 60, 5, None),
    (4, (1, 1), WHOLE, 2, 4, (5, 3), 32, 3, 1, 2, 60, 60, 10, 2),
    (4, (1, 1), SLICES, 2, 3, (5, 3), 96, 4, 2, 1, 2, 5, 10, 2),
    (4, (1, 1), (True, True), 2, 3, (4, 4), 96, 3, 1, 2, 9, 252, 20, 2),
    (4, (1, 4), WHOLE, 2, 4, (5, 4), 32, 4, 1, 2, 4, 5, 10, 2),
    (4, (1, 4), SLICES, 2, 4, (4, 3), 128, 3, 2, 1, 2, 5, 5, 2),
    (4, (2, 1), WHOLE, 2, 3, (5, 1), 128, 2, 2, 1, 300, 20, 7, 2),
    (4, (2, 1), SLICES, 2, 4, (5, 2), 128, 2, 2, 1, 60, 5, 41, 2),
    (2, (1, 1), WHOLE, 2, 3, (4, 3), 32, 3, 2, 2, 60, 120, 10, 2),
    (2, (1, 4), WHOLE, 2, 3, (5, 4), 32, 3, 2, 2, 4, 10, 7, 2),
    (2, (1, 4), SLICES, 2, 4, (5, 4), 128, 3, 2, 2, 9, 10, 7, 2),
]


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_blocked_endings_of_joint_tiles(case):
    elem_bytes, wavefronts, tiles, layer, layers, kernel, channels, schedule, cf, tf, batch, frames, bins, pooled = case
    params = ConvStackParams(layers=layers, kernel_time=kernel[0], kernel_freq=kernel[1], initial_channels=channels,
                             factor_schedule=schedule, channel_factor=cf, time_factor=tf, in_channels=1,
                             freq_pool_after=(pooled,) if pooled else ())
    p = plan(hip.AX_MCORR, elem_bytes, 1, list(stack_dims(batch, frames, bins, params))[layer])
    assert p["joint"] and (p["wm"], p["wk"]) == wavefronts and (p["whole"] > 0, p["rest"] > 0) == tiles, p
    torch.manual_seed(9700 + CASES.index(case))
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
            out = stack(x)
        assert ("StackBackward" in out.grad_fn.name()) == one_call
        grad = torch.randn_like(out) if grad is None else grad
        results.append([out.detach()] + list(torch.autograd.grad(out, leaves, grad)))
        for h in hooks:
            h.remove()
    assert torch.equal(results[0][0], results[1][0])
    # the outputs, and with them the ReLUs' choices, are the same; each layer rounds the gradient that it hands on, in either
    # order of summation: the bounds of the same comparison for seven layers
    for got, want in zip(*results):
        rel = float((got.double() - want.double()).norm() / want.double().norm())
        assert rel <= (2e-3 if elem_bytes == 2 else 2e-6), rel
