"""A stack's first layer storing the second's blocked input itself: the same bits as from a plain output that is laid out
afterwards, whichever kernel runs it."""
import pytest
import torch

import _mellin_hip as hip
from conv_stack import ConvStack, ConvStackParams
from test_block_plans import FIRST_BLOCKS, FIRST_OWN, FIRST_TILES, first_layer, stack_dims

pytestmark = pytest.mark.gpu

CASES = [
    # (mellin, kernel, channels, time_factor, c_in, batch, frames, bins)
    (True, (4, 4), 20, 1, 1, 2, 50, 41),          # channels that end inside a unit; few tiles
    (True, (4, 4), 32, 1, 1, 16, 300, 41),        # tiles of two positions a lane
    (True, (5, 3), 64, 2, 1, 400, 10, 41),        # two tiles of channels, windows: images end inside tiles
    (True, (3, 3), 70, 1, 3, 6, 90, 32),          # two blocks of channels, an image of whole tiles
    (False, (4, 4), 24, 1, 1, 8, 120, 40),        # linear
    (False, (3, 3), 40, 2, 5, 4, 64, 37),
    (True, (3, 3), 48, 1, 2, 1, 40, 20),          # an image, few tiles
    (True, (3, 3), 48, 1, 24, 3, 60, 20),         # the blocked kernels
    (False, (3, 3), 96, 1, 64, 1, 20, 20),        # the same, contracted channels in slices
    (True, (6, 4), 40, 2, 12, 2, 300, 41),        # half: the same, few channels on long rows
    (False, (6, 4), 20, 1, 12, 1, 120, 9),        # filters in chunks of channels: a plain output, laid out afterwards
    (True, (5, 2), 20, 1, 12, 1, 20, 9),
    (False, (6, 4), 48, 2, 12, 32, 60, 41),
]
#: which of them take which way, in fp32 and in half
ROUTES = 7 * [(FIRST_TILES, FIRST_TILES)] + 2 * [(FIRST_BLOCKS, FIRST_BLOCKS)] + [
    (FIRST_OWN, FIRST_BLOCKS), (FIRST_OWN, FIRST_TILES), (FIRST_OWN, FIRST_OWN), (FIRST_OWN, FIRST_OWN)]


@pytest.mark.parametrize("kind", ["f32", "f16", "amp"])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_first_layer_into_blocked_input(case, kind):
    mellin, kernel, channels, tf, c_in, batch, frames, bins = case
    torch.manual_seed(9100 + CASES.index(case))
    params = ConvStackParams(layers=2, mellin=mellin, kernel_time=kernel[0], kernel_freq=kernel[1], initial_channels=channels,
                             factor_schedule=2, time_factor=tf, in_channels=c_in)
    route = first_layer(hip.AX_MCORR if mellin else hip.AX_LCORR, 4 if kind == "f32" else 2,
                        next(iter(stack_dims(batch, frames, bins, params))))
    assert route == ROUTES[CASES.index(case)][kind != "f32"]
    stack = ConvStack(frames, bins, params).cuda()
    x = torch.randn(batch, c_in, frames, bins, device="cuda")
    if kind == "f16":
        stack, x = stack.half(), x.half()
    with torch.autocast("cuda", torch.float16, enabled=kind == "amp"):
        out = stack(x)
        with torch.no_grad():
            served = stack(x)
        want = x
        for conv in stack.convs:
            want = conv(want, activation="relu")
    assert "StackBackward" in out.grad_fn.name()
    assert torch.equal(out, want) and torch.equal(served, want)
