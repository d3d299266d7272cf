"""A stack's first layer storing the second's blocked input itself: the same bits as from a plain output that is laid out
afterwards, whichever kernel runs it."""
import pytest
import torch

from conv_stack import ConvStack, ConvStackParams

pytestmark = pytest.mark.gpu

CASES = [
    # (mellin, kernel, channels, time_factor, c_in, batch, frames, bins)
    (True, (4, 4), 20, 1, 1, 2, 50, 41),          # channels that end inside a unit; few tiles
    (True, (4, 4), 32, 1, 1, 16, 300, 41),        # tiles of two positions a lane
    (True, (5, 3), 64, 2, 1, 400, 10, 41),        # two tiles of channels, windows: images end inside tiles
    (True, (3, 3), 70, 1, 3, 6, 90, 32),          # two blocks of channels, an image of whole tiles
    (False, (4, 4), 24, 1, 1, 8, 120, 40),        # linear: few channels by the kernel of their own, half by tiles
    (False, (3, 3), 40, 2, 5, 4, 64, 37),
    (True, (3, 3), 48, 1, 2, 1, 40, 20),          # small enough for the blocked kernels themselves
    (True, (3, 3), 48, 1, 24, 3, 60, 20),
    (False, (3, 3), 96, 1, 64, 1, 20, 20),        # the same, contracted channels in slices
]


@pytest.mark.parametrize("kind", ["f32", "f16", "amp"])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_first_layer_into_blocked_input(case, kind):
    mellin, kernel, channels, tf, c_in, batch, frames, bins = case
    torch.manual_seed(9100 + CASES.index(case))
    stack = ConvStack(frames, bins, ConvStackParams(layers=2, mellin=mellin, kernel_time=kernel[0], kernel_freq=kernel[1],
                                                    initial_channels=channels, factor_schedule=2, time_factor=tf,
                                                    in_channels=c_in)).cuda()
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
