"""Sums and filters of a whole stack's layers that share launches: more layers than a launch takes, more classes of rows, and
partial sums that fill their memory, against the same layers called one by one."""
import pytest
import torch

from conv_stack import ConvStack, ConvStackParams

pytestmark = pytest.mark.gpu

CASES = [
    # (mellin, layers, kernel, channels, time_factor, pool_every, batch, frames, bins)
    (True, 20, (5, 3), 16, 1, 0, 2, 40, 9),       # more layers than jobs of a launch, and classes
    (False, 18, (2, 2), 24, 1, 6, 1, 60, 41),     # poolings between them; columns without a tap
    (True, 5, (4, 4), 256, 1, 2, 4, 120, 12),     # partial sums of some 30 MB a layer
]


@pytest.mark.parametrize("half", [False, True], ids=["f32", "amp"])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_shared_launches(case, half):
    mellin, layers, kernel, channels, tf, every, batch, frames, bins = case
    torch.manual_seed(9500 + CASES.index(case))
    stack = ConvStack(frames, bins, ConvStackParams(
        layers=layers, mellin=mellin, kernel_time=kernel[0], kernel_freq=kernel[1], initial_channels=channels,
        factor_schedule=layers + 1, time_factor=tf, in_channels=1,
        freq_pool_after=tuple(range(every, layers, every)) if every else ())).cuda()
    with torch.no_grad():
        for conv in stack.convs:
            conv.weight.uniform_(-1, 1).mul_((6 / conv.weight[0].numel()) ** 0.5)
            conv.bias.uniform_(-0.1, 0.1)
    x = torch.randn(batch, 1, frames, bins, device="cuda")
    leaves = list(stack.parameters())
    results, grad = [], None
    for one_call in (True, False):
        hooks = [] if one_call else [conv.register_forward_hook(lambda *a: None) for conv in stack.convs]
        with torch.autocast("cuda", torch.float16, enabled=half):
            out = stack(x)
        assert ("StackBackward" in out.grad_fn.name()) == one_call
        grad = torch.randn_like(out) if grad is None else grad
        results.append([out.detach()] + list(torch.autograd.grad(out, leaves, grad)))
        for h in hooks:
            h.remove()
    # each layer rounds what it hands on, in either order of summation: independent errors of 2^-11 (2^-24), passed on by
    # every layer, add up in squares; 2e-3 and 2e-6 bound the same comparison for seven layers
    bound = (2e-3 if half else 2e-6) * max(1, layers / 7) ** 0.5
    for got, want in zip(*results):
        rel = float((got.double() - want.double()).norm() / want.double().norm())
        assert rel <= bound, rel
