"""`ConvStack` through one call per direction (tensors blocked from layer to layer, ReLU masks, bias gradients and pooling
inside the kernels) against the same layers called one by one, which the checker covers."""
import pytest
import torch

from conv_stack import ConvStack, ConvStackParams

pytestmark = pytest.mark.gpu

CASES = [
    # (mellin, layers, kernel, channels, schedule, channel_factor, time_factor, pool_every, c_in, batch, frames, bins)
    (True, 2, (4, 4), 16, 2, 1, 1, 0, 3, 1, 37, 13),       # one blocked layer, few tiles: slices as the last layer's output
    (True, 5, (4, 4), 32, 3, 2, 1, 2, 3, 1, 200, 41),      # few tiles: slices with a mask, blocked and dense; odd columns pooled
    (False, 4, (5, 2), 20, 2, 1, 2, 3, 1, 20, 400, 20),    # channels that do not fill their last group
    (True, 4, (3, 3), 70, 2, 2, 2, 0, 1, 8, 100, 40),      # channels past a tile, strides, classes of rows
    (False, 7, (3, 4), 64, 3, 2, 1, 3, 3, 9, 90, 33),      # two poolings
    (True, 3, (5, 3), 64, 2, 1, 2, 0, 1, 300, 10, 41),     # windows: many small images
]


@pytest.mark.parametrize("half", [False, True], ids=["f32", "amp"])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_stack_in_one_call_matches_layer_by_layer(case, half):
    mellin, layers, kernel, channels, schedule, cf, tf, every, c_in, batch, frames, bins = case
    torch.manual_seed(8000 + CASES.index(case))
    stack = ConvStack(frames, bins, ConvStackParams(
        layers=layers, mellin=mellin, kernel_time=kernel[0], kernel_freq=kernel[1], initial_channels=channels,
        factor_schedule=schedule, channel_factor=cf, time_factor=tf, in_channels=c_in,
        freq_pool_after=tuple(range(every, layers + 1, every)) if every else ())).cuda()
    with torch.no_grad():
        for conv in stack.convs:
            conv.weight.uniform_(-1, 1).mul_((6 / conv.weight[0].numel()) ** 0.5)
            conv.bias.uniform_(-0.1, 0.1)
    x = torch.randn(batch, c_in, frames, bins, device="cuda")
    leaves = list(stack.parameters())
    results, grad = [], None
    for one_call in (True, False):
        hooks = [] if one_call else [conv.register_forward_hook(lambda *a: None) for conv in stack.convs]
        xg = x.clone().requires_grad_()
        with torch.autocast("cuda", torch.float16, enabled=half):
            with torch.no_grad():
                served = stack(xg)
            out = stack(xg)
        last = out.grad_fn.next_functions[0][0] if every and layers % every == 0 else out.grad_fn
        assert ("StackBackward" in last.name()) == one_call
        grad = torch.randn_like(out) if grad is None else grad
        grads = torch.autograd.grad(out, leaves + [xg], grad)
        assert torch.equal(served, out)
        assert all(g.dtype == torch.float32 for g in grads)
        results.append([out.detach()] + list(grads))
        for h in hooks:
            h.remove()
    for got, want in zip(*results):
        rel = float((got.double() - want.double()).norm() / want.double().norm())
        assert rel <= (2e-3 if half else 2e-6), rel


def test_stack_gives_the_gradients_that_are_asked_for():
    stack = ConvStack(60, 20, ConvStackParams(layers=4, mellin=True, kernel_time=3, kernel_freq=3, initial_channels=24,
                                              factor_schedule=2, time_factor=1, in_channels=3)).cuda()
    x = torch.randn(2, 3, 60, 20, device="cuda", requires_grad=True)
    out = stack(x)
    grad = torch.randn_like(out)
    leaves = list(stack.parameters())
    full = torch.autograd.grad(out, leaves + [x], grad, retain_graph=True)
    again = torch.autograd.grad(out, leaves + [x], grad, retain_graph=True)
    assert all(torch.equal(a, b) for a, b in zip(full, again))
    for pick in ([0], [5], [6], [7], [2, 3], [len(leaves)]):
        some = torch.autograd.grad(out, [(leaves + [x])[i] for i in pick], grad, retain_graph=True)
        assert all(torch.equal(some[k], full[i]) for k, i in enumerate(pick))
    stack.convs[0].weight.requires_grad_(False)
    stack.convs[0].bias.requires_grad_(False)
    out = stack(x.detach())
    out.backward(grad)
    assert stack.convs[0].weight.grad is None and torch.equal(stack.convs[1].weight.grad, full[2])
