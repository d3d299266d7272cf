"""`FrameClassifier` in half precision, whose projection is the last layer of the stack's call, against the same modules called
one by one (a hook on the projection), and both against float64."""
import pytest
import torch

from conv_stack import ConvStack, ConvStackParams, FrameClassifier

pytestmark = pytest.mark.gpu

CASES = [
    # (Mellin, layers, kernel, channels, channel_factor, pool after, batch, frames, bins, classes)
    (False, 3, (4, 4), 32, 2, (2,), 5, 91, 13, 62),        # 4 -> 1 bin
    (True, 3, (4, 4), 32, 2, (2, 3), 3, 70, 23, 62),       # pooled behind the last layer too: 5 bins
    (True, 2, (3, 3), 24, 1, (), 4, 33, 6, 7),             # 6 bins, a class count below a tile
    (False, 4, (3, 3), 40, 2, (2,), 2, 60, 12, 130),       # more classes than a tile
]


class Through(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("how", ["autocast", "half", "no bias", "frozen"])
@pytest.mark.parametrize("case", CASES, ids=range(len(CASES)))
def test_joined_and_apart(case, how):
    mellin, layers, kernel, channels, cf, pools, batch, frames, bins, classes = case
    torch.manual_seed(9600 + CASES.index(case))
    params = ConvStackParams(layers=layers, mellin=mellin, kernel_time=kernel[0], kernel_freq=kernel[1], initial_channels=channels,
                             factor_schedule=2, channel_factor=cf, time_factor=1, in_channels=3, freq_pool_after=pools)
    model = FrameClassifier(ConvStack(frames, bins, params), classes).cuda()
    with torch.no_grad():
        for conv in model.stack.convs:
            conv.weight.uniform_(-1, 1).mul_((6 / conv.weight[0].numel()) ** 0.5)
    if how == "no bias":
        model.out.bias = None
    if how == "frozen":
        model.stack.requires_grad_(False)
    if how == "half":
        model = model.half()
    x = torch.randn(batch, 3, frames, bins, device="cuda", dtype=torch.float16 if how == "half" else torch.float32)
    labels = torch.randint(classes, (batch * model.stack.out_size[0],), device="cuda")
    leaves = [p for p in model.parameters() if p.requires_grad]

    def step(net, x, leaves, dtype):
        with torch.autocast("cuda", torch.float16, enabled=dtype is None and how != "half"):
            out = net(x)
        loss = torch.nn.functional.nll_loss(out.flatten(0, 1).double(), labels)
        return [out.detach()] + list(torch.autograd.grad(loss * 64, leaves))

    with torch.autocast("cuda", torch.float16, enabled=how != "half"):
        assert model._scores(x) is not None
    joined = step(model, x, leaves, None)
    hook = model.out.register_forward_hook(lambda *a: None)
    assert model._scores(x) is None
    apart = step(model, x, leaves, None)
    hook.remove()
    assert joined[0].shape == apart[0].shape and joined[0].stride() == apart[0].stride() and joined[0].dtype == apart[0].dtype
    # the convolutions' outputs are the same bits, the projection's sums have another order: a rounding to half (2^-11) of
    # scores, and of each gradient that is handed on
    for got, want in zip(joined, apart):
        assert got.dtype == want.dtype
        rel = float((got.double() - want.double()).norm() / want.double().norm())
        assert rel < 4e-3, rel
    # neither is further from float64 than the other by more than such roundings
    with torch.no_grad():
        wide = FrameClassifier(ConvStack(frames, bins, params), classes).cuda()
        wide.out.bias = None if how == "no bias" else wide.out.bias
        wide.load_state_dict(model.state_dict())
        wide = wide.double()
    named = dict(wide.named_parameters())
    exact = step(wide, x.double(), [named[n] for n, p in model.named_parameters() if p.requires_grad], torch.float64)
    for a, b, ref in zip(joined, apart, exact):
        one, two = (float((v.double() - ref).norm() / ref.norm()) for v in (a, b))
        assert one < 1.2 * two + 2e-4, (one, two)


def test_sizes_and_types_that_stay_apart():
    params = ConvStackParams(layers=2, kernel_time=3, kernel_freq=3, initial_channels=32, factor_schedule=2, time_factor=1,
                             in_channels=3)
    model = FrameClassifier(ConvStack(40, 5, params), 9).cuda()
    x = torch.randn(2, 3, 40, 5, device="cuda")
    assert model._scores(x) is None and model._scores(x.double()) is None                        # float, double
    with torch.autocast("cuda", torch.bfloat16):
        assert model._scores(x) is None
    with torch.autocast("cuda", torch.float16):
        assert model._scores(x) is not None
        assert model._scores(torch.randn(2, 3, 17, 5, device="cuda")).shape == model(torch.randn(2, 3, 17, 5, device="cuda")).shape
        for bins in (7, 4):                                                                     # the projection refuses them
            with pytest.raises(RuntimeError, match="mat1 and mat2 shapes cannot be multiplied"):
                model(torch.randn(2, 3, 40, bins, device="cuda"))
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
            assert model._scores(x) is None
        with Through():
            assert model._scores(x) is None
        many = FrameClassifier(ConvStack(40, 7, params), 9).cuda()
        assert many._scores(torch.randn(2, 3, 40, 7, device="cuda")) is None                     # more than 6 bins


@pytest.mark.parametrize("how", ["autocast", "half", "no bias", "frozen"])
def test_second_derivatives_of_the_projection(how):
    params = ConvStackParams(layers=2, kernel_time=3, kernel_freq=3, initial_channels=32, factor_schedule=2, time_factor=1,
                             in_channels=3)
    torch.manual_seed(9700)
    model = FrameClassifier(ConvStack(40, 5, params), 9).cuda()
    if how == "no bias":
        model.out.bias = None
    if how == "frozen":
        model.stack.requires_grad_(False)
    x = torch.randn(2, 3, 40, 5, device="cuda")
    if how == "half":
        model, x = model.half(), x.half()
    labels = torch.randint(9, (80,), device="cuda")
    leaves = [p for p in model.parameters() if p.requires_grad]

    def penalty():
        with torch.autocast("cuda", torch.float16, enabled=how != "half"):
            out = model(x)
        loss = torch.nn.functional.nll_loss(out.flatten(0, 1).float(), labels)
        first = torch.autograd.grad(loss, list(model.out.parameters()), create_graph=True)
        return [v.detach() for v in first] + list(torch.autograd.grad(sum(v.float().square().sum() for v in first) * 64, leaves))

    joined = penalty()
    hook = model.out.register_forward_hook(lambda *a: None)
    apart = penalty()
    hook.remove()
    # half features, gradients and their gradients: a few roundings of 2^-11 each, in sums whose terms partly cancel
    for got, want in zip(joined, apart):
        assert got.dtype == want.dtype and got.shape == want.shape
        rel = float((got.double() - want.double()).norm() / want.double().norm())
        assert rel < 2e-2, rel
