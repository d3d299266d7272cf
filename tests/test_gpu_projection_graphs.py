"""Gradients with a graph of their own (``create_graph``) through the projection of a half `FrameClassifier` that runs in the stack's
call: they are those of the forward call's features and weights, whatever has been changed since, as where the modules run one
by one (a hook on the projection)."""
import gc
import weakref

import pytest
import torch

import conv_stack
from conv_stack import ConvStack, ConvStackParams, FrameClassifier

pytestmark = pytest.mark.gpu

CASES = [
    # (Mellin, layers, pooled after, frames, bins, classes)
    (True, 2, (), 40, 5, 9),
    (False, 3, (2,), 33, 11, 62),          # pooled inside: 5 bins
    (True, 3, (3,), 40, 10, 9),            # pooled behind the last convolution, an even number of bins
    (False, 3, (2, 3), 27, 23, 9),         # and an odd one: 5 bins of 11
]


def classifier(case, how):
    mellin, layers, pools, frames, bins, classes = case
    torch.manual_seed(9800 + CASES.index(case))
    params = ConvStackParams(layers=layers, mellin=mellin, kernel_time=3, kernel_freq=3, initial_channels=24, factor_schedule=2,
                             channel_factor=2, time_factor=1, in_channels=3, freq_pool_after=pools)
    model = FrameClassifier(ConvStack(frames, bins, params), classes).cuda()
    if how == "no bias":
        model.out.bias = None
    if how.startswith("frozen"):
        model.stack.requires_grad_(False)
    x = torch.randn(2, 3, frames, bins, device="cuda")
    if how.endswith("half"):
        model, x = model.half(), x.half()
    if how == "input":
        x.requires_grad_()
    labels = torch.randint(classes, (2 * model.stack.out_size[0],), device="cuda")
    leaves = [p for p in model.parameters() if p.requires_grad] + ([x] if x.requires_grad else [])
    return model, x, labels, leaves


def loss_of(model, x, labels, how):
    with torch.autocast("cuda", torch.float16, enabled=not how.endswith("half")):
        out = model(x)
    return torch.nn.functional.nll_loss(out.flatten(0, 1).float(), labels) * 64


def change(model, x):
    """What an optimizer's step and a reused input buffer do."""
    with torch.no_grad():
        for p in model.parameters():
            p.mul_(-0.5).add_(0.05)
        x.data.add_(1) if x.requires_grad else x.add_(1)


@pytest.mark.parametrize("changed", [False, True])
@pytest.mark.parametrize("how", ["autocast", "no bias", "frozen", "frozen half", "input"])
@pytest.mark.parametrize("case", CASES, ids=range(len(CASES)))
def test_gradients_are_those_of_the_forward_call(case, how, changed, monkeypatch):
    calls, counts, native = [], [], conv_stack._native_stack
    monkeypatch.setattr(conv_stack, "_native_stack", lambda *a: calls.append(len(a[2])) or native(*a))

    def penalty(apart):
        model, x, labels, leaves = classifier(case, how)
        if apart:
            model.out.register_forward_hook(lambda *a: None)
        del calls[:]
        loss = loss_of(model, x, labels, how)
        assert calls == [len(model.stack.convs) + (not apart)]
        if changed:
            change(model, x)
        plain = torch.autograd.grad(loss, list(model.out.parameters()), retain_graph=True)
        first = torch.autograd.grad(loss, list(model.out.parameters()), create_graph=True)
        second = torch.autograd.grad(sum(v.float().square().sum() for v in first) * 64, leaves)
        counts.append(len(calls))
        return list(plain) + [v.detach() for v in first] + list(second)

    # half features, gradients and their gradients: a few roundings of 2^-11 each, in sums whose terms partly cancel
    for got, want in zip(penalty(False), penalty(True)):
        assert got.dtype == want.dtype and got.shape == want.shape
        rel = float((got.double() - want.double()).norm() / want.double().norm())
        assert rel < 2e-2, rel
    assert counts == [1, 1]                            # (nothing is computed again)


@pytest.mark.parametrize("apart", [False, True])
def test_changes_of_saved_tensors_are_refused(apart):
    """Half parameters and inputs are saved themselves."""
    for what in ("weight", "input", "weight between"):
        model, x, labels, leaves = classifier(CASES[2], "half")
        if apart:
            model.out.register_forward_hook(lambda *a: None)
        loss = loss_of(model, x, labels, "half")
        changed = x if what == "input" else model.stack.convs[1].weight

        def alter():
            with torch.no_grad():
                changed.add_(1)

        if what != "weight between":
            alter()
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            first = torch.autograd.grad(loss, leaves if what != "weight between" else list(model.out.parameters()), create_graph=True)
            alter()
            torch.autograd.grad(sum(v.float().square().sum() for v in first), leaves)


def test_an_older_graph_holds_no_input():
    model, x, labels, leaves = classifier(CASES[0], "autocast")
    with torch.autocast("cuda", torch.float16):
        assert model._scores(x) is not None
    gone = weakref.ref(x)
    loss = loss_of(model, x, labels, "autocast")
    loss.backward()
    del x
    gc.collect()
    assert gone() is None and loss.grad_fn is not None


def test_stacks_that_are_not_joined_are_not_looked_through_twice(monkeypatch):
    looked = []
    plain = ConvStack._plain
    monkeypatch.setattr(ConvStack, "_plain", lambda self: looked.append(1) or plain(self))
    for layers, bins, classes in ((2, 7, 9), (1, 5, 9), (2, 5, 257)):              # more than six bins; one layer; many classes
        params = ConvStackParams(layers=layers, kernel_time=3, kernel_freq=3, initial_channels=32, factor_schedule=2, time_factor=1,
                                 in_channels=3)
        model, x = FrameClassifier(ConvStack(40, bins, params), classes).cuda(), torch.randn(2, 3, 40, bins, device="cuda")
        del looked[:]
        with torch.no_grad(), torch.autocast("cuda", torch.float16):
            model(x)
            assert model._scores(x) is None
        assert len(looked) == 1


def test_default_devices_change_nothing():
    model, x, labels, leaves = classifier(CASES[0], "autocast")
    for context in (torch.device("cuda"), torch.device("cpu")):
        with context, torch.autocast("cuda", torch.float16):
            assert model._scores(x) is not None
    with torch.autocast("cuda", torch.float16):
        joined = model(x)
        with torch.device("cpu"):
            assert torch.equal(model(x), joined)
