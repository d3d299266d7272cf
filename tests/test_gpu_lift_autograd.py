"""`LogCompressionLift` in its native autograd node, where PyTorch's own rules for a graph decide what a caller may do."""
import pytest
import torch

from layers import LogCompressionLift, log_compression_lift

pytestmark = pytest.mark.gpu


def _module_and_data():
    module = LogCompressionLift(dim=2).cuda()
    x = torch.randn(5, 1, 7, 9, device="cuda")
    return module, x, torch.randn_like(x)


@pytest.mark.parametrize("through", ["step", "data"])
def test_gradients_are_those_of_the_forward_call(through):
    """exp() keeps its result: a graph that is older than an optimiser's step gives the gradients of its own forward call."""
    module, x, grad = _module_and_data()
    xa, xb = x.clone().requires_grad_(), x.clone().requires_grad_()
    ya = module(xa)
    yb = log_compression_lift(xb, module.log_eps.exp(), module.log_tau.exp(), 2)
    assert "LogLiftBackward" in ya.grad_fn.name()
    with torch.no_grad():
        for p in module.parameters():
            (p.data if through == "data" else p).add_(0.5)
    got = torch.autograd.grad(ya, (xa, module.log_eps, module.log_tau), grad)
    want = torch.autograd.grad(yb, (xb, module.log_eps, module.log_tau), grad)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_gradients_have_memory_of_their_own():
    module, x, grad = _module_and_data()
    module(x).backward(grad)
    a, b = module.log_eps.grad, module.log_tau.grad
    assert a.untyped_storage().data_ptr() != b.untyped_storage().data_ptr()
    assert a.untyped_storage().nbytes() == b.untyped_storage().nbytes() == 4


class _NoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, y):
        return y * 1

    @staticmethod
    def backward(ctx, grad):
        return None


def test_a_gradient_that_is_not_there_counts_as_zeros():
    module, x, _ = _module_and_data()
    xg = x.requires_grad_()
    _NoGradient.apply(module(xg)).sum().backward()
    for g in (xg.grad, module.log_eps.grad, module.log_tau.grad):
        assert g is not None and not g.any()
