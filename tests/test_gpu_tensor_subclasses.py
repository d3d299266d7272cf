"""Subclasses of torch.Tensor go through PyTorch's own operations, whose overrides they may have, also where plain tensors take
a native call."""
import pytest
import torch

from conv_stack import pack_windows
from layers import LogCompressionLift

pytestmark = pytest.mark.gpu


class Followed(torch.Tensor):
    """Notes the operations that it passes through."""
    seen = []

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        cls.seen.append(getattr(func, "__name__", str(func)))
        return super().__torch_function__(func, types, args, kwargs or {})


def test_windows_of_a_subclass():
    x, lens = torch.randn(3, 20, 4, device="cuda"), torch.tensor([20, 7, 13])
    want, want_packed = pack_windows(x, lens, 5, 2)
    Followed.seen.clear()
    got, packed = pack_windows(x.as_subclass(Followed), lens, 5, 2)
    assert "unfold" in Followed.seen and type(got) is Followed
    assert torch.equal(got.as_subclass(torch.Tensor), want) and torch.equal(packed.batch_sizes, want_packed.batch_sizes)
    Followed.seen.clear()
    assert torch.equal(pack_windows(x, lens.as_subclass(Followed), 5, 2)[0], want) and "div" in Followed.seen


def test_lift_of_a_subclass():
    module, x = LogCompressionLift(dim=2).cuda(), torch.randn(3, 1, 6, 4, device="cuda")
    want = module(x)
    got = module(x.as_subclass(Followed))
    assert type(got) is Followed and torch.equal(got.as_subclass(torch.Tensor), want)
    module.log_tau = torch.nn.Parameter(module.log_tau.detach().as_subclass(Followed))
    Followed.seen.clear()
    got = module(x)
    assert "exp" in Followed.seen and torch.equal(got.as_subclass(torch.Tensor), want)
