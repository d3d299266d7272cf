"""The windows' front end in native calls -- packing (`pack_windows`), log compression and lift from the modules' own
parameters -- against the same through PyTorch and through `log_compression_lift`, bit for bit."""
import pytest
import torch

from conv_stack import pack_windows
from layers import LogCompressionLift, log_compression_lift

pytestmark = pytest.mark.gpu

CASES = [  # (utterances' lengths, longest, bins, window, stride)
    ([50, 17, 33, 8], 50, 12, 10, 3),
    ([30, 30, 12, 30, 12], 30, 41, 5, 1),              # equal lengths: the order of PyTorch's sort
    ([7], 7, 1, 1, 1),                                 # one bin, windows of one frame
    ([4, 9], 9, 40, 20, 4),                            # windows longer than any utterance
    ([23, 5, 17], 40, 13, 3, 7),                       # strides past a window, frames past the longest utterance
    ([2, 1] * 70, 2, 5, 2, 1),
]


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_pack_windows_as_pytorch_packs_them(case):
    lens, longest, bins, size, stride = case
    x = torch.randn(len(lens), longest, bins, device="cuda")
    lens = torch.tensor(lens)
    windows, packed = pack_windows(x, lens, size, stride)
    want, want_packed = pack_windows(x.clone().requires_grad_(), lens, size, stride)      # (differentiable: PyTorch's own copies)
    assert windows.shape == want.shape and windows.is_contiguous() and torch.equal(windows, want)
    assert packed.data.data_ptr() == windows.data_ptr()
    for name in ("data", "batch_sizes", "sorted_indices", "unsorted_indices"):
        got, ref = getattr(packed, name), getattr(want_packed, name)
        assert got.dtype == ref.dtype and got.device == ref.device and torch.equal(got, ref), name
    strided = x.transpose(1, 2).contiguous().transpose(1, 2)
    assert torch.equal(pack_windows(strided, lens, size, stride)[0], want)


def test_pack_windows_leaves_odd_lengths_to_pytorch():
    x = torch.randn(3, 20, 4, device="cuda")
    for lens in ([20, 0, 3], [20, 45, 3], [20, 3]):        # (accepted there, each in its way)
        got, want = (pack_windows(t, torch.tensor(lens), 5, 2)[1] for t in (x, x.clone().requires_grad_()))
        assert torch.equal(got.data, want.data) and torch.equal(got.batch_sizes, want.batch_sizes)
    with pytest.raises(RuntimeError, match="greater than 0"):
        pack_windows(x, torch.tensor([20, -5, 3]), 5, 2)


@pytest.mark.parametrize("shape,dim", [((37, 1, 10, 41), 2), ((5, 7), 1), ((2, 3, 4), -2)])
def test_lift_from_its_own_parameters(shape, dim):
    torch.manual_seed(3)
    module = LogCompressionLift(dim=dim).cuda()
    x = torch.randn(*shape, device="cuda")
    x.flatten()[::5] = 0
    grad = torch.randn(*shape, device="cuda")
    xa, xb = x.clone().requires_grad_(), x.clone().requires_grad_()
    ya = module(xa)
    yb = log_compression_lift(xb, module.log_eps.exp(), module.log_tau.exp(), dim)
    with torch.no_grad():
        assert torch.equal(module(x), ya)
    assert "LogLiftBackward" in ya.grad_fn.name() and torch.equal(ya, yb)
    got = torch.autograd.grad(ya, (xa, module.log_eps, module.log_tau), grad)
    want = torch.autograd.grad(yb, (xb, module.log_eps, module.log_tau), grad)
    assert all(a.shape == b.shape and torch.equal(a, b) for a, b in zip(got, want))
    only = torch.autograd.grad(module(x), (module.log_tau,), grad)         # (no gradient of the input)
    assert torch.equal(only[0], want[2])
