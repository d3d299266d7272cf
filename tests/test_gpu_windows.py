"""The windows' front end in native calls -- packing (`pack_windows`), log compression and lift from the modules' own
parameters -- against the same through PyTorch and through `log_compression_lift`, bit for bit."""
import pytest
import torch

import _mellin_hip as hip
from conv_stack import ConvStack, ConvStackParams, pack_windows
from test_block_plans import plan, stack_dims
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


def _layer64(x, weight, bias, lay, out_size):
    """A Mellin x linear layer of `layer_plan` in float64, a matrix product per output row."""
    (c_out, c_in, kx, ky), n, (ox, oy) = weight.shape, x.shape[0], out_size
    (sx, sy), (dx, dy), (px, py) = lay["s"], lay["d"], lay["p"]
    x = torch.nn.functional.pad(x, (py, max(0, sy * (oy - 1) + dy * (ky - 1) + 1 - x.shape[3] - py)))
    rows = []
    for h in range(ox):
        taps = [(f, (h + sx) * (f + dx) // (px + 1) - 1) for f in range(kx) if (h + sx) * (f + dx) % (px + 1) == 0]
        taps = [(f, g, fy) for f, g in taps if g < x.shape[2] for fy in range(ky)]
        row = bias.view(-1, 1).expand(c_out, n * oy)
        if taps:
            cols = torch.stack([x[:, :, g, fy * dy:fy * dy + sy * (oy - 1) + 1:sy] for _, g, fy in taps])      # (taps, n, c_in, oy)
            w = torch.stack([weight[:, :, f, fy] for f, _, fy in taps], 1).reshape(c_out, -1)
            row = row + w @ cols.permute(0, 2, 1, 3).reshape(-1, n * oy)
        rows.append(row.view(c_out, n, oy))
    return torch.stack(rows, 2).transpose(0, 1)


@pytest.mark.parametrize("lens,bins,window,stride,kernel,channels,layers", [
    ([190, 151, 77, 33], 41, 10, 1, (5, 3), 64, 4),    # joint tiles in the input gradients
    ([120, 64], 20, 7, 2, (3, 3), 24, 3),              # channels that end inside a tile
])
def test_training_step_against_float64_at_its_own_flags(lens, bins, window, stride, kernel, channels, layers):
    """A whole step, front end and stack, with the ReLUs' choices of the step itself: what another order of the sums makes of
    values near zero stays out of the comparison, and what is left is rounding."""
    torch.manual_seed(21)
    params = ConvStackParams(layers=layers, kernel_time=kernel[0], kernel_freq=kernel[1], initial_channels=channels, factor_schedule=2,
                             time_factor=2)
    stack, lift = ConvStack(window, bins, params).cuda(), LogCompressionLift(dim=2).cuda()
    with torch.no_grad():
        for conv in stack.convs:
            conv.weight.uniform_(-1, 1).mul_((6 / conv.weight[0].numel()) ** 0.5)
            conv.bias.uniform_(-0.1, 0.1)
    x = torch.randn(len(lens), max(lens), bins, device="cuda").exp()
    windows, _ = pack_windows(x, torch.tensor(lens), window, stride)
    out = stack(lift(windows))
    grad = torch.randn_like(out)
    leaves = list(stack.parameters()) + list(lift.parameters())
    got = [out.detach()] + list(torch.autograd.grad(out, leaves, grad))
    if channels == 64:
        dims = list(stack_dims(windows.shape[0], window, bins, params))
        assert any(plan(hip.AX_MCORR, 4, 1, d)["joint"] for d in dims[1:])
    # the flags: a layer's output is that of the stack that ends there
    flags = []
    with torch.no_grad():
        for k in range(1, layers + 1):
            shorter = ConvStackParams(**{**vars(params), "layers": k})
            part = ConvStack(window, bins, shorter).cuda()
            for a, b in zip(part.convs, stack.convs):
                a.load_state_dict(b.state_dict())
            flags.append(part(lift(windows)) > 0)
    assert torch.equal(flags[-1], out > 0)
    leaves64 = [p.detach().double().requires_grad_() for p in leaves]
    log_eps, log_tau = leaves64[-2:]
    t = torch.arange(1, window + 1, device="cuda", dtype=torch.float64).view(-1, 1)
    y = (log_eps.exp() + windows.double().abs()).log() * t ** log_tau.exp()
    y.retain_grad()
    first = y
    for i, (lay, d) in enumerate(zip(stack.plan, stack_dims(windows.shape[0], window, bins, params))):
        y = _layer64(y, leaves64[2 * i], leaves64[2 * i + 1], lay, d[7:9]) * flags[i]
    y.backward(grad.double())
    want = [y.detach()] + [p.grad for p in leaves64]
    # the lift's gradients are sums that nearly cancel: their scale is the 2-norm of what is added
    scales = [float(w.norm()) for w in want[:-2]]
    inner = first.grad * t ** log_tau.detach().exp()
    a = log_eps.detach().exp() + windows.double().abs()
    scales += [float((inner * log_eps.detach().exp() / a).norm()),
               float((inner * a.log() * t.log() * log_tau.detach().exp()).norm())]
    # fp32 sums of up to 10^3 products a layer, `layers` of them behind each other, forward and backward: 2^-24 each, times
    # the square root of their number and of the layers, with room of three
    bound = 3 * 2 ** -24 * (2 * layers) ** 0.5 * 10
    for name, g, w, scale in zip(["out"] + [n for n, _ in stack.named_parameters()] + ["log_eps", "log_tau"], got, want, scales):
        assert float((g.double() - w).norm()) <= bound * scale, (name, float((g.double() - w).norm()) / scale)
