"""Packing with one position a thread (few blocks) and with four: planes around the edges of a block's positions, on either side
of the number of blocks that decides, against the same sums in float64."""
import pytest
import torch

import mconv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("plane", [1, 255, 256, 257, 1023, 1024, 1025])
@pytest.mark.parametrize("batch", [1, 300, 700])               # 2 groups of channels in, 3 out: 1024 blocks of four positions between
def test_planes_at_the_edges_of_blocks(batch, plane, half):
    torch.manual_seed(9800 + plane)
    dtype = torch.float16 if half else torch.float32
    layer = mconv.LCorr1d(16, 23, 1).cuda().to(dtype)
    x = torch.randn(batch, 16, plane, device="cuda", dtype=dtype, requires_grad=True)
    leaves = [x, layer.weight, layer.bias]
    with torch.no_grad():
        layer.bias.fill_(0.1)
    out = layer(x, activation="relu")
    grad = torch.randn_like(out)
    got = [out.detach()] + list(torch.autograd.grad(out, leaves, grad))
    w, b, xd = layer.weight.detach().double()[:, :, 0], layer.bias.detach().double(), x.detach().double()
    masked = torch.where(out.detach() > 0, grad, 0).double()
    rows, cols = (t.transpose(0, 1).flatten(1) for t in (masked, xd))
    want = [torch.relu(torch.matmul(w, xd) + b[:, None]), torch.matmul(w.t().contiguous(), masked), (rows @ cols.t())[:, :, None], rows.sum(1)]
    # one rounding of results to half (2^-11); fp32 products and sums of up to 7e5 terms in many partial sums: a few 2^-24 each
    tol = 2.0 ** -11 if half else 1e-5
    for a, c in zip(got, want):
        assert a.shape == c.shape and a.dtype == dtype
        assert float((a.double() - c).norm()) <= tol * float(c.norm()) + 1e-12
