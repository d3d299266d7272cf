"""Float layers whose two gradients are section 2's, asked for together -- the sums that end the weight gradient then run in the
input gradient's last launch, whichever that is -- and one at a time: the same bits."""
import pytest
import torch

import _mellin_hip as hip
import mconv
from test_gpu_kept_inputs import dims_of

CASES = [
    # (module, channels in and out, kernel, input size, s, d, p, r, batch), by the input gradient's kernels (ROUTES)
    (mconv.LCorrLCorr, 3, 64, (8, 4), (128, 41), (1, 1), (1, 1), (0, 0), (0, 0), 32),      # strips, whose boundary rows are summed
    (mconv.LCorrLCorr, 1, 40, (5, 3), (301, 37), (1, 1), (1, 1), (2, 1), (2, 1), 16),
    (mconv.LCorrLCorr, 2, 64, (5, 3), (200, 30), (1, 1), (1, 1), (2, 1), (2, 1), 32),
    (mconv.LCorrLCorr, 3, 48, (3, 3), (300, 60), (2, 1), (1, 1), (1, 1), (1, 1), 32),
    (mconv.LCorrLCorr, 6, 40, (5, 4), (365, 60), (1, 1), (1, 1), (0, 2), (0, 2), 16),
    (mconv.MCorrLCorr, 3, 64, (8, 4), (512, 41), (1, 1), (1, 1), (0, 0), (0, 0), 32),      # taps, folded
    (mconv.MCorrLCorr, 1, 64, (5, 3), (10, 41), (1, 1), (1, 1), (2, 1), (4, 1), 1177),
    (mconv.MCorrLCorr, 7, 33, (4, 4), (300, 20), (1, 1), (1, 1), (1, 1), (50, 2), 16),
    (mconv.LCorrLCorr, 15, 12, (8, 4), (297, 20), (1, 1), (1, 1), (0, 2), (0, 2), 16),     # two passes, the second a fold
    (mconv.MCorrLCorr, 15, 12, (6, 2), (106, 60), (1, 1), (1, 1), (1, 1), (0, 1), 16),
    (mconv.LCorr1d, 3, 100, 11, (8088,), 1, 1, 1, 1, 8),                                   # strips of one column
    (mconv.LCorr1d, 2, 128, 8, (3838,), 2, 1, 1, 1, 32),
]
ROUTES = ["mfma-fused"] * 5 + ["mfma-taps+fold"] * 3 + ["mfma+fold"] * 2 + ["mfma-fused"] * 2


@pytest.mark.parametrize("case", CASES, ids=range(len(CASES)))
def test_last_launches_are_shared(case):
    """Both gradients need workspace -- partial sums of the weights; rows that strips share, or products to fold -- and have it
    side by side."""
    kind, dims = dims_of(case)
    both, one, other = (hip.lib.mellin_layer_backward_workspace(kind, 4, want, *dims) for want in (3, 1, 2))
    assert one > 0 and other > 0 and both == one + other


@pytest.mark.gpu
@pytest.mark.parametrize("relu", [False, True])
@pytest.mark.parametrize("case", CASES, ids=range(len(CASES)))
def test_gradients_together_and_apart(case, relu):
    cls, ci, co, k, size, s, d, p, r, n = case
    torch.manual_seed(9400 + CASES.index(case))
    layer = cls(ci, co, k, s=s, d=d, p=p, r=r).cuda()
    x = torch.randn(n, ci, *size, device="cuda", requires_grad=True)
    leaves = [x, layer.weight, layer.bias]
    out = layer(x, activation="relu" if relu else None)
    grad = torch.randn_like(out)
    together = torch.autograd.grad(out, leaves, grad, retain_graph=True)
    again = torch.autograd.grad(out, leaves, grad, retain_graph=True)
    apart = [torch.autograd.grad(out, [x], grad, retain_graph=True)[0]]
    assert hip.last_variant() == ROUTES[CASES.index(case)]
    apart += list(torch.autograd.grad(out, leaves[1:], grad))
    for a, b, c in zip(together, again, apart):
        assert torch.equal(a, b) and torch.equal(a, c)
