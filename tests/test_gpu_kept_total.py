"""The blocked inputs that layers' forward calls keep for their weight gradients have a bound in sum, behind which layers block
their input again: the same bits, and a network of many layers holds no more than the bound on top of what it saves."""
import pytest
import torch

import _mellin_hip as hip
import mconv

pytestmark = pytest.mark.gpu

KEPT_TOTAL = 1 << 30


@pytest.mark.parametrize("half", [False, True])
def test_all_live_graphs_together(half):
    torch.manual_seed(9950)
    layer = mconv.LCorrLCorr(32, 32, (3, 1)).cuda()
    x = torch.randn(32, 32, 1200, 40 if half else 14, device="cuda")
    if half:
        layer, x = layer.half(), x.half()
    want = None
    kept = hip.lib.mellin_layer_kept_bytes(hip.AX_LCORR, 2 if half else 4, 32, 32, 32, 3, 1, 1200, x.shape[3], 1198, x.shape[3],
                                           1, 1, 1, 1, 0, 0, 1, 1)
    assert kept > 64 << 20
    n = KEPT_TOTAL // kept + 6
    for _ in range(2):                                 # (what a graph held is there for the next ones)
        torch.cuda.synchronize()
        before, outs = torch.cuda.memory_allocated(), []
        for _ in range(n):
            outs.append(layer(x))
        held = torch.cuda.memory_allocated() - before - sum(o.numel() * o.element_size() for o in outs)
        # (each allocation is rounded up, to 2 MiB at most)
        assert KEPT_TOTAL - kept <= held <= KEPT_TOTAL + n * (4 << 20)
        for out in outs:
            got = torch.autograd.grad(out, [layer.weight, layer.bias], torch.ones_like(out))
            want = want or got
            assert all(torch.equal(a, b) for a, b in zip(got, want))
        del outs, out
    # graphs that nobody goes back through give it back as well
    out = [layer(x) for _ in range(n)]
    del out
    before = torch.cuda.memory_allocated()
    out = layer(x)
    assert torch.cuda.memory_allocated() - before >= kept + out.numel() * out.element_size()
