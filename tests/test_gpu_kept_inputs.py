"""Training steps whose weight gradient reads the blocked input that the forward call has kept, against the same steps that
block it again (hooks on saved tensors keep nothing): the same kernels on the same values, so the same bits."""
import pytest
import torch

import _mellin_hip as hip
import mconv

CASES = [
    # (module, channels in and out, kernel, input size, s, d, p, r, batch)
    (mconv.MCorr1d, 41, 128, 8, (391,), 1, 1, 3, 0, 300),
    (mconv.LCorr1d, 17, 33, 3, (1001,), 2, 2, 1, 1, 300),
    (mconv.MCorrLCorr, 64, 40, (3, 3), (31, 11), (1, 1), (2, 1), (2, 1), (2, 1), 300),
    (mconv.LCorrLCorr, 16, 96, (5, 3), (33, 37), (1, 1), (1, 1), (2, 1), (2, 1), 300),
]


def dims_of(case):
    cls, ci, co, k, size, s, d, p, r, n = case
    two = lambda v, unit: list(v) if isinstance(v, tuple) else [v, unit]       # noqa: E731
    k, s, d, p, r = two(k, 1), two(s, 1), two(d, 1), two(p, 0), two(r, 0)
    g = list(size) + [1] * (2 - len(size))
    mellin = cls in (mconv.MCorr1d, mconv.MCorrLCorr)
    valid = mconv.mcorr_valid_size if mellin else mconv.lcorr_valid_size
    h = [valid(k[0], g[0], s[0], d[0], p[0]) + r[0], mconv.lcorr_valid_size(k[1], g[1], s[1], d[1], p[1]) + r[1]]
    return hip.AX_MCORR if mellin else hip.AX_LCORR, [n, ci, co, *k, *g, *h, *s, *d, *p, 1, 1]


@pytest.mark.parametrize("elem_bytes", [4, 2])
@pytest.mark.parametrize("case", CASES, ids=range(len(CASES)))
def test_what_is_kept_leaves_the_scratch_memory(case, elem_bytes):
    kind, dims = dims_of(case)
    n, ci, _, _, _, gx, gy = dims[:7]
    kept = hip.lib.mellin_layer_kept_bytes(kind, elem_bytes, *dims)
    assert kept == -(-n * -(-ci // 8) * (gx * gy + 1) * (48 if elem_bytes == 4 else 16) // 256) * 256
    for name, args in (("forward", []), ("backward", [7])):
        with_, without = (getattr(hip.lib, "mellin_layer_" + name + w)(kind, elem_bytes, *args, *dims) for w in ("_kept_workspace", "_workspace"))
        assert without - with_ == kept
    few = list(dims)
    few[1] = 3                                         # section 2's forward pass
    assert hip.lib.mellin_layer_kept_bytes(kind, elem_bytes, *few) == 0
    for batch in (-(-(n << 28) // kept) + 1, n * (10 << 20) // kept - 1):           # more than 256 MiB, less than 10
        assert hip.lib.mellin_layer_kept_bytes(kind, elem_bytes, batch, *dims[1:]) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["float", "half", "autocast"])
@pytest.mark.parametrize("case", CASES, ids=range(len(CASES)))
def test_kept_inputs_change_nothing(case, kind):
    cls, ci, co, k, size, s, d, p, r, n = case
    assert hip.lib.mellin_layer_kept_bytes(dims_of(case)[0], 4 if kind == "float" else 2, *dims_of(case)[1]) > 0
    torch.manual_seed(9900 + CASES.index(case))
    layer = cls(ci, co, k, s=s, d=d, p=p, r=r).cuda()
    if kind == "half":
        layer = layer.half()
    x = torch.randn(n, ci, *size, device="cuda", dtype=torch.float32 if kind == "float" else torch.float16, requires_grad=True)
    leaves, grad, results = [x, layer.weight, layer.bias], None, []
    for hooked in (False, True):
        with torch.autocast("cuda", torch.float16, enabled=kind == "autocast"):
            if hooked:
                with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
                    out = layer(x)
            else:
                out = layer(x)
        grad = torch.randn_like(out) if grad is None else grad
        for again in (True, False):                    # (what is kept is there for a second backward call too)
            results.append([out.detach()] + list(torch.autograd.grad(out, leaves, grad, retain_graph=again)))
        with pytest.raises(RuntimeError):              # (and gone with the rest of the graph)
            torch.autograd.grad(out, leaves, grad)
    for other in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))
    # an input that has changed since is refused as before, and a layer that does not learn needs its input's gradient only
    base = x.detach().clone()
    out = layer(base) if kind != "autocast" else None
    if out is not None:
        base.add_(1)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            torch.autograd.grad(out, [layer.weight], grad)
    layer.requires_grad_(False)
    with torch.autocast("cuda", torch.float16, enabled=kind == "autocast"):
        (gx,) = torch.autograd.grad(layer(x), [x], grad)
    assert torch.equal(gx, results[0][1])
