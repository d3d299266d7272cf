"""`ConvStack` through one call per direction (tensors blocked from layer to layer, ReLU masks, bias gradients and pooling
inside the kernels) against the same layers called one by one, which the checker covers."""
import ctypes
import io

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import _mellin_hip as hip
import mconv
from conv_stack import ConvStack, ConvStackParams

pytestmark = pytest.mark.gpu

CASES = [
    # (mellin, layers, kernel, channels, schedule, channel_factor, time_factor, pool_every, c_in, batch, frames, bins)
    (True, 2, (4, 4), 16, 2, 1, 1, 0, 3, 1, 37, 13),       # one blocked layer, few tiles: slices as the last layer's output
    (True, 5, (4, 4), 32, 3, 2, 1, 2, 3, 1, 200, 41),      # few tiles: slices with a mask, blocked and dense; odd columns pooled
    (False, 4, (5, 2), 20, 2, 1, 2, 3, 1, 20, 400, 20),    # channels that do not fill their last group
    (True, 4, (3, 3), 70, 2, 2, 2, 0, 1, 8, 100, 40),      # channels past a tile, strides, classes of rows
    (False, 7, (3, 4), 64, 3, 2, 1, 3, 3, 9, 90, 33),      # two poolings
    (True, 3, (5, 3), 64, 2, 1, 2, 0, 1, 300, 10, 41),     # windows: many small images
]


@pytest.mark.parametrize("half", [False, True], ids=["f32", "amp"])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_stack_in_one_call_matches_layer_by_layer(case, half):
    mellin, layers, kernel, channels, schedule, cf, tf, every, c_in, batch, frames, bins = case
    torch.manual_seed(8000 + CASES.index(case))
    stack = ConvStack(frames, bins, ConvStackParams(
        layers=layers, mellin=mellin, kernel_time=kernel[0], kernel_freq=kernel[1], initial_channels=channels,
        factor_schedule=schedule, channel_factor=cf, time_factor=tf, in_channels=c_in,
        freq_pool_after=tuple(range(every, layers + 1, every)) if every else ())).cuda()
    with torch.no_grad():
        for conv in stack.convs:
            conv.weight.uniform_(-1, 1).mul_((6 / conv.weight[0].numel()) ** 0.5)
            conv.bias.uniform_(-0.1, 0.1)
    x = torch.randn(batch, c_in, frames, bins, device="cuda")
    leaves = list(stack.parameters())
    results, grad = [], None
    for one_call in (True, False):
        hooks = [] if one_call else [conv.register_forward_hook(lambda *a: None) for conv in stack.convs]
        xg = x.clone().requires_grad_()
        with torch.autocast("cuda", torch.float16, enabled=half):
            with torch.no_grad():
                served = stack(xg)
            out = stack(xg)
        last = out.grad_fn.next_functions[0][0] if every and layers % every == 0 else out.grad_fn
        assert ("StackBackward" in last.name()) == one_call
        grad = torch.randn_like(out) if grad is None else grad
        grads = torch.autograd.grad(out, leaves + [xg], grad)
        assert torch.equal(served, out)
        assert all(g.dtype == torch.float32 for g in grads)
        results.append([out.detach()] + list(grads))
        for h in hooks:
            h.remove()
    for got, want in zip(*results):
        rel = float((got.double() - want.double()).norm() / want.double().norm())
        assert rel <= (2e-3 if half else 2e-6), rel


def test_stack_gives_the_gradients_that_are_asked_for():
    stack = ConvStack(60, 20, ConvStackParams(layers=4, mellin=True, kernel_time=3, kernel_freq=3, initial_channels=24,
                                              factor_schedule=2, time_factor=1, in_channels=3)).cuda()
    x = torch.randn(2, 3, 60, 20, device="cuda", requires_grad=True)
    out = stack(x)
    grad = torch.randn_like(out)
    leaves = list(stack.parameters())
    full = torch.autograd.grad(out, leaves + [x], grad, retain_graph=True)
    again = torch.autograd.grad(out, leaves + [x], grad, retain_graph=True)
    assert all(torch.equal(a, b) for a, b in zip(full, again))
    for pick in ([0], [5], [6], [7], [2, 3], [len(leaves)]):
        some = torch.autograd.grad(out, [(leaves + [x])[i] for i in pick], grad, retain_graph=True)
        assert all(torch.equal(some[k], full[i]) for k, i in enumerate(pick))
    stack.convs[0].weight.requires_grad_(False)
    stack.convs[0].bias.requires_grad_(False)
    out = stack(x.detach())
    out.backward(grad)
    assert stack.convs[0].weight.grad is None and torch.equal(stack.convs[1].weight.grad, full[2])


def _small_stack():
    torch.manual_seed(5)
    stack = ConvStack(60, 20, ConvStackParams(layers=4, mellin=True, kernel_time=3, kernel_freq=3, initial_channels=24,
                                              factor_schedule=2, time_factor=1, in_channels=3)).cuda()
    return stack, torch.randn(2, 3, 60, 20, device="cuda", requires_grad=True)


def test_hooks_on_saved_tensors_see_the_layers_own():
    stack, x = _small_stack()
    want = torch.autograd.grad(stack(x).square().sum(), list(stack.parameters()) + [x])
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t.dtype), t.cpu())[1], lambda t: t.cuda()):
        out = stack(x)
    assert "StackBackward" not in out.grad_fn.name() and set(seen) == {torch.float32}
    got = torch.autograd.grad(out.square().sum(), list(stack.parameters()) + [x])
    for a, b in zip(got, want):
        assert float((a - b).norm()) <= 4e-6 * float(b.norm())     # (two orders of float32 sums, through four layers)
    layer = stack.convs[1]
    seen.clear()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(tuple(t.shape)), t)[1], lambda t: t):
        layer(torch.randn(2, 24, 60, 20, device="cuda", requires_grad=True), activation="relu")
    assert len(seen) == 3                                          # input, weight, output


def test_settings_changed_between_the_directions():
    stack, x = _small_stack()
    grad = torch.randn_like(stack(x))
    leaves = list(stack.parameters()) + [x]
    want = torch.autograd.grad(stack(x), leaves, grad)
    out = stack(x)
    assert "StackBackward" in out.grad_fn.name()
    try:
        hip.set_math(hip.MATH_FP32)
        got = torch.autograd.grad(out, leaves, grad)
    finally:
        hip.set_math(hip.MATH_BF16X3)
    for a, b in zip(got, want):
        assert float((a - b).norm()) <= 2e-6 * float(b.norm())


def test_whoever_follows_the_calls_is_shown_the_autograd_function():
    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    stack, x = _small_stack()
    plain = stack(x)
    with Mode():
        out = stack(x)
        one = mconv.mcorrlcorr(x, stack.convs[0].weight)
    assert "StackBackward" in plain.grad_fn.name() and "Corr2dFunction" in out.grad_fn.name() and "Corr2dFunction" in one.grad_fn.name()
    assert float((out - plain).detach().norm()) <= 1e-6 * float(plain.detach().norm())
    for transform in (torch.func.vmap(lambda v: mconv.mcorrlcorr(v[None], stack.convs[0].weight)),
                      torch.func.grad(lambda v: mconv.mcorrlcorr(v, stack.convs[0].weight).sum())):
        with pytest.raises(RuntimeError):
            transform(x.detach())


def test_a_stack_read_from_a_file_runs():
    stack, x = _small_stack()
    file = io.BytesIO()
    torch.save(stack, file)                                        # (written and read here)
    file.seek(0)
    again = torch.load(file, weights_only=False)
    assert torch.equal(again(x), stack(x))


@pytest.mark.parametrize("half", [False, True], ids=["f32", "amp"])
@pytest.mark.parametrize("frozen,pool_after", [(4, ()), (5, (4,)), (3, (3,)), (4, (5,))])
def test_frozen_layers_below_keep_nothing(frozen, pool_after, half):
    torch.manual_seed(6)
    stack = ConvStack(400, 40, ConvStackParams(layers=6, mellin=True, kernel_time=3, kernel_freq=3, initial_channels=32, factor_schedule=7,
                                               in_channels=3, freq_pool_after=pool_after)).cuda()
    x = torch.randn(2, 3, 400, 40, device="cuda")
    grad, held, grads = None, [], []
    for n in (0, frozen):
        for conv in stack.convs[:n]:
            conv.requires_grad_(False)
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        with torch.autocast("cuda", torch.float16, enabled=half):
            out = stack(x)
        held.append(torch.cuda.memory_allocated() - before)
        grad = torch.randn_like(out) if grad is None else grad
        leaves = [p for conv in stack.convs[frozen:] for p in conv.parameters()]
        grads.append([out.detach()] + list(torch.autograd.grad(out, leaves, grad)))
        assert "StackBackward" in out.grad_fn.name()
        del out
    # what is kept then: the inputs of the layers that learn in blocks (six bytes a value in float32), a byte for each value
    # that was pooled above the first of them, the filters of half tensors, the output
    size, value = (2 if half else 4), (2 if half else 6)
    bins = [40 // 2 if pool_after and i + 1 >= pool_after[0] else 40 for i in range(6)]      # of a layer's output
    most = 32 * 2 * 400 * (sum(b * (value + 1) for b in bins[frozen - 1:5]) + bins[5] * size)
    assert held[1] <= most + (1 << 18), (held, most)
    assert held[1] < held[0]
    for a, b in zip(*grads):
        assert float((a.double() - b.double()).norm()) <= (2e-3 if half else 2e-6) * float(a.double().norm())


class _Layer(ctypes.Structure):
    """mellin_stack_layer of include/mellin_hip.h."""
    _fields_ = [("dims", ctypes.c_int64 * 17), ("pool", ctypes.c_int)] + [
        (name, ctypes.c_void_p) for name in ("weight", "bias", "weight_half", "grad_weight", "grad_bias")]


@pytest.mark.parametrize("mellin,channels,frames,half", [(True, 100, 337, False), (False, 36, 100, False), (True, 100, 337, True),
                                                         (False, 100, 337, True)])
def test_channels_past_the_last_are_zeros_whatever_the_scratch_memory_held(mellin, channels, frames, half):
    """One utterance, channel counts that are no multiple of eight: the layers' sums come in slices through the workspace, and
    the rest of a layer's last group of eight channels has no sums there.  What the scratch memory held -- large values, which
    are infinities in half precision, infinities and NaN -- must not pass into a result."""
    kind, elem, dtype = (hip.AX_MCORR if mellin else hip.AX_LCORR), (2 if half else 4), (torch.float16 if half else torch.float32)
    torch.manual_seed(70)
    stack = ConvStack(frames, 41, ConvStackParams(layers=5, mellin=mellin, initial_channels=channels, time_factor=1, in_channels=3,
                                                  freq_pool_after=(3,)))
    n, c, x, y = len(stack.plan), 3, frames, 41
    layers, tensors, sliced = (_Layer * n)(), [], []
    for i, (lay, conv) in enumerate(zip(stack.plan, stack.convs)):
        co, (nf, nhy) = lay["out_channels"], (lay["kernel"], lay["out_size"][1])
        nh = (lay["out_size"][0], y if lay["pool"] else nhy)
        dims = hip._dims(1, c, co, nf, (x, y), nh, lay["s"], lay["d"], lay["p"], (1, 1))
        w = torch.empty(co, c, *nf, device="cuda").uniform_(-1, 1).mul_((6 / (c * nf[0] * nf[1])) ** 0.5).to(dtype)
        b = torch.empty(co, device="cuda").uniform_(0, 0.1).to(dtype)
        gw, gb = torch.empty_like(w), torch.empty_like(b)
        layers[i].dims[:], layers[i].pool = list(dims), int(lay["pool"])
        layers[i].weight, layers[i].bias, layers[i].grad_weight, layers[i].grad_bias = (t.data_ptr() for t in (w, b, gw, gb))
        tensors.append((w, b, gw, gb))
        if i:
            # what a layer's workspace has beside the blocked signal and filter: the sums of slices
            unit, groups, up = (16 if half else 48), (c + 7) // 8, lambda v: (v + 255) // 256 * 256
            filters = 2 * ((co + 63) // 64) * (groups * nf[0] * nf[1] + 1) * 32 * unit + (8 * nh[0] if mellin else 0)
            sliced.append(hip.lib.mellin_layer_forward_workspace(kind, elem, *dims) - up(groups * (x * y + 1) * unit) - up(filters) > 0)
        c, x, y = co, lay["out_size"][0], nhy
    assert any(sliced[:-1])                            # (the last layer's output is not blocked)
    inp = torch.randn(1, 3, frames, 41, device="cuda").to(dtype)
    out = torch.empty(1, c, x, y, device="cuda", dtype=dtype)
    grad, gi = torch.randn_like(out), torch.empty_like(inp)
    sizes = [ctypes.c_size_t() for _ in range(3)]
    assert hip.lib.mellin_stack_bytes(kind, elem, 1, n, layers, *(ctypes.addressof(s) for s in sizes)) == 1
    saved, fw, bw = (torch.empty(max(s.value, 4) // 4, device="cuda") for s in sizes)
    results = []
    for held in (0.0, 1e30, float("inf"), float("nan")):
        for t in (saved, fw, bw):
            t.fill_(held)
        for t in [out, gi] + [g for ts in tensors for g in ts[2:]]:
            t.fill_(float("nan"))
        hip._check(hip.lib.mellin_stack_forward(kind, elem, 1, n, layers, hip._dp(inp), hip._dp(out), hip._dp(saved), sizes[0].value,
                                                hip._dp(fw), sizes[1].value, hip._stream(inp.device)))
        hip._check(hip.lib.mellin_stack_backward(kind, elem, n, layers, hip._dp(inp), hip._dp(out), hip._dp(grad), hip._dp(saved),
                                                 sizes[0].value, hip._dp(gi), hip._dp(bw), sizes[2].value, hip._stream(inp.device)))
        results.append([t.clone() for t in [out, gi] + [g for ts in tensors for g in ts[2:]]])
    assert all(bool(t.isfinite().all()) for t in results[0]) and bool((results[0][0] > 0).any())
    for other in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))
    # a forward call for gradients of the layers from the fourth on keeps less, and a backward call that wants more is refused
    fewer = [ctypes.c_size_t() for _ in range(3)]
    assert hip.lib.mellin_stack_bytes(kind, elem, 1 | 3 << 8, n, layers, *(ctypes.addressof(s) for s in fewer)) == 1
    assert fewer[0].value < sizes[0].value
    assert hip.lib.mellin_stack_backward(kind, elem, n, layers, hip._dp(inp), hip._dp(out), hip._dp(grad), hip._dp(saved),
                                         fewer[0].value, hip._dp(gi), hip._dp(bw), sizes[2].value, hip._stream(inp.device)) == 3
