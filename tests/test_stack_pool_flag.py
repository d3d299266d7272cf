"""`mellin_stack_layer.pool`: whatever is not zero pools behind an inner layer; the last layer is an output layer without a ReLU
where it is MELLIN_STACK_NO_RELU, and nothing else but zero; nothing pools behind the first."""
import ctypes

import pytest
import torch

import _mellin_hip as hip

NO_RELU = 2
POOLS = [1, 2, 3, 255, -1]


class _Layer(ctypes.Structure):
    _fields_ = [("dims", ctypes.c_int64 * 17), ("pool", ctypes.c_int)] + [
        (name, ctypes.c_void_p) for name in ("weight", "bias", "weight_half", "grad_weight", "grad_bias")]


def stack(pools, batch=2, bins=22):
    """Four linear layers of 24 channels, 3 x 3 taps, sizes kept."""
    layers, y = (_Layer * 4)(), bins
    for i, layer in enumerate(layers):
        layer.dims[:] = list(hip._dims(batch, 24, 24, (3, 3), (30, y), (30, y), (1, 1), (1, 1), (1, 1), (1, 1)))
        layer.pool = pools[i]
        y = y // 2 if i in (1, 2) and pools[i] else y
    return layers, y


def sizes(layers, elem_bytes, train=1):
    got = [ctypes.c_size_t() for _ in range(3)]
    if not hip.lib.mellin_stack_bytes(hip.AX_LCORR, elem_bytes, train, 4, layers, *(ctypes.addressof(s) for s in got)):
        return None
    return [s.value for s in got]


@pytest.mark.parametrize("elem_bytes", [4, 2])
@pytest.mark.parametrize("train", [0, 1])
def test_values_of_pool(elem_bytes, train):
    for inner in ((1, 0), (0, 1), (1, 1)):
        want = sizes(stack([0, *inner, 0])[0], elem_bytes, train)
        assert want and (not train or want != sizes(stack([0, 0, 0, 0])[0], elem_bytes, train))
        for flag in POOLS:
            pools = [0] + [flag * p for p in inner]
            assert sizes(stack(pools + [0])[0], elem_bytes, train) == want
            assert sizes(stack(pools + [NO_RELU])[0], elem_bytes, train) == want
    for flag in POOLS:
        assert sizes(stack([flag, 0, 0, 0])[0], elem_bytes, train) is None
        assert (sizes(stack([0, 0, 0, flag])[0], elem_bytes, train) is None) == (flag != NO_RELU)


@pytest.mark.gpu
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("bins", [22, 23])              # pooled by the products themselves; by a pass of its own in front of the second
def test_all_values_pool_alike(bins, half):
    dtype, elem = (torch.float16, 2) if half else (torch.float32, 4)
    torch.manual_seed(9960)
    weights = [torch.randn(24, 24, 3, 3, device="cuda").mul_(0.1).to(dtype) for _ in range(4)]
    inp = torch.randn(2, 24, 30, bins, device="cuda").to(dtype)
    want = None
    for flag in POOLS:
        layers, y = stack([0, flag, flag, 0], bins=bins)
        grads = [torch.zeros_like(w) for w in weights]
        for layer, w, g in zip(layers, weights, grads):
            layer.weight, layer.grad_weight = w.data_ptr(), g.data_ptr()
        out = torch.zeros(2, 24, 30, y, device="cuda", dtype=dtype)
        gi = torch.zeros_like(inp)
        need = sizes(layers, elem)
        saved, fw, bw = (torch.empty(max(n, 1), dtype=torch.uint8, device="cuda") for n in need)
        hip._check(hip.lib.mellin_stack_forward(hip.AX_LCORR, elem, 1, 4, layers, hip._dp(inp), hip._dp(out), hip._dp(saved), need[0],
                                                hip._dp(fw), need[1], hip._stream(inp.device)))
        hip._check(hip.lib.mellin_stack_backward(hip.AX_LCORR, elem, 4, layers, hip._dp(inp), hip._dp(out), hip._dp(out), hip._dp(saved),
                                                 need[0], hip._dp(gi), hip._dp(bw), need[2], hip._stream(inp.device)))
        got = [out, gi] + grads
        if want is None:
            want = got
            assert bool((out > 0).any()) and all(bool(g.isfinite().all()) and bool(g.any()) for g in got)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
