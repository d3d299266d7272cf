"""Which tiles the blocked kernels take for a pass (`mellin_layer_plan`; the plans are made on the host)."""
import ctypes
import random
import time

import pytest

import _mellin_hip as hip
import mconv
from conv_stack import ConvStackParams, layer_plan

WORDS = "mt nt wm wk joint F G whole rest slices".split()


def stack_dims(batch, frames, bins, params):
    """The dimensions of a stack's layers as the library's entry points take them."""
    x, y = frames, bins
    for lay in layer_plan(params, frames, bins):
        (kx, ky), s, d, p, r = lay["kernel"], lay["s"], lay["d"], lay["p"], lay["r"]
        valid = mconv.mcorr_valid_size if params.mellin else mconv.lcorr_valid_size
        ox, oy = valid(kx, x, s[0], d[0], p[0]) + r[0], mconv.lcorr_valid_size(ky, y, s[1], d[1], p[1]) + r[1]
        yield [batch, lay["in_channels"], lay["out_channels"], kx, ky, x, y, ox, oy, *s, *d, *p, 1, 1]
        x, y = lay["out_size"]


def plan(kind, elem_bytes, gradient, dims):
    words = (ctypes.c_int * len(WORDS))()
    if not hip.lib.mellin_layer_plan(kind, elem_bytes, gradient, *dims, words):
        return None
    return dict(zip(WORDS, words))


WANT_INPUT, WANT_WEIGHT, WANT_BIAS, WANT_RELU = 1, 2, 4, 8
BIAS_OWN, BIAS_BESIDE_WEIGHT, BIAS_PACKED = 1, 2, 3
FIRST_OWN, FIRST_BLOCKS, FIRST_TILES = 0, 1, 2


def bias_route(kind, elem_bytes, want, dims):
    """Where a layer's bias gradient is made: BIAS_*."""
    return hip.lib.mellin_layer_bias_route(kind, elem_bytes, want, *dims)


def first_layer(kind, elem_bytes, dims):
    """How a layer runs as the first of a stack: FIRST_*."""
    return hip.lib.mellin_stack_first_layer(kind, elem_bytes, *dims)


# (kernel, channels, layers, batch, frames, bins)
SMALL_IMAGES = [((5, 3), 64, 5, 1177, 10, 41), ((5, 3), 64, 3, 300, 10, 41), ((5, 3), 128, 3, 250, 10, 40), ((4, 3), 128, 4, 200, 7, 23)]


@pytest.mark.parametrize("elem_bytes", [4, 2])
@pytest.mark.parametrize("case", SMALL_IMAGES)
def test_joint_tiles_are_for_input_gradients(case, elem_bytes):
    """The order of a forward pass's sums decides which values a ReLU lets through."""
    kernel, channels, layers, batch, frames, bins = case
    params = ConvStackParams(layers=layers, kernel_time=kernel[0], kernel_freq=kernel[1], initial_channels=channels, factor_schedule=2,
                             time_factor=2)
    dims = list(stack_dims(batch, frames, bins, params))[1:]
    plans = [[plan(hip.AX_MCORR, elem_bytes, gradient, d) for d in dims] for gradient in (0, 1)]
    assert not any(p["joint"] for p in plans[0])
    assert any(p["joint"] for p in plans[1])


class _StackLayer(ctypes.Structure):
    _fields_ = [("dims", ctypes.c_int64 * 17), ("pool", ctypes.c_int)] + [(n, ctypes.c_void_p) for n in "weight bias half gw gb".split()]


def stack_bytes(batch, frames, bins, params, elem_bytes, train):
    """What a stack's calls ask for: bytes of what is kept, of the forward and of the backward workspace."""
    layers, sizes = (_StackLayer * params.layers)(), [ctypes.c_size_t() for _ in range(3)]
    for layer, dims in zip(layers, stack_dims(batch, frames, bins, params)):
        layer.dims[:] = dims
    kind = hip.AX_MCORR if params.mellin else hip.AX_LCORR
    assert hip.lib.mellin_stack_bytes(kind, elem_bytes, train, params.layers, ctypes.cast(layers, ctypes.c_void_p), *map(ctypes.byref, sizes))
    return [size.value for size in sizes]


@pytest.mark.parametrize("elem_bytes", [4, 2])
@pytest.mark.parametrize("c_in, kernel, frames, batch, own", [
    (1, (4, 4), 780, 32, False),                       # the tiled kernel stores the second layer's input
    (24, (4, 4), 100, 4, False),                       # the blocked kernels do
    (5, (5, 3), 780, 32, True),                        # float: staged in chunks of channels, and laid out afterwards
])
def test_first_layers_output_takes_workspace_where_it_is_a_tensor(c_in, kernel, frames, batch, own, elem_bytes):
    params = ConvStackParams(layers=2, kernel_time=kernel[0], kernel_freq=kernel[1], initial_channels=32, factor_schedule=2,
                             time_factor=1, in_channels=c_in)
    n, _, channels, _, _, ngx, ngy, nhx, nhy = next(iter(stack_dims(batch, frames, 41, params)))[:9]
    forward = stack_bytes(batch, frames, 41, params, elem_bytes, 1)[1]
    # (besides: where the blocked kernels take the first layer, its signal in their layout)
    signal = n * c_in * (ngx * ngy + 1) * (6 if elem_bytes == 4 else 2) if c_in >= 16 else 0
    assert (forward - signal >= n * channels * nhx * nhy * elem_bytes) == (own and elem_bytes == 4)


def test_new_sizes_are_planned_in_little_time():
    """A batch's longest utterance changes from step to step: what the choice of tiles takes comes on top of each.  (A count of all
    tiles of all images for every tile shape took 1150 us, this takes 35.)"""
    params = ConvStackParams(layers=10, kernel_time=4, kernel_freq=4, initial_channels=32, factor_schedule=3, channel_factor=2,
                             time_factor=1, in_channels=3)
    sizes, times = [ctypes.c_size_t() for _ in range(3)], []
    for frames in range(640, 700):
        layers = (_StackLayer * params.layers)()
        for layer, dims in zip(layers, stack_dims(32, frames, 41, params)):
            layer.dims[:] = dims
        begin = time.perf_counter()
        assert hip.lib.mellin_stack_bytes(hip.AX_MCORR, 4, 1, params.layers, ctypes.cast(layers, ctypes.c_void_p), *map(ctypes.byref, sizes))
        times.append(time.perf_counter() - begin)
    assert sorted(times)[len(times) // 4] < 3e-4, sorted(times)


def test_every_slice_has_a_stage():
    """A slice without channels would still run a stage, on channels that are another's."""
    rng = random.Random(9970)
    size = lambda low, high: int(round(low * (high / low) ** rng.random()))      # noqa: E731
    seen = {"slices": 0, "gradients by shared tiles": 0}
    for _ in range(4000):
        kind, c_in, c_out, batch = rng.choice((hip.AX_MCORR, hip.AX_LCORR)), size(8, 700), size(8, 700), size(1, 32)
        kx, ky, x, y = rng.randint(1, 8), rng.randint(1, 4), size(5, 800), rng.choice((1, 2, 5, 10, 41))
        d, p = rng.choice((1, 1, 2)), rng.randint(0, 3)
        valid = mconv.mcorr_valid_size if kind == hip.AX_MCORR else mconv.lcorr_valid_size
        ox, oy = valid(kx, x, 1, d, p) + (0 if kind == hip.AX_MCORR else p), mconv.lcorr_valid_size(ky, y, 1, 1, ky // 2) + ky // 2
        if ox < 1 or oy < 1:
            continue
        dims = [batch, c_in, c_out, kx, ky, x, y, ox, oy, 1, 1, d, 1, p, ky // 2, 1, 1]
        for elem_bytes in (4, 2):
            for gradient in (0, 1, 2):
                got = plan(kind, elem_bytes, gradient, dims)
                if got and got["rest"]:
                    groups = (c_out if gradient == 1 else c_in) + 7 >> 3
                    assert groups % got["G"] == 0 and 1 <= got["slices"] <= groups // got["G"], (dims, elem_bytes, gradient, got)
                    seen["slices"] += 1
                    seen["gradients by shared tiles"] += gradient == 1 and got["wk"] > 1
    assert all(n > 200 for n in seen.values()), seen


@pytest.mark.parametrize("elem_bytes", [4, 2])
def test_pooled_passes_of_even_columns_have_the_layers_own_plan(elem_bytes):
    """Such a plan is taken from the one without pooling, not made again."""
    params = ConvStackParams(layers=10, kernel_time=4, kernel_freq=4, initial_channels=32, factor_schedule=3, channel_factor=2,
                             time_factor=1, in_channels=3)
    for mellin in (True, False):
        params.mellin = mellin
        kind, pooled = hip.AX_MCORR if mellin else hip.AX_LCORR, 0
        for batch, frames, bins in ((1, 337, 40), (32, 780, 20), (3, 100, 10), (7, 61, 2)):
            for dims in list(stack_dims(batch, frames, bins, params))[1:]:
                if dims[8] % 2:
                    continue
                words = [(ctypes.c_int * len(WORDS))() for _ in range(2)]
                took = [hip.lib.mellin_layer_plan(kind, elem_bytes, gradient, *dims, w) for gradient, w in zip((0, 2), words)]
                assert took[0] == (took[1] > 0) and list(words[0]) == list(words[1])
                pooled += took[1] == 2
        assert pooled
