"""What users of this package run, as cases that can be timed and whose results can be compared.

Three kinds of program, all through the public modules:

    layer    one convolution layer (`MCorr1d`, `LCorr1d`, `MCorrLCorr`, `LCorrLCorr`): a call
             without gradients, or a training step of it (output, input gradient and parameter
             gradients for an upstream gradient), in float32 or under ``torch.autocast``
    stack    `FrameClassifier`: the 2-D convolution stack over fbank features with its linear
             output layer, as a training step on frame labels or as a call without gradients
    windows  the acoustic model's own order: features of ragged utterances cut into windows and
             packed (`pack_windows`), `LogCompressionLift`, then the stack over the windows

The listed sizes are those of this repository's configurations (time_layers.py)
and tests, with one ragged size of each kind beside them; `draw` covers the ranges between.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "cnn-mellin_amd"))

import mconv  # noqa: E402
from conv_stack import ConvStack, ConvStackParams, FrameClassifier, layer_plan, pack_windows  # noqa: E402
from layers import LogCompressionLift  # noqa: E402

#: classes of the output layer: 61 phones and a blank
TARGETS = 62
#: a drawn case has at most this many multiply-adds in its forward pass, and this many values in
#: its largest tensor (about the widest listed layer and the larger listed stack)
MOST_MACS = 95e9
MOST_VALUES = 85e6


def _layer(name, op, batch, c_in, c_out, kernel, size, s=(1, 1), d=(1, 1), p=(0, 0), r=(0, 0), half=False,
           train=True, ragged=False):
    return dict(name=name, what="layer", op=op, batch=batch, c_in=c_in, c_out=c_out, kx=kernel[0], ky=kernel[1],
                tx=size[0], ty=size[1], sx=s[0], sy=s[1], dx=d[0], dy=d[1], px=p[0], py=p[1], rx=r[0], ry=r[1],
                half=half, train=train, ragged=ragged)


def _stack(name, batch, frames, bins, mellin, layers, kernel, channels, schedule, channel_factor, time_factor,
           pool_every, half=False, train=True, c_in=3):
    return dict(name=name, what="stack", batch=batch, tx=frames, ty=bins, mellin=mellin, layers=layers,
                kx=kernel[0], ky=kernel[1], channels=channels, schedule=schedule, channel_factor=channel_factor,
                time_factor=time_factor, pool_every=pool_every, half=half, train=train, c_in=c_in)


def _windows(name, batch, longest, bins, window, stride, mellin, layers, kernel, channels, schedule,
             channel_factor, time_factor, train=True):
    return dict(name=name, what="windows", batch=batch, longest=longest, ty=bins, tx=window, stride=stride,
                mellin=mellin, layers=layers, kx=kernel[0], ky=kernel[1], channels=channels, schedule=schedule,
                channel_factor=channel_factor, time_factor=time_factor, pool_every=0, half=False, train=train, c_in=1)


def listed():
    return [
        # configuration 1: a small 1-D Mellin layer called without gradients; nothing but latency
        _layer("mcorr1d small", "mcorr1d", 8, 3, 16, (16, 1), (256, 1), train=False),
        # configuration 2: 1-D layers over a batch of utterances of 100 to 780 frames, padded to 780;
        # the Mellin layer with p = 3 (outputs at all four residues), the linear one strided and dilated
        # and in half precision
        _layer("mcorr1d train", "mcorr1d", 32, 41, 128, (8, 1), (780, 1), p=(3, 0), ragged=True),
        _layer("lcorr1d train half", "lcorr1d", 32, 41, 128, (8, 1), (780, 1), s=(2, 1), d=(2, 1), half=True, ragged=True),
        # configuration 3, the benchmark: three channels of fbank features into 64
        _layer("mconv2d train", "mcorrlcorr", 32, 3, 64, (8, 4), (512, 41)),
        _layer("lconv2d train", "lcorrlcorr", 32, 3, 64, (8, 4), (512, 41)),
        # a ragged layer of the inner kind served in half precision: odd sizes on every axis, padded
        # on both, fewer images than the chip has dies
        _layer("lconv2d ragged infer half", "lcorrlcorr", 7, 33, 67, (5, 3), (333, 37), p=(2, 1), r=(2, 1), half=True, train=False),
        # configuration 4: the widest layer, linear in float32 and Mellin under autocast
        _layer("wide lconv2d train", "lcorrlcorr", 32, 128, 256, (3, 3), (256, 41), d=(2, 1), p=(2, 1), r=(2, 1)),
        _layer("wide mconv2d train half", "mcorrlcorr", 32, 128, 256, (3, 3), (256, 41), d=(2, 1), p=(2, 1), r=(2, 1), half=True),
        # configuration 5: training steps of the 10-layer stacks, 3 -> 256 channels, and one utterance
        # of an odd length decoded by the Mellin one
        _stack("mellin stack train", 32, 780, 41, True, 10, (4, 4), 32, 3, 2, 1, 3),
        _stack("linear stack train half", 32, 780, 41, False, 10, (4, 4), 32, 3, 2, 1, 3, half=True),
        _stack("mellin stack decode", 1, 337, 41, True, 10, (4, 4), 32, 3, 2, 1, 3, train=False),
        # the acoustic model as it trains: windows of ten frames every three, the stack's default layers
        _windows("windows train", 8, 780, 41, 10, 3, True, 5, (5, 3), 64, 2, 1, 2),
    ]


# ---------------------------------------------------------------------------
# drawn cases
# ---------------------------------------------------------------------------
def _log(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _draw_layer(rng):
    two = rng.random() < 0.6
    mellin = rng.random() < 0.5
    kx = rng.randint(3, 8) if two else rng.randint(3, 16)
    ky = rng.randint(2, 4) if two else 1
    px = rng.randint(0, 3)
    py = rng.randint(0, ky // 2) if two else 0
    rx = px if not mellin else rng.choice((0, 0, rng.randint(1, 8)))
    return _layer("", ("mcorrlcorr" if mellin else "lcorrlcorr") if two else ("mcorr1d" if mellin else "lcorr1d"),
                  _log(rng, 1, 32), rng.choice((1, 3, _log(rng, 4, 128), _log(rng, 4, 128))), _log(rng, 8, 256), (kx, ky),
                  (_log(rng, 100, 780), rng.choice((40, 41, rng.randint(10, 80))) if two else 1),
                  s=(rng.choice((1, 1, 2)), 1), d=(rng.choice((1, 1, 2)), 1), p=(px, py), r=(rx, py),
                  half=rng.random() < 0.35, train=rng.random() < 0.65, ragged=rng.random() < 0.5)


def _draw_stack(rng):
    train = rng.random() < 0.6
    return _stack("", _log(rng, 1, 32) if train else _log(rng, 1, 4), _log(rng, 100, 780), rng.choice((40, 41, rng.randint(20, 80))),
                  rng.random() < 0.5, rng.randint(3, 10), (rng.randint(3, 5), rng.randint(3, 4)), rng.choice((16, 24, 32, 64)),
                  rng.randint(2, 3), rng.randint(1, 2), rng.randint(1, 2), rng.choice((0, 3)), half=rng.random() < 0.4,
                  train=train, c_in=rng.choice((1, 3)))


def _draw_windows(rng):
    return _windows("", _log(rng, 1, 16), _log(rng, 100, 780), rng.choice((40, 41, rng.randint(20, 80))), rng.randint(5, 20),
                    rng.randint(1, 4), rng.random() < 0.5, rng.randint(2, 5), (rng.randint(3, 5), 3), rng.choice((16, 32, 64)),
                    2, rng.randint(1, 2), 2, train=rng.random() < 0.7)


def draw(rng):
    while True:
        kind = rng.random()
        case = _draw_layer(rng) if kind < 0.6 else _draw_stack(rng) if kind < 0.85 else _draw_windows(rng)
        try:
            plan = _geometry(case)
        except ValueError:                     # a stack whose output would be empty
            continue
        if any(min(lay["out"]) < 1 for lay in plan):
            continue
        if sum(lay["macs"] for lay in plan) > MOST_MACS or max(max(lay["values"]) for lay in plan) > MOST_VALUES or \
                sum(sum(lay["values"]) for lay in plan) > 6 * MOST_VALUES:
            continue
        del case["name"]
        return case


# ---------------------------------------------------------------------------
# sizes
# ---------------------------------------------------------------------------
def _taps(mellin, kernel, size, out, s, d, p):
    """(output, filter) index pairs of one axis that meet a value of the input."""
    h, f = np.arange(out)[:, None], np.arange(kernel)[None, :]
    if mellin:
        product = (h + s) * (f + d)
        return int(np.count_nonzero((product % (p + 1) == 0) & (product // (p + 1) - 1 < size)))
    at = s * h + d * f - p
    return int(np.count_nonzero((at >= 0) & (at < size)))


def _stack_params(case):
    every = case["pool_every"]
    return ConvStackParams(layers=case["layers"], mellin=case["mellin"], kernel_time=case["kx"], kernel_freq=case["ky"],
                           initial_channels=case["channels"], factor_schedule=case["schedule"],
                           channel_factor=case["channel_factor"], time_factor=case["time_factor"], in_channels=case["c_in"],
                           freq_pool_after=tuple(range(every, case["layers"] + 1, every)) if every else ())


def _lengths(case):
    """Utterance lengths: from 100 frames (or the longest, where that is shorter) to the longest, which is there."""
    longest = case["longest"] if case["what"] == "windows" else case["tx"]
    n = case["batch"]
    low = min(100, longest)
    return [longest - (i * (longest - low)) // max(1, n - 1) for i in range(n)]


def _images(case):
    if case["what"] != "windows":
        return case["batch"]
    return sum((length - 1) // case["stride"] + 1 for length in _lengths(case))


def _geometry(case):
    """One dict per layer: its output size, multiply-adds, and the values of its input, output and parameters."""
    n = _images(case)
    if case["what"] == "layer":
        layers = [dict(mellin=case["op"].startswith("m"), in_channels=case["c_in"], out_channels=case["c_out"],
                       kernel=(case["kx"], case["ky"]), s=(case["sx"], case["sy"]), d=(case["dx"], case["dy"]),
                       p=(case["px"], case["py"]), r=(case["rx"], case["ry"]), pool=False)]
    else:
        layers = [dict(lay, mellin=case["mellin"]) for lay in layer_plan(_stack_params(case), case["tx"], case["ty"])]
    x, y = case["tx"], case["ty"]
    plan = []
    for lay in layers:
        (kx, ky), s, d, p, r = lay["kernel"], lay["s"], lay["d"], lay["p"], lay["r"]
        valid = mconv.mcorr_valid_size if lay["mellin"] else mconv.lcorr_valid_size
        ox = valid(kx, x, s[0], d[0], p[0]) + r[0]
        oy = mconv.lcorr_valid_size(ky, y, s[1], d[1], p[1]) + r[1]
        ci, co = lay["in_channels"], lay["out_channels"]
        macs = n * ci * co * _taps(lay["mellin"], kx, x, ox, s[0], d[0], p[0]) * _taps(False, ky, y, oy, s[1], d[1], p[1])
        plan.append(dict(out=(ox, oy), macs=float(macs), values=(n * ci * x * y, n * co * ox * oy), weights=co * ci * kx * ky + co,
                         pool=lay["pool"]))
        x, y = ox, (oy // 2 if lay["pool"] else oy)
    return plan


def work(case):
    """Layer for layer: the forward pass reads the input and writes the output (which no chip keeps for
    the next layer at these sizes), a training step reads the upstream gradient and the input again (not
    for a layer alone, whose passes could share one reading) and writes the input's gradient; parameters
    are read, their gradients written.  The first layer of a stack over plain features has no input
    gradient.  Pooling keeps the larger of two."""
    plan = _geometry(case)
    size = 2 if case["half"] else 4
    values, macs, weights = 0.0, 0.0, 0
    for i, lay in enumerate(plan):
        x, out = lay["values"]
        passes, v = 1, x + out
        if case["train"]:
            first = i == 0 and case["what"] == "stack"
            passes += 1 if first else 2
            v += out + (0 if first else x) + (x if case["what"] != "layer" else 0)
        if lay["pool"]:
            v += (3 if case["train"] else 1.5) * out
        values += v
        macs += passes * lay["macs"]
        weights += lay["weights"] * (2 if case["train"] else 1)
    if case["what"] == "stack":
        n, (t, f) = case["batch"], plan[-1]["out"]
        rows = n * t
        wide = plan[-1]["values"][1] // rows // (2 if plan[-1]["pool"] and f > 1 else 1)
        macs += (3 if case["train"] else 1) * rows * wide * TARGETS
        weights += wide * TARGETS * (2 if case["train"] else 1)
    if case["what"] == "windows":
        values += plan[0]["values"][0] * (4 if case["train"] else 2)
    return {"bytes": size * values + 4.0 * weights, "flops": 2 * macs}


def tolerance(case):
    half = case["half"]
    if case["what"] == "layer":
        # float32 products summed in float32: sums of up to a million terms differ by their order;
        # half: one rounding (2^-11) of results whose exact sums agree
        return {"rel": 1e-3, "max": 5e-3} if half else {"rel": 1e-5, "max": 4e-4}
    if not case["train"]:
        return {"rel": 5e-3, "max": 0.05} if half else {"rel": 1e-5, "max": 4e-4}
    # behind every layer a ReLU, and pooling behind some: where a value lies within its rounding error
    # of the kink (or of its neighbour), another order of summation passes a whole gradient on or does
    # not.  A share e of such places changes a gradient by sqrt(e) in the 2-norm, layer upon layer, and
    # single values by as much as they are.  Two ways of forming the same float32 products measure 1e-3
    # on the 10-layer stack and 5e-3 on log_eps, whose gradient is one sum that nearly cancels; half
    # precision with another order of its float32 sums measures 1e-2.
    return {"rel": 0.03, "max": 0.9} if half else {"rel": 1e-2, "max": 0.5}


# ---------------------------------------------------------------------------
# a user's program
# ---------------------------------------------------------------------------
_MODULES = {"mcorr1d": mconv.MCorr1d, "lcorr1d": mconv.LCorr1d, "mcorrlcorr": mconv.MCorrLCorr, "lcorrlcorr": mconv.LCorrLCorr}


def _initialise(module, gen):
    """Kaiming-uniform weights for ReLU, which keep the variance through a deep stack as a trained
    network does, and biases of the layers' own range; log_eps and log_tau from N(0, 1)."""
    for m in module.modules():
        for name, p in m.named_parameters(recurse=False):
            with torch.no_grad():
                if name.startswith("log_"):
                    p.normal_(generator=gen)
                else:
                    bound = m.weight[0].numel() ** -0.5 * (6 ** 0.5 if name == "weight" else 1.0)
                    p.uniform_(-bound, bound, generator=gen)
    return module


def _zero_past(x, lengths, dim):
    t = torch.arange(x.shape[dim], device=x.device)
    keep = t[None, :] < torch.tensor(lengths, device=x.device)[:, None]
    return x.mul_(keep.view([x.shape[0]] + [-1 if i == dim else 1 for i in range(1, x.dim())]))


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    state = dict(case)
    if case["what"] == "layer":
        one = case["op"].endswith("1d")

        def pick(a):
            return case[a + "x"] if one else (case[a + "x"], case[a + "y"])
        state["model"] = _initialise(_MODULES[case["op"]](case["c_in"], case["c_out"], pick("k"), s=pick("s"), d=pick("d"),
                                                          p=pick("p"), r=pick("r")).to(dev), gen)
        x = torch.randn([case["batch"], case["c_in"], case["tx"]] + ([] if one else [case["ty"]]), device=dev, generator=gen)
        if case["ragged"]:
            _zero_past(x, _lengths(case), 2)
        # a layer's input and its upstream gradient come from neighbours that ran in the same precision
        kind = torch.float16 if case["half"] else torch.float32
        state["x"] = x.to(kind).requires_grad_(case["train"])
        if case["train"]:
            out = _geometry(case)[0]["out"]
            state["grad"] = torch.randn([case["batch"], case["c_out"], out[0]] + ([] if one else [out[1]]), device=dev,
                                        generator=gen).to(kind)
        return state
    stack = ConvStack(case["tx"], case["ty"], _stack_params(case))
    if case["what"] == "stack":
        state["model"] = _initialise(FrameClassifier(stack, TARGETS).to(dev), gen)
        state["x"] = _zero_past(torch.randn(case["batch"], case["c_in"], case["tx"], case["ty"], device=dev, generator=gen),
                                _lengths(case), 2)
        if case["train"]:
            state["labels"] = torch.randint(TARGETS, (case["batch"] * stack.out_size[0],), device=dev, generator=gen)
        return state
    state["lift"] = _initialise(LogCompressionLift(dim=2).to(dev), gen)
    state["model"] = _initialise(stack.to(dev), gen)
    lengths = _lengths(case)
    # filter bank energies: log-normal
    state["x"] = _zero_past(torch.randn(case["batch"], case["longest"], case["ty"], device=dev, generator=gen).exp_(), lengths, 1)
    state["lens"] = torch.tensor(lengths)
    if case["train"]:
        # the recurrent layers' gradient on the features (channels x bins of a window, summed over its frames)
        state["grad"] = torch.randn(_images(case), stack.out_channels * stack.out_size[1], device=dev, generator=gen)
    return state


def _features(state):
    windows, _ = pack_windows(state["x"], state["lens"], state["tx"], state["stride"])
    return state["model"](state["lift"](windows)).sum(2).flatten(1)


def run(state):
    model = state["model"]
    call = _features if state["what"] == "windows" else lambda st: st["model"](st["x"])
    if not state["train"]:
        with torch.no_grad(), torch.autocast("cuda", torch.float16, enabled=state["half"]):
            return call(state)
    leaves = list(model.parameters())
    if state["what"] == "windows":
        leaves += list(state["lift"].parameters())
    if state["x"].requires_grad:
        leaves.append(state["x"])
    for leaf in leaves:
        leaf.grad = None
    with torch.autocast("cuda", torch.float16, enabled=state["half"]):
        out = call(state)
    if state["what"] == "stack":
        loss = torch.nn.functional.nll_loss(out.flatten(0, 1), state["labels"])
        if state["half"]:
            loss = loss * 4096.0               # the loss scale that training in half precision takes
        loss.backward()
    else:
        out.backward(state["grad"])
    return [out.detach()] + [leaf.grad for leaf in leaves]
