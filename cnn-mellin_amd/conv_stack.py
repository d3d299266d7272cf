"""The convolutional front end of the reference's acoustic model, as a module.

`ConvStack` builds the layer list the way ``AcousticModel.__init__`` does
(models.py:277-339): per-layer stride / dilation / padding and, above all, the
extra output length ``r = expected - valid`` that pins every layer's output
size to ``input // factor`` (models.py:292-327; without it a stack of Mellin
layers shrinks to nothing after a few layers), and applies it the way
``AcousticModel.forward`` does (models.py:423-437): non-linearity after every
layer.  Two things go beyond the reference, both optional and off by default:
more than one input channel (the reference feeds one channel of windows; a
fbank batch with deltas has three), and a frequency max-pool after chosen
layers.  Layers are this package's `MCorrLCorr` (Mellin x linear) or
`LCorrLCorr` (linear x linear, in place of the reference's
``torch.nn.Conv2d``, models.py:329-338, with the same padding rule).
"""
from typing import Callable, List, Optional, Sequence, Tuple

import torch
from torch.utils._device import DeviceContext

import mconv
import _mellin_hip as _hip

_native_stack = _hip.native.stack
# hooks that PyTorch runs for every module
_GLOBAL_HOOKS = [getattr(torch.nn.modules.module, name) for name in (
    "_global_forward_hooks", "_global_forward_pre_hooks", "_global_backward_hooks", "_global_backward_pre_hooks")
    if hasattr(torch.nn.modules.module, name)]

__all__ = ["ConvStackParams", "ConvStack", "FrameClassifier", "layer_plan", "pack_windows"]


class _FreqMaxPool(torch.autograd.Function):
    """max_pool2d(x, (1, 2)) for dense float32 or float16 GPU tensors through the library's pair kernels:
    one byte per output is kept for the backward pass instead of PyTorch's 8-byte indices."""

    @staticmethod
    def forward(ctx, x):
        y, which = _hip.pool_pairs_forward(x.contiguous())
        ctx.save_for_backward(which)
        ctx.f = x.shape[-1]
        return y

    @staticmethod
    def backward(ctx, grad_y):
        (which,) = ctx.saved_tensors
        return _hip.pool_pairs_backward(grad_y.contiguous(), which, ctx.f)


def freq_max_pool(x: torch.Tensor) -> torch.Tensor:
    """Maximum over pairs of neighbouring frequency bins, ``max_pool2d(x, (1, 2))``."""
    if x.is_cuda and x.dtype in (torch.float32, torch.float16):
        return _FreqMaxPool.apply(x)
    return torch.nn.functional.max_pool2d(x, (1, 2))


class ConvStackParams:
    """The convolutional fields of ``AcousticModelParams`` (models.py:45-118)."""

    def __init__(self, layers: int = 5, mellin: bool = True, kernel_time: int = 5, kernel_freq: int = 3,
                 initial_channels: int = 64, factor_schedule: int = 2, channel_factor: int = 1,
                 time_factor: int = 2, freq_factor: int = 1,
                 nonlinearity: Callable[[torch.Tensor], torch.Tensor] = torch.relu,
                 in_channels: int = 1, freq_pool_after: Sequence[int] = (), seed: Optional[int] = None):
        self.layers, self.mellin = layers, mellin
        self.kernel_time, self.kernel_freq = kernel_time, kernel_freq
        self.initial_channels, self.factor_schedule = initial_channels, factor_schedule
        self.channel_factor, self.time_factor, self.freq_factor = channel_factor, time_factor, freq_factor
        self.nonlinearity = nonlinearity
        self.in_channels = in_channels
        self.freq_pool_after = tuple(freq_pool_after)     # 1-based layer numbers followed by max_pool (1, 2)
        self.seed = seed


def layer_plan(params: ConvStackParams, time_dim: int, freq_dim: int) -> List[dict]:
    """Per-layer geometry by the rule of models.py:277-339.

    Returns one dict per layer: in/out channels, kernel, s, d, p, r and the
    output extent (after the optional frequency pool)."""
    x, y = time_dim, freq_dim
    kx, ky = params.kernel_time, params.kernel_freq
    ci, co = params.in_channels, params.initial_channels
    up_c, decim_x, on_sy = params.channel_factor, params.time_factor, params.freq_factor
    px, py = (kx - 1) // 2, (ky - 1) // 2
    off_s = dy = off_dx = 1
    if params.mellin:
        on_sx, on_dx = 1, (decim_x - 1) * kx + 1
    else:
        on_sx, on_dx = decim_x, 1
    plan = []
    for layer_no in range(1, params.layers + 1):
        if layer_no % params.factor_schedule:             # "off": output size unchanged
            dx, sx, sy, Dx, Dy = off_dx, off_s, off_s, 1, 1
        else:                                             # "on": output size divided
            dx, sx, sy, co, Dx, Dy = on_dx, on_sx, on_sy, up_c * co, decim_x, on_sy
        if params.mellin:
            new_x = mconv.mcorr_valid_size(kx, x, sx, dx, px)
            rx = max(x // Dx, 1) - new_x
            new_y = mconv.lcorr_valid_size(ky, y, sy, dy, py)
            ry = max(y // Dy, 1) - new_y
            lay = dict(kind="mcorrlcorr", p=(px, py), r=(rx, ry))
            x, y = new_x + rx, new_y + ry
        else:
            # torch.nn.Conv2d with symmetric padding (px_, py_): left padding p, right padding r
            px_ = px if (x + 2 * px - kx) // sx + 1 > 0 else px + 1
            py_ = py if (y + 2 * py - ky) // sy + 1 > 0 else py + 1
            out_x, out_y = (x + 2 * px_ - kx) // sx + 1, (y + 2 * py_ - ky) // sy + 1
            rx = out_x - mconv.lcorr_valid_size(kx, x, sx, dx, px_)
            ry = out_y - mconv.lcorr_valid_size(ky, y, sy, dy, py_)
            lay = dict(kind="lcorrlcorr", p=(px_, py_), r=(rx, ry))
            x, y = out_x, out_y
        lay.update(in_channels=ci, out_channels=co, kernel=(kx, ky), s=(sx, sy), d=(dx, dy),
                   pool=layer_no in params.freq_pool_after)
        if lay["pool"]:
            y = y // 2
        lay["out_size"] = (x, y)
        if x <= 0 or y <= 0:
            raise ValueError("layer %d of the stack has an empty output (%d x %d)" % (layer_no, x, y))
        plan.append(lay)
        ci = co
    return plan


def pack_windows(x: torch.Tensor, lens: torch.Tensor, window_size: int, window_stride: int):
    """Feature batch ``(N, T, F)`` with lengths -> the windows the convolutions see.

    As ``AcousticModel.forward`` (models.py:395-411): pad ``window_size - 1`` frames at the
    end, cut windows of ``window_size`` frames every ``window_stride``, keep only the
    ``(len - 1) // stride + 1`` windows of each utterance that start on a real frame, and fuse
    utterance and window index (time-major, as ``pack_padded_sequence`` orders them).  Returns
    the windows ``(N', 1, window_size, F)``, the convolution stack's input, and the
    ``PackedSequence`` whose ``batch_sizes`` / ``unsorted_indices`` undo the packing."""
    if x.is_cuda:
        # one copy of the windows' index and one launch (None: tensors and lengths that are not for it)
        packed = _hip.native.pack_windows(x, lens, window_size, window_stride)
        if packed is not None:
            packed = torch.nn.utils.rnn.PackedSequence(*packed)
            return packed.data.unsqueeze(1), packed
    if window_size > 1:
        x = torch.nn.functional.pad(x, (0, 0, 0, window_size - 1))
    windows = x.unfold(1, window_size, window_stride).transpose(2, 3)      # (N, T', w, F)
    lens_ = torch.div(lens - 1, window_stride, rounding_mode="trunc") + 1
    packed = torch.nn.utils.rnn.pack_padded_sequence(windows, lens_.cpu(), batch_first=True,
                                                     enforce_sorted=False)
    return packed.data.unsqueeze(1).contiguous(), packed


class ConvStack(torch.nn.Module):
    """``x (N, C_in, T, F) -> (N, C_out, T', F')`` through the planned layers."""

    def __init__(self, time_dim: int, freq_dim: int, params: ConvStackParams):
        super().__init__()
        self.params = params
        self.plan = layer_plan(params, time_dim, freq_dim)
        self.convs = torch.nn.ModuleList()
        for lay in self.plan:
            cls = mconv.MCorrLCorr if lay["kind"] == "mcorrlcorr" else mconv.LCorrLCorr
            self.convs.append(cls(lay["in_channels"], lay["out_channels"], lay["kernel"], s=lay["s"],
                                  d=lay["d"], p=lay["p"], r=lay["r"]))
        if params.seed is not None:
            self.reset_parameters()

    @property
    def out_channels(self) -> int:
        return self.plan[-1]["out_channels"]

    @property
    def out_size(self) -> Tuple[int, int]:
        return self.plan[-1]["out_size"]

    def reset_parameters(self) -> None:
        if self.params.seed is not None:
            torch.manual_seed(self.params.seed)
        for conv in self.convs:
            conv.reset_parameters()

    def _plain(self) -> bool:
        """Whether calling the layers one by one would run nothing but them: no hooks, no replaced modules."""
        if any(_GLOBAL_HOOKS):
            return False
        cls = mconv.MCorrLCorr if self.params.mellin else mconv.LCorrLCorr
        for conv in self.convs:
            d = conv.__dict__
            if (type(conv) is not cls or "forward" in d or d["_forward_hooks"] or d["_forward_pre_hooks"] or
                    d["_backward_hooks"] or d["_backward_pre_hooks"]):
                return False
        return len(self.convs) == len(self.plan)

    def _fused(self) -> bool:
        return self.params.nonlinearity in (torch.relu, torch.nn.functional.relu)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        # ReLU, the reference's default (models.py:96-101), is applied by the convolution
        # kernel itself on the way out; any other callable runs as a pass of its own
        fused = self._fused()
        if fused and x.is_cuda and self._plain():
            # the whole stack in one call, its tensors in the kernels' layout from layer to layer
            kind = _hip.AX_MCORR if self.params.mellin else _hip.AX_LCORR
            # (a pool behind the last layer stays outside)
            pools = [bool(lay["pool"]) for lay in self.plan[:-1]] + [False]
            y = _native_stack(kind, x, [(conv.weight, conv.bias, conv.s, conv.d, conv.p, conv.r, pool)
                                        for conv, pool in zip(self.convs, pools)])
            if y is not None:
                return freq_max_pool(y) if self.plan[-1]["pool"] else y
        for lay, conv in zip(self.plan, self.convs):
            x = conv(x, activation="relu") if fused else self.params.nonlinearity(conv(x))
            if lay["pool"]:
                x = freq_max_pool(x)
        return x


def _unhooked(module: torch.nn.Module, cls: type) -> bool:
    """Whether calling ``module`` runs ``cls.forward`` and nothing else (hooks for every module aside)."""
    d = module.__dict__
    return type(module) is cls and not ("forward" in d or d["_forward_hooks"] or d["_forward_pre_hooks"] or
                                        d["_backward_hooks"] or d["_backward_pre_hooks"])


def _shown_to_modes() -> bool:
    """Whether a function mode sees the calls one by one.  That of ``torch.device`` and ``torch.set_default_device`` is shown
    nothing that it would change."""
    return any(type(torch._C._get_function_stack_at(i)) is not DeviceContext for i in range(torch._C._len_torch_function_stack()))


#: A projection joins the stack's call up to this many bins and classes (`FrameClassifier._scores`)
_JOIN_BINS, _JOIN_CLASSES = 6, 256


class FrameClassifier(torch.nn.Module):
    """Convolution stack, then a linear projection of every frame's features to log-probabilities.

    The output stage of the reference's acoustic model without its recurrent layers
    (models.py:437-454: the convolutional features of a frame, channels x bins flattened, go
    through ``torch.nn.Linear`` to ``target_dim`` scores): ``x (N, C_in, T, F) ->
    (N, T', n_out)`` log-probabilities.  In half precision the projection, a linear
    correlation over a frame's few bins, is the last layer of the stack's one call; else it is PyTorch's."""

    def __init__(self, stack: ConvStack, n_out: int = 62):
        super().__init__()
        self.stack = stack
        self.out = torch.nn.Linear(stack.out_channels * stack.out_size[1], n_out)

    def _scores(self, x: torch.Tensor) -> Optional[torch.Tensor]:
        """The scores ``(N, T', n_out)`` by one call, or None where the modules have to be called one by one.

        The projection of a frame's channels x bins is a correlation with a kernel of one frame and all bins, so the last
        convolution's output and its gradient need not leave the kernels' layout: as modules they are laid out as features and
        back around PyTorch's products.  In half precision, us a step of ten layers, 3 -> 256 channels on 32 x 780 x 41:
        Mellin layers (5 bins behind the last) 3690 -> 3435, linear ones (1 bin) 2854 -> 2700; eight other half stacks 0.90 to
        1.00 up to 6 bins.  Its input gradient multiplies all bins' taps, of which one meets a frame: at 10 bins 1.00 to 1.02, and
        in float32, where a product costs six times as much, nothing is left at 5 either.  The layouts that it spares do not grow
        with the classes, and PyTorch's product is the faster of the two: four stacks of two to four layers, 128 and 256 channels,
        3 to 6 bins, 1 to 64 utterances of 780 frames, training and not: joined over apart 0.52 to 1.01 with 256 classes, 0.51 to
        1.10 with 448, 0.55 to 1.32 with 1000, 0.68 to 2.06 with 4000."""
        # (what no call of this module can change comes first, and in front of the walk over the layers, which the stack makes
        # again: 5 us of the 105 that a call with 41 bins and seven layers takes the host)
        stack, out = self._modules.get("stack"), self._modules.get("out")
        if type(stack) is not ConvStack or stack.plan[-1]["out_size"][1] > _JOIN_BINS or len(stack.plan) < 2:
            return None
        if type(out) is not torch.nn.Linear or out.out_features > _JOIN_CLASSES:
            return None
        half = torch.get_autocast_dtype("cuda") == torch.float16 if torch.is_autocast_enabled("cuda") else x.dtype == torch.float16
        if not (half and x.is_cuda and x.dim() == 4):
            return None
        if not (_unhooked(stack, ConvStack) and _unhooked(out, torch.nn.Linear) and stack._fused() and stack._plain()) or _shown_to_modes():
            return None
        bins, channels = stack.out_size[1], stack.out_channels
        weight = out.weight
        if weight.dim() != 2 or weight.shape[1] != channels * bins or not weight.is_contiguous():
            return None
        kind = _hip.AX_MCORR if stack.params.mellin else _hip.AX_LCORR
        # (a Mellin axis of one tap, s = d = 1 and p = 0 is the identity on the frames)
        y = _native_stack(kind, x, [(conv.weight, conv.bias, conv.s, conv.d, conv.p, conv.r, bool(lay["pool"]))
                                    for conv, lay in zip(stack.convs, stack.plan)] +
                          [(weight.view(-1, channels, 1, bins), out.bias, (1, 1), (1, 1), (0, 0), (0, 0), None)])
        if y is None:
            return None
        return y.squeeze(3).transpose(1, 2).contiguous()

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        scores = self._scores(x)
        if scores is not None:
            return torch.nn.functional.log_softmax(scores, dim=-1)
        h = self.stack(x)                                   # (N, C, T', F')
        h = h.permute(0, 2, 1, 3).flatten(2)                # (N, T', C * F')
        return torch.nn.functional.log_softmax(self.out(h), dim=-1)
