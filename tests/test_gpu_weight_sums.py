"""The sums that make a weight gradient of its workgroups' partial ones (`block_finish.hip`), where a block of threads takes all
taps of its channels, some of them, or one; where the taps or the input channels do not fill the last block; where filter columns
without a tap are left to zeros: against float64."""
import ctypes

import pytest
import torch

import _mellin_hip as hip
import mconv
from test_gpu_kept_inputs import dims_of

CASES = [
    # channels in and out, kernel, input size, s, d, p, r, batch
    (16, 1, (1, 1), (40, 30), (1, 1), (1, 1), (0, 0), (0, 0), 2),      # one weight a channel, 32 parts
    (41, 128, (8, 1), (391, 1), (1, 1), (1, 1), (3, 0), (0, 0), 4),    # a last block of channels that is not full
    (32, 32, (4, 4), (60, 41), (1, 1), (1, 1), (1, 1), (1, 1), 8),     # one tap a block
    (64, 64, (5, 3), (50, 41), (1, 1), (1, 1), (2, 1), (2, 1), 9),     # a last block of taps that is not full
    (130, 130, (3, 3), (20, 21), (1, 1), (1, 1), (1, 1), (1, 1), 2),
    (256, 128, (3, 3), (20, 20), (1, 1), (2, 1), (2, 1), (2, 1), 2),   # all nine taps a block
    (512, 40, (8, 4), (20, 10), (1, 1), (1, 1), (3, 1), (3, 1), 2),    # 32 taps: a part
    (513, 33, (9, 4), (20, 10), (1, 1), (1, 1), (3, 1), (3, 1), 2),    # more taps than a block has threads for
    (40, 48, (3, 5), (30, 2), (1, 1), (1, 1), (1, 2), (1, 2), 3),      # columns 0 and 4 of five meet padding only
    (24, 40, (3, 4), (30, 1), (1, 1), (1, 1), (1, 1), (1, 1), 3),      # filter columns without a tap
]

# taps of a block of threads; whether there are filter columns without a tap
ROUTES = [({1}, False), ({4}, False), ({1}, False), ({2}, False), ({5, 9}, False), ({9}, False), ({32}, False), ({32}, False),
          ({1}, True), ({1}, True)]


def test_cases_have_the_blocks_that_they_are_there_for():
    for (ci, co, kernel, size, s, d, p, r, batch), (chunks, columns) in zip(CASES, ROUTES):
        seen = set()
        for cls in (mconv.MCorrLCorr, mconv.LCorrLCorr):
            kind, dims = dims_of((cls, ci, co, kernel, size, s, d, p, r, batch))
            for elem_bytes in (4, 2):
                words = (ctypes.c_int * 4)()
                assert hip.lib.mellin_layer_weight_sums(kind, elem_bytes, *dims, words)
                chunk, parts, blocks, zeros = words
                seen.add(chunk)
                assert parts == 32 // chunk and blocks == co * -(-ci // 32) * -(-kernel[0] * live(kernel, size, s, d, p, dims) // chunk)
                assert (zeros > 0) == columns
        assert seen == chunks


def live(kernel, size, s, d, p, dims):
    """Filter columns with a tap."""
    return sum(any(0 <= s[1] * oy + d[1] * fy - p[1] < size[1] for oy in range(dims[8])) for fy in range(kernel[1]))


@pytest.mark.gpu
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("mellin", [False, True])
@pytest.mark.parametrize("case", CASES, ids=range(len(CASES)))
def test_weight_gradients_of_all_block_shapes(case, mellin, half):
    ci, co, kernel, size, s, d, p, r, batch = case
    torch.manual_seed(9300 + CASES.index(case))
    cls = mconv.MCorrLCorr if mellin else mconv.LCorrLCorr
    layer = cls(ci, co, kernel, s=s, d=d, p=p, r=r).cuda()
    x = torch.randn(batch, ci, *size, device="cuda")
    if half:
        layer, x = layer.half(), x.half()
    out = layer(x)
    grad = torch.randn_like(out)
    gw, gb = torch.autograd.grad(out, [layer.weight, layer.bias], grad)
    # sum over images and output positions of grad_out times the tap's input value, in float64 on the CPU
    xd, gd = x.double().cpu(), grad.double().cpu()
    want = torch.zeros(co, ci, *kernel, dtype=torch.float64)
    for fx in range(kernel[0]):
        for fy in range(kernel[1]):
            taps = []
            for ox in range(out.shape[2]):
                product = (ox + s[0]) * (fx + d[0])
                gx = product // (p[0] + 1) - 1 if mellin and product % (p[0] + 1) == 0 else -1 if mellin else s[0] * ox + d[0] * fx - p[0]
                if 0 <= gx < size[0]:
                    taps.append((ox, gx))
            cols = [(oy, s[1] * oy + d[1] * fy - p[1]) for oy in range(out.shape[3])]
            cols = [(oy, gy) for oy, gy in cols if 0 <= gy < size[1]]
            if taps and cols:
                ox, gx = map(list, zip(*taps))
                oy, gy = map(list, zip(*cols))
                a, b = gd[:, :, ox][:, :, :, oy].transpose(0, 1).flatten(1), xd[:, :, gx][:, :, :, gy].transpose(0, 1).flatten(1)
                want[:, :, fx, fy] = a @ b.t()
    # partial sums in float32 (1e-6 of the result's norm for up to 1e5 terms); half results are rounded once, 2^-12 on average
    for got, ref in ((gw, want), (gb, gd.sum((0, 2, 3)))):
        rel = float((got.double().cpu() - ref).norm() / ref.norm())
        assert rel < (5e-4 if half else 2e-6), rel
        assert torch.equal(got.cpu() == 0, ref == 0) or half
