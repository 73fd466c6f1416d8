"""Where infinite and NaN source pixels show in the kernels whose products take pairs of neighbouring pixels: in the
outputs whose filter windows hold the pixel, and as NaN in at most one column on either side of them (the other pixel of
a pair, whose tap there is zero).  Everything else is what it is without the pixel."""

import pytest
import torch
from helpers import gpu_args, to_gpu

from spio_amd.compiler import compile_kernel_configs
from spio_amd.hip import get_device_attributes
from spio_amd.kernels import (
    Conv2dGw8BgradConfig,
    Conv2dGw8Config,
    Conv2dGw8Params,
    conv2d_gw8_bgrad_kernel_factory,
    conv2d_gw8_kernel_factory,
)

pytestmark = pytest.mark.gpu

# every width whose last product has columns of no window, and those without
FILTERS = [(3, 1), (3, 2), (3, 3), (4, 4), (2, 4), (5, 5), (5, 6), (7, 7)]
PIXELS = [(3, 6, float("inf")), (4, 7, float("-inf")), (0, 0, float("inf")), (9, 16, float("nan"))]  # (row, column, value)


def _reached(params, row, column, igrad, beyond):
    """Destination pixels whose window holds a source pixel, and `beyond` columns on either side of them."""
    if igrad:  # dx[h] takes dy[h + py - r]
        rows = range(row - params.padding_h, row - params.padding_h + params.r)
        first, last = column - params.padding_w, column - params.padding_w + params.s - 1
        height, width = params.h, params.w
    else:  # y[p] takes x[p + r - py]
        rows = range(row + params.padding_h - params.r + 1, row + params.padding_h + 1)
        first, last = column + params.padding_w - params.s + 1, column + params.padding_w
        height, width = params.p, params.q
    mask = torch.zeros(height, width, dtype=torch.bool)
    rows = [r for r in rows if 0 <= r < height]
    if rows:
        mask[rows[0]:rows[-1] + 1, max(first - beyond, 0):max(last + beyond + 1, 0)] = True
    return mask


@pytest.mark.parametrize("filter_size", FILTERS, ids=str)
@pytest.mark.parametrize("kind", ["forward", "data gradient", "fused backward"])
def test_infinities_stay_with_their_windows(kind, filter_size):
    r, s = filter_size
    params = Conv2dGw8Params(n=2, c=24, h=10, w=17, r=r, s=s, padding=(r // 2, s // 2))
    igrad = kind != "forward"
    x, w, _bias, dy = gpu_args(params)
    source = dy if igrad else x
    attr = get_device_attributes(0)
    if kind == "fused backward":
        factory, kw = conv2d_gw8_bgrad_kernel_factory, {}
        configs = [Conv2dGw8BgradConfig(groups=3, prefetch=2), Conv2dGw8BgradConfig(groups=2, block_h=4, block_n=2, prefetch=2)]
    else:
        factory, kw = conv2d_gw8_kernel_factory, {"igrad": True} if igrad else {}
        configs = [Conv2dGw8Config(groups=3, block_p=4, prefetch=2), Conv2dGw8Config(groups=2, block_p=3, block_n=2, prefetch=2)]
    configs = [c for c in configs if factory.is_legal(params, c, **kw)]
    if not configs:
        assert kind == "fused backward" and r == 7
        pytest.skip("two kernels")
    # where images lie side by side without a zero column between them, "next to" is the last column of the one before
    halo = {"forward": s // 2, "data gradient": s - 1 - s // 2, "fused backward": s - 1 - s // 2}[kind]
    shape = params.input_shape if igrad else params.output_shape
    for kernel in compile_kernel_configs(factory, params, configs=configs, device_attr=attr, **kw):
        kernel.load(0)

        def result(src):
            out = torch.full(shape, -42.0, device="cuda", dtype=torch.float16).contiguous(memory_format=torch.channels_last)
            if kind == "fused backward":
                dw = torch.zeros(params.weight_shape, device="cuda").contiguous(memory_format=torch.channels_last)
                kernel(out, dw, to_gpu(x), to_gpu(src), to_gpu(w))
            else:
                kernel(out, to_gpu(src), to_gpu(w), None)
            return out.cpu()

        for row, column, value in PIXELS:
            row, column = min(row, source.shape[2] - 1), min(column, source.shape[3] - 1)
            hit, without = source.clone(), source.clone()
            hit[1, 9, row, column] = value  # group 1
            without[1, 9, row, column] = 0
            got, plain = result(hit), result(without)
            assert torch.isfinite(plain).all()
            window = _reached(params, row, column, igrad, 0)
            near = _reached(params, row, column, igrad, 1)
            assert not torch.isfinite(got[1, 8:16][:, window]).any(), "outputs that take the pixel"
            expected = plain.clone()
            expected[1, 8:16][:, near] = 0
            kept = got.clone()
            kept[1, 8:16][:, near] = 0
            if halo == 0 and column == 0:
                expected[0, 8:16][:, near.any(dim=1), -1] = 0
                kept[0, 8:16][:, near.any(dim=1), -1] = 0
            assert torch.equal(kept, expected), f"{kernel.config}: ({row}, {column}) = {value} reaches further"
        kernel.unload()
