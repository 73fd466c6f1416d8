"""GPU parity of the kernels whose products take pairs of neighbouring pixels, where tiles and chunks of 32 pixels
end: rows of 31 to 33 and of 64 pixels, every filter width, step loops in chunks, row blocks that do not divide the
image.  Oracle and tolerances are those of the other kernel tests."""

import pytest
from helpers import run_bgrad_kernel_test, run_grad_kernel_test, run_kernel_test

from spio_amd.kernels import (
    Conv2dGw8BgradConfig,
    Conv2dGw8Config,
    Conv2dGw8Params,
    Conv2dGw8WgradConfig,
    conv2d_gw8_bgrad_kernel_factory,
    conv2d_gw8_kernel_factory,
    conv2d_gw8_wgrad_kernel_factory,
)

pytestmark = pytest.mark.gpu

SHAPES = [
    # (n, c, h, w, r, s, padding, bias)
    (3, 24, 9, 31, 3, 3, 1, True),
    (3, 16, 7, 32, 3, 3, 1, True),  # a chunk, which begins a pixel early, more than a tile
    (2, 16, 6, 33, 5, 5, 2, False),
    (2, 24, 5, 64, 3, 3, 1, True),
    (5, 16, 11, 9, 5, 5, 2, True),  # three images and their shared halo fill a tile
    (4, 40, 6, 14, 5, 4, (2, 1), False),
    (3, 8, 5, 13, 1, 1, 0, True),
    (3, 16, 8, 15, 2, 2, 1, True),
    (2, 16, 9, 10, 3, 1, (0, 0), False),
    (2, 16, 70, 6, 3, 3, 1, True),  # step loops in chunks
    (2, 16, 67, 6, 5, 3, (2, 1), True),
]


def _params(shape):
    n, c, h, w, r, s, padding, bias = shape
    return Conv2dGw8Params(n=n, c=c, h=h, w=w, r=r, s=s, padding=padding, has_bias=bias)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_fused_backward(shape):
    params = _params(shape)
    groups, h, images = min(params.groups, 4), params.h, min(params.n, 3)
    B = Conv2dGw8BgradConfig
    configs = [
        B(groups=groups, block_n=1, block_n_iters=params.n, prefetch=2),
        B(groups=groups, block_n=images if params.w < 32 else 1, block_h=4, prefetch=4),
        B(groups=groups, block_h=h if h < 40 else 13, block_n=2 if params.r < 5 else 1, prefetch=2, two_stage=1),
    ]
    if params.w > 32:
        configs.append(B(groups=groups, block_h=5, prefetch=2, split=2))
    run_bgrad_kernel_test(conv2d_gw8_bgrad_kernel_factory, params, configs=configs)


@pytest.mark.parametrize("shape", [*SHAPES, (2, 16, 8, 15, 7, 7, 3, True), (2, 8, 6, 7, 3, 3, 4, True)], ids=str)
def test_weight_gradient(shape):
    """Also a filter of 14 accumulators, and padding that leaves grad_output rows which meet no input row."""
    params = _params(shape)
    groups, images = min(params.groups, 4), min(params.n, 3)
    W = Conv2dGw8WgradConfig
    configs = [
        W(groups=groups, block_h=params.p, block_n=images, prefetch=2),
        W(groups=groups, block_h=params.p, block_n=1, block_n_iters=params.n, prefetch=2, rows=2, pipe=1, two_stage=1),
        W(groups=groups, block_h=4, block_n=2, prefetch=4, pipe=1),
        W(groups=groups, block_h=3, block_n=1, prefetch=2, rows=2, two_stage=1),
    ]
    if params.w > 32:
        configs.append(W(groups=groups, block_h=params.p, block_n=1, prefetch=2, split=2))
    run_grad_kernel_test(conv2d_gw8_wgrad_kernel_factory, params, configs=configs)


FORWARD_SHAPES = [*SHAPES, (2, 16, 8, 15, 7, 7, 3, True), (2, 8, 6, 7, 3, 3, 4, True), (2, 104, 6, 33, 3, 3, 1, True)]


@pytest.mark.parametrize("shape", FORWARD_SHAPES, ids=str)
@pytest.mark.parametrize("igrad", [False, True])
def test_forward_and_data_gradient(shape, igrad):
    """Also a filter of seven accumulators, and padding that makes rows without any input (they are the bias alone)."""
    params = _params(shape)
    groups, images, rows = min(params.groups, 4), min(params.n, 3), params.h if igrad else params.p
    C = Conv2dGw8Config
    configs = [
        C(groups=groups, block_p=min(rows, 40), block_n=images if params.w < 32 else 1, prefetch=2),
        C(groups=groups, block_p=min(rows, 4), block_n=1, prefetch=4),
        C(groups=1, block_p=min(rows, 3), block_n=1, prefetch=2, split=2),
        C(groups=groups, block_p=min(rows, 3), block_p2=1, block_n=1, prefetch=2),
    ]
    if params.w >= 31:
        configs.append(C(groups=groups, block_p=min(rows, 5), block_q=17, prefetch=2))
    if params.groups > 8:  # two blocks, the second with a group less
        configs.append(C(groups=7, block_p=min(rows, 4), prefetch=2))
    if igrad:
        run_grad_kernel_test(conv2d_gw8_kernel_factory, params, configs=configs, igrad=True)
    else:
        run_kernel_test(conv2d_gw8_kernel_factory, params, configs=configs)


@pytest.mark.parametrize("shape", [(2, 24, 7, 140, 3, 3, 1, True), (1, 16, 9, 95, 5, 5, 2, False), (2, 8, 6, 63, 2, 4, 1, True)], ids=str)
def test_fused_backward_in_column_blocks_of_whole_chunks(shape):
    """Column blocks one short of 32-pixel tiles, whose chunks begin a pixel before the block; the last block is
    narrower, or a whole one."""
    params = _params(shape)
    B = Conv2dGw8BgradConfig
    configs = [
        B(groups=2 if params.groups > 1 else 1, block_h=3, block_q=32, narrow=1, prefetch=2),
        B(groups=1, block_q=64, narrow=1, prefetch=4, split=2, two_stage=1),
        B(groups=params.groups, block_h=4, block_q=64, narrow=1, block_n_iters=params.n, prefetch=2),
    ]
    run_bgrad_kernel_test(conv2d_gw8_bgrad_kernel_factory, params, configs=configs)
