"""Fused backward kernel family of conv2d_gw8: grad_input and grad_weight in one pass.

The reference launches its data-gradient and weight-gradient kernels one after
the other (spio/functional/conv2d_gw8_function.py:119-146); both stream
grad_output.  This family reads grad_output once and produces both gradients
(and grad_bias when the params have a bias), which removes a quarter of the
backward step's HBM traffic.  The kernel computes a size-preserving convolution;
every other padding is one on a larger domain in which the input and the output
sit at fitting offsets (`bgrad_domain`).

Kernel arguments: (grad_input, grad_weight, x, grad_output, weight[, grad_bias]);
grad_weight (and grad_bias) are accumulated into, so the caller zeroes them first, unless the
configuration is two-stage (`KernelSpec.overwrites_output`): then both are stored whole.
"""

from dataclasses import dataclass, replace
from typing import Dict, List, Tuple

import torch

from ..util.math import balanced, divup
from .conv2d_gw8_kernel import (
    _policies_are_legal,
    _shape_defines,
    fits_float32_output,
    lane_registers,
    stage_pitch,
    with_joined_stores,
)
from .conv2d_gw8_params import Conv2dGw8Params
from .conv2d_gw8_wgrad_kernel import image_block_runs
from .conv2d_stats import Conv2dStats
from .kernel import KernelSpec
from .kernel_factory import KernelFactory
from .launch_params import LaunchParams

SOURCE = "conv2d_gw8_bgrad_mfma.hip"

MAX_WAVES = 16
MAX_LDS_BYTES = 128 * 1024
MAX_LOADS_PER_THREAD = 4
MAX_REGISTERS = 256  # estimated fragments + accumulators + prefetch buffers, in 32-bit registers
# Accumulators of the weight gradient.  The 14 of a 7x7 filter fit, but one pass is mostly slower there than two kernels, which
# the arithmetic bounds.  Fused against data and weight gradient and the 2.2 us of a launch, best of 16 each: 256n 256c 14x14
# 55.4 and 39.8 us, 64n 96c 56x56 59.4 and 52.4, 128n 192c 28x28 54.7 and 55.2, 32n 128c 56x56 36.0 and 40.9; 16n 64c 112x112
# has none of whole rows.
MAX_SUMS = 14
GEOMETRIES_PER_HEIGHT = 6
MAX_UNROLLED_STEPS = 40  # SPIO_MAX_UNROLL of the kernel: longer step loops run in chunks


@dataclass(frozen=True)
class Conv2dGw8BgradConfig:
    """Tile configuration of the fused backward kernel.

    Attributes:
        groups: channel groups per workgroup (one wave each, times `split`).
        block_h: rows of grad_input (and of grad_output for the weight gradient) per
            workgroup; 0 = the whole image.  Smaller blocks give more workgroups at the price
            of re-reading the padding rows of grad_output and x at the block borders.
        block_n: images whose rows are laid side by side in one staged row.
        block_n_iters: image blocks a workgroup processes before it publishes grad_weight.
        prefetch: rows of global loads in flight ahead of the computed row (even).
        split: waves per group; they share the 32-pixel chunks (weight gradient) and the
            32-pixel tiles (data gradient) of a row.
        halo_cached: 1 = rows shared with the neighbouring row blocks are loaded with the default
            cache policy (the second reader can hit in L2), the others with the non-temporal hint.
        xcd_chunk: consecutive tiles that go to the same XCD before the next run goes to the next
            one; 0 = one contiguous range of tiles per XCD.
        two_stage: 1 = workgroups store their grad_weight (and grad_bias) sums into blocks of a
            workspace and a second kernel stores the blocks' sum into grad_weight and grad_bias,
            which then need no zero fill; 0 = workgroups add into zeroed tensors with fp32
            atomics.  Atomic additions of different workgroups to one line retire one after the
            other, and in a one-round grid all workgroups publish at the same time.
        block_q: columns per workgroup (0: the whole width; else a multiple of 32 with
            block_n = 1).  The workgroup stages block_q + S - 1 columns of x and of grad_output, so
            rows of any width fit.
        nontemporal: 1 = store grad_input with the non-temporal hint.
        narrow: 1 = a workgroup has one column less than block_q.  The weight gradient's 32-pixel
            chunks begin a pixel before the block, so block_q columns take one more of them than
            block_q / 32 and block_q - 1 do not.
    """

    groups: int = 4
    block_h: int = 0
    block_n: int = 1
    block_n_iters: int = 1
    prefetch: int = 4
    split: int = 1
    halo_cached: int = 1
    xcd_chunk: int = 4
    block_q: int = 0
    two_stage: int = 0
    nontemporal: int = 1
    narrow: int = 0


def bgrad_is_supported(params: Conv2dGw8Params) -> bool:
    """The fused kernel takes every shape the operator takes.

    It computes a size-preserving convolution on the domain `bgrad_domain` returns, in which the
    input and the output sit at offsets that reproduce the problem's padding.  Whether a shape
    has a legal configuration is a separate question (large filters run out of registers).
    """
    return params.r >= 1 and params.s >= 1


def bgrad_domain(params: Conv2dGw8Params) -> Tuple[int, int]:
    """Rows and columns of the images the fused kernel works on.

    The domain's own padding is r // 2 rows above (s // 2 columns left) and the rest of r - 1
    (s - 1) below (right); the input starts max(padding - r // 2, 0) rows into the domain, the
    output max(r // 2 - padding, 0), and the domain ends where the later of the two ends.
    """

    def extent(size, out_size, filt, padding):
        shift = filt // 2 - padding
        return max(max(-shift, 0) + size, max(shift, 0) + out_size)

    return (extent(params.h, params.p, params.r, params.padding_h),
            extent(params.w, params.q, params.s, params.padding_w))  # fmt: skip


def bgrad_geometry(params: Conv2dGw8Params, config: Conv2dGw8BgradConfig) -> Dict[str, int]:
    """Host mirror of the compile-time constants of conv2d_gw8_bgrad_mfma.hip."""
    r, s = params.r, params.s
    gb, nb, iters, ts, pf = config.groups, config.block_n, config.block_n_iters, config.split, config.prefetch
    dh, dw = bgrad_domain(params)
    pb, pr = r - 1 - r // 2, s - 1 - s // 2  # the domain's padding below and right
    bh = config.block_h or dh
    nb4 = divup(s, 4)
    bq = config.block_q - config.narrow if config.block_q else dw
    wpi = bq + s - 1
    f = nb * wpi
    kspan = (nb - 1) * wpi + bq
    kc = divup(kspan + 1, 32)
    cpw = divup(kc, ts)
    kb = divup(s + 1, 4)
    wt = divup(f - s + 1, 32)
    tpw = divup(wt, ts)

    def group_cells(pixels):
        plane = divup(pixels, 2)
        plane += (8 - plane) % 16
        return plane + pixels // 2 + ((9 if gb > 4 else 2 if gb > 2 else 4) - plane - pixels // 2) % 16

    dl = max(pr, 1)
    gsx = group_cells(32 * cpw * ts + 4 * nb4 - 2)
    gsd = group_cells(max(dl + 32 * cpw * ts, dl - pr + 32 * tpw * ts + 4 * kb - 2))
    threads = 64 * gb * ts
    # every ring row carries a spare unit behind its last group (see the kernel)
    ring_units = 2 * (gb * gsx + 1) + 2 * (gb * gsd + 1)
    out_row_bytes = 2 * (16 * tpw * ts * stage_pitch(gb) + 128)
    stream_bytes = ring_units * 16 + 2 * out_row_bytes
    filter_bytes = gb * 8 * r * s * 16
    publish_bytes = (gb * ts * r * s * 64 + (gb * ts * 8 if params.has_bias else 0)) * 4
    lptx = divup(f * gb, threads)
    lptd = divup((f if config.block_q else nb * dw) * gb, threads)  # grad_output loads per row
    registers = (
        4 * (r * nb4 + 1)  # weight-gradient accumulators (+ bias)
        + 4 * tpw * r  # data-gradient accumulators
        + 4 * r * kb  # filter fragments
        + 4 * r * cpw  # fragments of the last grad_output rows
        + 4 * (cpw * nb4 + tpw * kb)  # other operand fragments of one step
        + 4 * pf * (lptx + lptd)  # prefetch buffers
    )
    g = dict(
        NB4=nb4, KB=kb, KC=kc, CPW=cpw, WT=wt, TPW=tpw, THREADS=threads,
        LDS_BYTES=max(stream_bytes, filter_bytes, publish_bytes),
        LPTX=lptx, LPTD=lptd, REGISTERS=registers,
        STEPS=bh + pb + r - 1,
        BH=bh, GBLKS=divup(params.groups, gb), PBLKS=divup(dh, bh), NBLKS=divup(params.n, nb * iters),
        BQ=bq, QBLKS=divup(dw, bq),
        PIXEL_EFF=(nb * bq) / (32.0 * kc),
    )  # fmt: skip
    g["NUM_BLOCKS"] = g["GBLKS"] * g["PBLKS"] * g["QBLKS"] * g["NBLKS"]
    return g


def _config_is_legal(params, config) -> bool:
    if not bgrad_is_supported(params):
        return False
    g = bgrad_geometry(params, config)
    return (
        config.groups * config.split <= MAX_WAVES
        and config.split <= min(g["KC"], g["WT"])
        and 0 <= config.block_h <= bgrad_domain(params)[0]
        and 0 <= config.block_q <= bgrad_domain(params)[1] + config.narrow
        and (config.block_q == 0 or (config.block_q % 32 == 0 and config.block_n == 1))
        and 0 <= config.narrow <= min(config.block_q, 1)
        and g["LPTD"] <= MAX_LOADS_PER_THREAD
        and config.block_n <= max(params.n, 1) and config.block_n * (config.block_n_iters - 1) < max(params.n, 1)
        and g["LDS_BYTES"] <= MAX_LDS_BYTES
        and g["LPTX"] <= MAX_LOADS_PER_THREAD
        and g["REGISTERS"] <= MAX_REGISTERS
        and params.r * g["NB4"] < MAX_SUMS
        and config.prefetch >= 2
        and config.prefetch % 2 == 0
        and config.block_n * params.c * max(params.h * params.w, params.p * params.q) * 2 < 2**31
    )


def _fits(params, config) -> bool:
    """Whether a lane's registers hold the sums, the filters, the rows in flight and a step's operands, or most of them.
    The weights were fitted to what the compiler reports for 402 kernels of 67 shapes.  The line lies a tenth above the
    registers there are: up to there the compiler keeps 20 to 130 bytes a lane in memory, if any, which costs little;
    beyond it hundreds (16 waves mostly), which costs a multiple."""
    g = bgrad_geometry(params, config)
    kept = params.r * (g["NB4"] + g["TPW"] + g["KB"] + g["CPW"]) + 1
    operands = g["CPW"] * g["NB4"] + g["TPW"] * g["KB"]
    loads = g["LPTX"] + g["LPTD"]
    needed = 3.6 * kept + 13.9 * operands + 5.2 * config.prefetch * loads + 21
    return needed <= 1.1 * lane_registers(config.groups * config.split)


def _recorded_config_is_legal(params, config) -> bool:
    return (
        min(config.groups, config.block_n, config.block_n_iters, config.split) >= 1
        and config.two_stage in (0, 1)
        and _policies_are_legal(config)
        and _config_is_legal(params, config)
    )


def _score(params, config, num_cus) -> float:
    """Rough relative cost used only to order (and cap) the sweep; lower is better."""
    g = bgrad_geometry(params, config)
    group_eff = params.groups / (g["GBLKS"] * config.groups)
    quant = divup(g["NUM_BLOCKS"], num_cus) * num_cus / g["NUM_BLOCKS"]
    quant *= g["PBLKS"] * g["BH"] / bgrad_domain(params)[0]  # the last, shorter tiles
    quant *= g["QBLKS"] * g["BQ"] / bgrad_domain(params)[1]
    quant *= g["NBLKS"] * config.block_n * config.block_n_iters / params.n
    halo = 1.0 + (2.0 / 3.0) * (params.r - 1 if g["PBLKS"] > 1 else 0) / g["BH"]
    dh, dw = bgrad_domain(params)
    stream_us = halo * 6.0 * params.n * params.c * dh * dw / 5.0e6
    publish_us = g["NUM_BLOCKS"] * config.groups * params.r * params.s * 64.0 / (128 * 2.1e3)
    split_line = 1.0 if (config.groups * 16) % 128 == 0 or config.groups == params.groups else 1.12
    return (quant * split_line / (g["PIXEL_EFF"] ** 0.3 * group_eff)) * (1.0 + publish_us / stream_us)


def _get_configs(params: Conv2dGw8Params, device_attr=None) -> List[Conv2dGw8BgradConfig]:
    """Legal configurations, most promising first; empty when the shape is not supported."""
    num_cus = getattr(device_attr, "multiprocessor_count", 256) or 256
    G = params.groups
    # powers of two, the whole pixel, and half a pixel where the group count is not a power of two
    # (96 channels: 12 groups = 2 x 6)
    group_choices = sorted({g for g in (4, 8, 16, G, G // 2 if G % 2 == 0 and G & (G - 1) else G)
                            if 0 < g <= min(G, MAX_WAVES)}) or [min(G, MAX_WAVES)]
    # Rank the geometries of every row-block height separately and keep the best few of each:
    # whether whole images or row blocks win depends on the shape in ways the score does not
    # capture (contiguity of the channel block, halo re-reads, workgroups per compute unit).
    dh, dw = bgrad_domain(params)
    row_choices = [0] + balanced(dh, [bh for bh in (7, 14, 28) if bh < dh])[::-1]
    # images side by side: powers of two, and for rows shorter than a 32-pixel chunk of the weight
    # gradient's contraction the counts that fill the chunks clearly better (as in the
    # weight-gradient kernel's configuration space)
    wpi = dw + params.s - 1

    def chunk_fill(nb):
        return nb * dw / (32.0 * divup((nb - 1) * wpi + dw + 1, 32))

    image_counts = [1, 2, 4, 8]
    if wpi < 32:
        best = max(chunk_fill(nb) for nb in image_counts)
        image_counts += [nb for nb in (3, 5, 6, 7) if chunk_fill(nb) > best + 0.05]
    # Column blocks for wide rows only: narrower ones fit whole.  A chunk of the weight gradient begins a pixel before the
    # block, so 64 columns take three and 63 two.  Which is better depends on the shape, best of 24 configurations with 64 and
    # 63: 4n 96c 100x300 5x5 43.8 and 31.6 us, 32n 64c 224x224 116.6 and 115.3, 8n 64c 64x1024 42.1 and 41.5, but 16n 64c
    # 128x512 76.9 and 78.8, 8n 24c 144x256 20.1 and 21.0 (127 columns are no better than 128 anywhere).
    col_choices = [(0, 0)] + [(bq, less) for bq, less in ((64, 1), (64, 0), (128, 0)) if dw >= 2 * (bq - less) and dw > 128]
    configs, of_each = [], []
    for bh in row_choices:
        geometries = []
        for bq, less in col_choices:
            for gb in group_choices:
                for nb in image_counts if bq == 0 else (1,):
                    tiles = divup(G, gb) * divup(dh, bh or dh) * divup(dw, bq or dw)
                    for iters in image_block_runs(divup(params.n, nb), tiles, num_cus, (1, 2, 4)):
                        for ts in (1, 2):
                            cfg = Conv2dGw8BgradConfig(groups=gb, block_h=bh, block_n=nb, block_n_iters=iters,
                                                       prefetch=4, split=ts, block_q=bq, narrow=less)  # fmt: skip
                            if _config_is_legal(params, cfg):
                                geometries.append((_score(params, cfg, num_cus), cfg))
        geometries.sort(key=lambda sc: sc[0])
        ranked = [cfg for _, cfg in geometries]
        # the best, and as many of those that fit the registers
        fitting = [cfg for cfg in ranked if _fits(params, cfg)][:GEOMETRIES_PER_HEIGHT]
        configs += ranked[:GEOMETRIES_PER_HEIGHT] + [cfg for cfg in fitting if cfg not in ranked[:GEOMETRIES_PER_HEIGHT]]
        of_each += [cfg for gb in group_choices for cfg in [c for c in ranked if c.groups == gb and _fits(params, c)][:2]]
    # ... and, where a sweep has time for them, two of every number of groups: the score has many ties, which one number
    # can fill (128n 384c 14x14 from memory: 8 groups in blocks of four images 15.0 us, the best of the others 17.0)
    configs += [cfg for cfg in of_each if cfg not in configs]
    # what keeps much of its registers in memory comes last
    configs.sort(key=lambda cfg: not _fits(params, cfg))
    # a shallower and a deeper pipeline for the first few: the shallow one wins where rows are short
    first = configs[:GEOMETRIES_PER_HEIGHT]
    configs += [replace(cfg, prefetch=2) for cfg in first]
    configs += [replace(cfg, prefetch=8) for cfg in first[:3] if _config_is_legal(params, replace(cfg, prefetch=8))]
    # ... and the other memory-system policies
    configs += [replace(cfg, halo_cached=hc, xcd_chunk=ch) for cfg in first[:2] for hc, ch in ((0, 4), (1, 0))]
    # ... and two-stage publishing for the leaders of every height
    configs += [replace(cfg, two_stage=1) for cfg in list(configs) if cfg.prefetch == 4 and cfg.halo_cached == 1
                and cfg.xcd_chunk == 4][:2 * GEOMETRIES_PER_HEIGHT]  # fmt: skip
    return with_joined_stores(params, configs)


def _float32_prefetch(prefetch: int) -> int:
    """Rows in flight where grad_output is float32: half as many.  (All of them: 128n 384c 14x14 29.7 us, half
    28.7.)"""
    return max(2, prefetch // 4 * 2)


def bgrad_reads_float32(params: Conv2dGw8Params, config: Conv2dGw8BgradConfig) -> bool:
    """Whether a configuration has a version that reads a float32 grad_output: its rows in flight take twice
    the registers."""
    config = replace(config, prefetch=_float32_prefetch(config.prefetch))
    g = bgrad_geometry(params, config)
    return g["REGISTERS"] + 4 * config.prefetch * g["LPTD"] <= MAX_REGISTERS and fits_float32_output(params, config)


def _get_kernel_name(out_f32: bool = False, src_f32: bool = False) -> str:
    return "spio_conv2d_gw8_bgrad" + ("_f32" if out_f32 else "") + ("_srcf32" if src_f32 else "")


def _get_kernel_spec(params: Conv2dGw8Params, config: Conv2dGw8BgradConfig, _device_attr=None,
                     out_f32: bool = False, src_f32: bool = False) -> KernelSpec:  # fmt: skip
    """Macros and launch geometry; `out_f32`: grad_input is a float32 tensor, `src_f32`: grad_output is."""
    params.validate()
    assert _config_is_legal(params, config), f"illegal configuration {config} for {params}"
    g = bgrad_geometry(params, config)
    defines = _shape_defines(params)
    if out_f32:
        assert fits_float32_output(params, config), f"no float32 output for {config} and {params}"
        defines["SPIO_DST_F32"] = 1
    if src_f32:
        assert bgrad_reads_float32(params, config), f"no float32 grad_output for {config} and {params}"
        defines["SPIO_SRC_F32"] = 1
    defines.update(SPIO_GB=config.groups, SPIO_BH=g["BH"], SPIO_NB=config.block_n,
                   SPIO_ITERS=config.block_n_iters,
                   SPIO_PF=_float32_prefetch(config.prefetch) if src_f32 else config.prefetch, SPIO_TS=config.split,
                   SPIO_HALO_CACHED=config.halo_cached, SPIO_XCD_CHUNK=config.xcd_chunk,
                   SPIO_NT=config.nontemporal, SPIO_HAS_BIAS=int(params.has_bias))  # fmt: skip
    if config.block_q:
        defines["SPIO_BQ"] = config.block_q - config.narrow
    spec = KernelSpec(defines, LaunchParams(grid=g["NUM_BLOCKS"], block=g["THREADS"]), SOURCE, notes=g)
    if config.two_stage:
        # one block per workgroup: its groups' grad_weight values, then its 8 bias sums per group
        part_floats = config.groups * params.r * params.s * 64 + (config.groups * 8 if params.has_bias else 0)
        npart = g["NBLKS"] * g["PBLKS"] * g["QBLKS"]
        defines.update(SPIO_PARTIALS=1)
        spec.workspace_bytes = g["GBLKS"] * npart * part_floats * 4
        spec.workspace_arg = 1  # the workspace takes the place of grad_weight
        spec.epilogue_suffix = "_reduce"
        spec.epilogue_half_suffix = "_reduce_h"
        spec.epilogue_extra_args = (5,)  # grad_bias, or None where there is none
        spec.epilogue_launch_params = LaunchParams(grid=g["GBLKS"] * divup(part_floats // 4, 8), block=256)
        spec.epilogue_half_launch_params = spec.epilogue_launch_params
        spec.overwrites_output = True
    return spec


def _make_test_args(params: Conv2dGw8Params, device):
    """Synthetic (grad_input, grad_weight, x, dy, weight[, grad_bias]) for timing."""
    cl = torch.channels_last
    x = torch.randn(params.input_shape, device=device, dtype=torch.float16).contiguous(memory_format=cl)
    dy = torch.randn(params.output_shape, device=device, dtype=torch.float16).contiguous(memory_format=cl)
    w = torch.randn(params.weight_shape, device=device, dtype=torch.float16).contiguous(memory_format=cl)
    dx = torch.empty_like(x)
    dw = torch.zeros(params.weight_shape, device=device, dtype=torch.float32).contiguous(memory_format=cl)
    if params.has_bias:
        return (dx, dw, x, dy, w, torch.zeros(params.c, device=device, dtype=torch.float32))
    return (dx, dw, x, dy, w)


conv2d_gw8_bgrad_kernel_factory = KernelFactory(
    Conv2dGw8Params,
    Conv2dGw8BgradConfig,
    Conv2dStats,
    kernel_name=_get_kernel_name,
    configs=_get_configs,
    kernel_spec=_get_kernel_spec,
    make_test_args=_make_test_args,
    is_legal=_recorded_config_is_legal,
)
