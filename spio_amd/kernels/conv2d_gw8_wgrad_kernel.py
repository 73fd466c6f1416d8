"""Weight-gradient kernel family of conv2d_gw8.

Kernel arguments: (grad_weight, x, grad_output) and, when the params have a
bias, a fourth `grad_bias` ([K] fp32, pre-zeroed like grad_weight, or None):
the kernels then also sum grad_output per channel in the same pass, which the
reference leaves to a separate reduction (spio/functional/conv2d_gw8_function.py:134-136).

Reference: spio/kernels/conv2d_gw8_wgrad_kernel.py:27-285.  The kernel adds
its partial sums into a pre-zeroed fp32 tensor laid out [K][R][S][8]
(spio/functional/conv2d_gw8_function.py:124-130).
"""

from dataclasses import dataclass, replace
from typing import Dict, List

import torch

from ..util.math import balanced, divup
from .conv2d_gw8_kernel import _shape_defines, lane_registers
from .conv2d_gw8_params import Conv2dGw8Params
from .conv2d_stats import Conv2dStats
from .kernel import KernelSpec
from .kernel_factory import KernelFactory
from .launch_params import LaunchParams

DIRECT_SOURCE = "conv2d_gw8_direct.hip"
MFMA_SOURCE = "conv2d_gw8_wgrad_mfma.hip"

MAX_WAVES = 16
MAX_LDS_BYTES = 128 * 1024
MAX_LOADS_PER_THREAD = 8
MAX_ACCUMULATORS = 32
MAX_UNROLLED_STEPS = 64  # SPIO_MAX_UNROLL of the kernel: longer step loops run in chunks
MAX_GEOMETRIES = 20  # that enter the sweep, with the pipelines about 100 candidates (20 s)
PIPELINE_CHOICES = ((2, 1, 0), (4, 1, 0), (2, 2, 0), (2, 1, 1), (4, 1, 1))  # (prefetch, rows, pipe)
LEADING_PIPELINES = 3  # of these, for the leading geometries at the head of the list


@dataclass(frozen=True)
class Conv2dGw8WgradConfig:
    """Tile configuration of the weight-gradient kernel.

    Attributes:
        groups: channel groups (waves) per workgroup.
        block_h: rows of grad_output per workgroup.
        block_n: images whose rows are laid side by side in one staged row.
        block_n_iters: image blocks a workgroup accumulates before its atomics.
        chunks: (direct variant only) pixel chunks per group.
        prefetch: steps of global loads in flight ahead of the computed step (even).
        rows: rows of x (and of grad_output) a workgroup multiplies between two barriers,
            1 or 2; two rows halve the barriers at the price of a deeper LDS ring (grad_output
            fragments stay in registers across rows with either).
        split: waves sharing the 32-pixel chunks of one group; their sums are added in LDS
            before publishing, so bigger workgroups do not publish more.
        two_stage: 1 = workgroups store partial sums to a workspace and a second kernel
            stores their sum into grad_weight (no zero fill needed, deterministic); 0 =
            workgroups add into a zeroed grad_weight with fp32 atomics.
        variant: "mfma" (row-streaming MFMA kernel) or "direct" (any shape).
        block_q: grad_output columns per workgroup (0: the whole width); the workgroup stages
            block_q + S - 1 columns of x opposite them, so rows of any width fit.
        pipe: 1 = the MFMAs of a step are issued one step later, from a second set of fragment
            registers, with the next step's LDS reads, row loads and ring writes dealt out
            between them; 0 = every step reads its fragments, then multiplies.
    """

    groups: int = 8
    block_h: int = 14
    block_n: int = 1
    block_n_iters: int = 1
    chunks: int = 0
    variant: str = "mfma"
    prefetch: int = 2
    two_stage: int = 0
    split: int = 1
    rows: int = 1
    block_q: int = 0
    pipe: int = 0


def image_placement(params: Conv2dGw8Params, nb: int, block_q: int = 0) -> Dict[str, int]:
    """Where the images of a staged row sit (mirror of the kernel's constants).

    Images follow one another GAP = max(px, S-1-px) zero cells apart (the right halo of one is
    the left halo of the next).  The contraction runs over 32-pixel chunks of the grad_output
    row; where a chunk holds whole images and that takes fewer chunks than the images laid end
    to end, every chunk gets its own images (PACKED).  A chunk begins one pixel before its first
    image, so 31 of its pixels are the images'.
    """
    s, px = params.s, params.padding_w
    nb4 = divup(s, 4)
    bq = block_q or params.q
    gap = max(px, s - 1 - px)
    ip = bq + s - 1 if block_q else bq + gap
    ipc_max = (31 + ip - bq) // ip
    kc_flat = divup((nb - 1) * ip + bq + 1, 32)
    kc_packed = divup(nb, ipc_max) if ipc_max > 0 else kc_flat
    packed = kc_packed < kc_flat
    kc = kc_packed if packed else kc_flat
    xcp = 16 * divup(32 + 4 * nb4 - 2, 16) if packed else 32
    return dict(IP=ip, IPC=ipc_max if packed else nb, KC=kc, PACKED=int(packed), XCP=xcp,
                FPX=kc * xcp if packed else 32 * kc + 4 * nb4 - 2)  # fmt: skip


def wgrad_geometry(params: Conv2dGw8Params, config: Conv2dGw8WgradConfig) -> Dict[str, int]:
    """Host mirror of the compile-time constants of conv2d_gw8_wgrad_mfma.hip."""
    r, s = params.r, params.s
    gb, bh, nb, iters, ts = config.groups, config.block_h, config.block_n, config.block_n_iters, config.split
    nb4 = divup(s, 4)
    bq = config.block_q or params.q
    wpi = bq + s - 1
    f = nb * wpi
    place = image_placement(params, nb, config.block_q)
    kc = place["KC"]
    chunks = divup(kc, ts) * ts  # past the last one: zeros
    fpx = place["FPX"] + (chunks - kc) * place["XCP"]
    gsx = fpx + ((9 - fpx % 16) + 16) % 16
    fpd = 32 * chunks + 1
    gsd = fpd + ((9 - fpd % 16) + 16) % 16
    rb = config.rows
    pblks = divup(params.p, bh)
    rows = bh + r - 1
    skip = pblks == 1 and params.padding_h < r and divup(rows, rb) <= MAX_UNROLLED_STEPS  # kSkipPadding of the kernel
    lead = params.padding_h // rb * rb if skip else 0
    threads = 64 * gb * ts
    # rows carry 16 spare units behind the last group
    lds_rings = (2 * rb * (gb * gsx + 16) + (lead + 2 * rb) * (gb * gsd + 16)) * 16
    # the same LDS block holds every group's R*S*64 sums at the end
    lds_scratch = (gb * r * s * 64 + (gb * ts * 8 if params.has_bias else 0)) * 4
    g = dict(
        NB4=nb4, WPI=wpi, F=f, KC=kc, CPW=chunks // ts, GSX=gsx, GSD=gsd, THREADS=threads,
        LDS_BYTES=max(lds_rings, lds_scratch), RING_BYTES=lds_rings, SCRATCH_BYTES=lds_scratch,
        LPTX=divup(f * gb, threads), LPTD=divup(nb * bq * gb, threads),
        BQ=bq, QBLKS=divup(params.q, bq),
        GBLKS=divup(params.groups, gb), PBLKS=pblks,
        NBLKS=divup(params.n, nb * iters),
        STEPS=divup(rows, rb),
        PIXEL_EFF=(nb * bq) / (32.0 * kc), IPC=place["IPC"], PACKED=place["PACKED"],
    )  # fmt: skip
    g["NUM_BLOCKS"] = g["GBLKS"] * g["PBLKS"] * g["QBLKS"] * g["NBLKS"]
    return g


def _mfma_config_is_legal(params, config) -> bool:
    g = wgrad_geometry(params, config)
    return (
        config.groups * config.split <= MAX_WAVES
        and config.split <= g["KC"]
        and config.block_h <= params.p
        and config.block_n <= max(params.n, 1) and config.block_n * (config.block_n_iters - 1) < max(params.n, 1)
        and g["LDS_BYTES"] <= MAX_LDS_BYTES
        and g["LPTX"] <= MAX_LOADS_PER_THREAD
        and params.r * g["NB4"] <= MAX_ACCUMULATORS
        and config.prefetch >= 2
        and config.prefetch % 2 == 0
        and config.rows in (1, 2)
        and config.pipe in (0, 1)
        and 0 <= config.block_q <= params.q
        and (g["LPTX"] + g["LPTD"]) * config.prefetch * config.rows <= 32
        # one row of all images side by side lies within 32-bit buffer offsets
        and ((config.block_n - 1) * max(params.h * params.w, params.p * params.q) + max(params.w, params.q))
        * params.c * 2 < 2**31
        # general bound on the tensors' 16-byte units
        and params.n * params.groups * max(params.h * params.w, params.p * params.q) < 2**31
    )


def _fits(params, config) -> bool:
    """Whether a lane's registers hold the sums, the last grad_output rows, the rows in flight and a step's operands
    (weights fitted to what the compiler reports for 480 kernels of 80 shapes: of 9 that used memory 3 pass, all by
    16 bytes or less but one, of 471 others 3 do not)."""
    g = wgrad_geometry(params, config)
    loads = g["LPTX"] + g["LPTD"]
    operands = g["CPW"] * config.rows * (g["NB4"] + 1) * (2 if config.pipe else 1)
    needed = (4.1 * params.r * g["NB4"] + 3.6 * params.r * g["CPW"] + 2.0 * operands
              + 2.9 * config.prefetch * config.rows * loads + 3.7 * loads + 23)  # fmt: skip
    return needed <= 1.02 * lane_registers(config.groups * config.split)


def _config_is_legal(params, config) -> bool:
    """Whether the MFMA kernel can run a configuration."""
    return (
        config.variant == "mfma"
        and min(config.groups, config.block_h, config.block_n, config.block_n_iters, config.split) >= 1
        and config.two_stage in (0, 1)
        and _mfma_config_is_legal(params, config)
    )


def image_block_runs(blocks: int, tiles: int, num_cus: int, sizes) -> List[int]:
    """Image blocks a workgroup takes one after the other: as many workgroups as `sizes` give, but with equal
    shares, and those with which the grid of `tiles` per image block is one or two whole rounds of the device.

    A round lasts as long as its longest workgroup.  Weight gradient 20n 1024c 27x27 5x5, two images a block:
    runs of 8 are 8 and 2 blocks."""
    runs = set(balanced(blocks, sizes))
    for rounds in (1, 2):
        workgroups = min(blocks, num_cus * rounds // tiles)
        if workgroups:
            runs.add(divup(blocks, workgroups))
    return sorted(r for r in runs if r <= 16)


def _mfma_score(params, config, num_cus) -> float:
    """Rough relative cost used only to order (and cap) the sweep; lower is better."""
    g = wgrad_geometry(params, config)
    halo = (config.block_h + params.r - 1) / config.block_h
    traffic = 1.0 + 0.5 * (halo - 1.0) + 0.25 * (params.s - 1) / g["BQ"]
    group_eff = params.groups / (g["GBLKS"] * config.groups)
    # compute units idle in the last round of workgroups, and in the last, shorter tiles
    quant = divup(g["NUM_BLOCKS"], num_cus) * num_cus / g["NUM_BLOCKS"]
    quant *= g["PBLKS"] * config.block_h / params.p * g["NBLKS"] * config.block_n * config.block_n_iters / params.n
    quant *= g["QBLKS"] * g["BQ"] / params.q
    # Publishing costs R*S*64 values per (workgroup, group): atomics retire at roughly 128 per
    # clock device-wide; partial stores plus the reduction kernel cost bandwidth and a launch.
    stream_bytes = 4.0 * params.n * params.c * params.h * params.w
    stream_us = stream_bytes / 5.0e6
    values = g["NUM_BLOCKS"] * config.groups * params.r * params.s * 64.0
    if config.two_stage:
        publish_us = 4.5 + 2.0 * 4.0 * values / 5.0e6
    else:
        publish_us = values / (128 * 2.1e3)
    # blocks of part of a line; they cost more where a pixel is not whole lines, so that blocks straddle them (184n
    # 288c 31x31 3x3: 4 groups 50.4 us, 8 groups, of which the last block has half, 42.1; best of a first use over ten
    # such shapes with 1.12 and 1.2: that one 47.0 and 41.0, 23n 1360c 29x18 22.9 and 21.2, the others equal)
    split_line = 1.0 if (config.groups * 16) % 128 == 0 or config.groups == params.groups else (
        1.12 if params.c % 64 == 0 else 1.2)
    return (traffic * quant * split_line / (g["PIXEL_EFF"] ** 0.3 * group_eff)) * (
        1.0 + publish_us / stream_us
    )


def _get_configs(params: Conv2dGw8Params, device_attr=None) -> List[Conv2dGw8WgradConfig]:
    """Legal configurations, most promising first; a direct-kernel configuration closes the list."""
    num_cus = getattr(device_attr, "multiprocessor_count", 256) or 256
    G = params.groups
    # powers of two, the whole pixel, and half a pixel where the group count is not a power of two
    # (96 channels: 12 groups = 2 x 6)
    group_choices = sorted({g for g in (4, 8, 16, G, G // 2 if G % 2 == 0 and G & (G - 1) else G)
                            if 0 < g <= min(G, MAX_WAVES)}) or [min(G, MAX_WAVES)]
    row_choices = balanced(params.p, (4, 7, 8, 14, 16, 28, 32, 56, params.p))
    # Images side by side.  The contraction runs over 32-pixel chunks of the flattened row, so
    # where a padded image row is shorter than a chunk the count decides how full the chunks
    # are: besides the powers of two, the counts that fill them clearly better (7x7 images with
    # one halo column each side: 8 images fill 56 of 96 pixels, 7 images 49 of 64).
    def chunk_fill(nb):
        return nb * params.q / (32.0 * image_placement(params, nb)["KC"])

    image_counts = [1, 2, 4, 8]
    if params.q + params.s - 1 < 32:
        best = max(chunk_fill(nb) for nb in image_counts)
        image_counts += [nb for nb in (3, 5, 6, 7) if chunk_fill(nb) > best + 0.05]
    # Rank the tile geometries first and keep the best few; each of them is then tried with the
    # pipeline variants (prefetch distance, rows per step), which the score cannot tell apart.
    # column blocks for wide rows only: narrower ones fit whole
    # (one less than whole chunks, which begin a pixel before the block)
    col_choices = [bq for bq in (63, 127, 255) if params.q >= 2 * bq and params.q > 128]
    col_choices = [0] + sorted({*col_choices, *balanced(params.q, col_choices)})
    geometries = []
    for bq in col_choices:
        for gb in group_choices:
            for nb in image_counts if bq == 0 else (1,):
                for bh in row_choices:
                    tiles = divup(G, gb) * divup(params.p, bh) * divup(params.q, bq or params.q)
                    for iters in image_block_runs(divup(params.n, nb), tiles, num_cus, (1, 2, 4, 8)):
                        for two_stage in (0, 1):
                            for ts in (1, 2):
                                cfg = Conv2dGw8WgradConfig(groups=gb, block_h=bh, block_n=nb, block_n_iters=iters,
                                                           prefetch=2, two_stage=two_stage, split=ts, block_q=bq)  # fmt: skip
                                if _mfma_config_is_legal(params, cfg):
                                    geometries.append((_mfma_score(params, cfg, num_cus), cfg))
    geometries.sort(key=lambda sc: sc[0])
    # The head of the list, which is all that a sweep inside an operator call tries, holds three geometries:
    # the score is not good enough to spend it on the pipelines of one.
    head, rest = [], []
    for i, (_, base) in enumerate(geometries[:MAX_GEOMETRIES]):
        for j, (pf, rows, pipe) in enumerate(PIPELINE_CHOICES):
            if pf > 2 and pf * rows > base.block_h + params.r - 1:
                continue
            cfg = replace(base, prefetch=pf, rows=rows, pipe=pipe)
            if _mfma_config_is_legal(params, cfg):
                (head if i < 3 and j < LEADING_PIPELINES else rest).append(cfg)
    # what keeps part of its registers in memory comes last (64n 96c 56x56 7x7: 500 us, 35 without)
    configs = sorted(head + rest, key=lambda cfg: not _fits(params, cfg))
    total_pix = params.n * params.p * params.q
    chunks = max(1, min(divup(8 * num_cus, params.groups), divup(total_pix, 64)))
    configs.append(Conv2dGw8WgradConfig(groups=1, block_h=1, block_n=1, block_n_iters=1,
                                        chunks=chunks, variant="direct"))  # fmt: skip
    return configs


def _get_kernel_spec(params: Conv2dGw8Params, config: Conv2dGw8WgradConfig, _device_attr=None) -> KernelSpec:
    params.validate()
    defines = _shape_defines(params)
    # with a bias the kernels take a fourth pointer and also accumulate grad_bias
    defines["SPIO_HAS_BIAS"] = int(params.has_bias)
    if config.variant == "direct":
        threads = 256
        defines.update(SPIO_WGRAD=1, SPIO_BLOCK_THREADS=threads, SPIO_WGRAD_CHUNKS=config.chunks)
        return KernelSpec(
            defines, LaunchParams(grid=params.groups * config.chunks, block=threads), DIRECT_SOURCE
        )
    if config.variant != "mfma":
        raise ValueError(f"unknown kernel variant {config.variant!r}")
    assert _mfma_config_is_legal(params, config), f"illegal configuration {config} for {params}"
    g = wgrad_geometry(params, config)
    defines.update(SPIO_GB=config.groups, SPIO_BH=config.block_h, SPIO_NB=config.block_n,
                   SPIO_ITERS=config.block_n_iters, SPIO_PF=config.prefetch,
                   SPIO_TS=config.split, SPIO_RB=config.rows)  # fmt: skip
    if config.pipe:
        defines["SPIO_PIPE"] = 1
    if config.block_q:
        defines["SPIO_BQ"] = config.block_q
    spec = KernelSpec(defines, LaunchParams(grid=g["NUM_BLOCKS"], block=g["THREADS"]), MFMA_SOURCE, notes=g)
    if config.two_stage:
        num_partials = g["NBLKS"] * g["PBLKS"] * g["QBLKS"]
        # float4 columns of a partial image: grad_weight, and the groups missing in the last channel block
        cols = g["GBLKS"] * config.groups * params.r * params.s * 16
        # columns per workgroup of the second stage
        reduce_cols = 32 if cols >= 32 * 256 else 8
        defines.update(SPIO_PARTIALS=1, SPIO_REDUCE_COLS=reduce_cols)
        bias_floats = num_partials * g["GBLKS"] * config.groups * 8 if params.has_bias else 0
        spec.workspace_bytes = num_partials * cols * 16 + bias_floats * 4
        spec.epilogue_suffix = "_reduce"
        spec.epilogue_half_suffix = "_reduce_h"  # with a bias it takes grad_bias as well and stores it
        spec.overwrites_output = True  # the second stage stores grad_weight whole
        spec.epilogue_launch_params = LaunchParams(grid=divup(cols, reduce_cols), block=256)
        bias_blocks = g["GBLKS"] if params.has_bias else 0
        spec.epilogue_half_launch_params = LaunchParams(grid=divup(cols, reduce_cols) + bias_blocks, block=256)
    return spec


# Partial sums up to this many bytes are published in two stages where grad_weight ends as float16.  Atomics take
# longer the more sums there are, too: forward and weight gradient, atomics -> two stages, 64n 256c 28x28 5x5 with 16
# MB 51 -> 47 us, with 32 MB 65 -> 56, 128n 256c 14x14 7x7 with 15 MB 43 -> 36, 3x3 with 25 MB 128n 64c 56x56 64 -> 60 and
# 64n 256c 28x28 45 -> 46.  (Chosen configurations have 15 MB at most, and those with more than 7 are two-stage
# ones by the sweep's choice.)
STORED_SUMS_BYTES = 32 * 1024 * 1024


def stored_sums(factory, params: Conv2dGw8Params, config):
    """The configuration to run where grad_weight is wanted as float16: `config`, or its two-stage version.

    A kernel that adds its sums with atomics needs them cleared before and rounded to float16 after it, a
    launch each; the second stage of a two-stage kernel stores float16 itself.  Fill + kernel + rounding ->
    two stages, captured in a graph: fused backward 32n 64c 56x56 19.7 -> 17.6 us, 128n 41.1 -> 38.1, 512n
    131.1 -> 127.6, 128n 96c 64.8 -> 60.1, 2n 1024c 20x20 12.9 -> 12.9; weight gradient 4n 120c 39x39 11.4 ->
    9.5, 128n 768c 7x7 15.0 -> 12.6.  With float32 sums only the fill is saved and the two are equal (128n 38.0
    and 38.1), so there the sweep's choice stands."""
    if config.two_stage or getattr(config, "variant", "mfma") != "mfma":
        return config
    stored = replace(config, two_stage=1)
    try:
        spec = factory.get_kernel_spec(params, stored)
    except AssertionError:  # its scratch does not fit
        return config
    return stored if spec.workspace_bytes <= STORED_SUMS_BYTES else config


def _make_test_args(params: Conv2dGw8Params, device):
    """Synthetic (grad_weight, x, dy[, grad_bias]) for timing."""
    cl = torch.channels_last
    x = torch.randn(params.input_shape, device=device, dtype=torch.float16).contiguous(memory_format=cl)
    dy = torch.randn(params.output_shape, device=device, dtype=torch.float16).contiguous(memory_format=cl)
    dw = torch.zeros(params.weight_shape, device=device, dtype=torch.float32).contiguous(memory_format=cl)
    if params.has_bias:
        return (dw, x, dy, torch.zeros(params.c, device=device, dtype=torch.float32))
    return (dw, x, dy)


conv2d_gw8_wgrad_kernel_factory = KernelFactory(
    Conv2dGw8Params,
    Conv2dGw8WgradConfig,
    Conv2dStats,
    kernel_name="spio_conv2d_gw8_wgrad",
    configs=_get_configs,
    kernel_spec=_get_kernel_spec,
    make_test_args=_make_test_args,
    is_legal=_config_is_legal,
)
