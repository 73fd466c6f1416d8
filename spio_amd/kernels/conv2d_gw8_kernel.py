"""Forward / data-gradient kernel family of conv2d_gw8.

Reference: spio/kernels/conv2d_gw8_kernel.py:30-238 (`Conv2dGw8Config`,
`_get_configs`, `_get_kernel_spec`; `igrad=True` selects the data gradient,
which reuses the forward kernel with the flipped, group-transposed filter and
padding (R-1-py, S-1-px), :73-83).  The tile configuration is re-designed for
CDNA4: see csrc/conv2d_gw8_mfma.hip (row-streaming kernel) and
csrc/conv2d_gw8_image_mfma.hip (whole-image kernel for small images) for what
the fields mean on the device.
"""

from dataclasses import dataclass, replace
from typing import Dict, List

import torch

from ..util.math import balanced, divup
from .conv2d_gw8_params import Conv2dGw8Params
from .conv2d_stats import Conv2dStats
from .kernel import KernelSpec
from .kernel_factory import KernelFactory
from .launch_params import LaunchParams

MFMA_SOURCE = "conv2d_gw8_mfma.hip"
IMAGE_SOURCE = "conv2d_gw8_image_mfma.hip"
DIRECT_SOURCE = "conv2d_gw8_direct.hip"

MAX_WAVES = 16
MAX_LDS_BYTES = 128 * 1024
MAX_UNROLLED_STEPS = 64  # SPIO_MAX_UNROLL of the kernel: up to here the step loop is fully unrolled
MAX_LOADS_PER_THREAD = 8
MAX_ACCUMULATORS = 18
DEVICE_LDS_BYTES = 160 * 1024
MAX_IMAGE_CONFIGS = 10  # whole-image configurations that enter the sweep
MOVER_WAVES = 4  # data-mover waves of the whole-image kernel where it has any: one per SIMD
PREFETCH_CHOICES = (2, 4, 8, 10, 12, 16)
COLUMN_BLOCK_CHOICES = (64, 128, 256)  # output columns per workgroup where rows are tiled
MAX_GEOMETRIES = 40  # tile geometries that enter the sweep, 20 with two prefetch distances; the best few also try the other cache/XCD policies


@dataclass(frozen=True)
class Conv2dGw8Config:
    """Tile configuration of the forward / data-gradient kernel.

    Attributes:
        groups: channel groups per workgroup (one wave per group and split).
        block_p: output rows per workgroup.
        block_n: images whose rows are laid side by side in one staged row.
        split: waves sharing the 16-pixel tiles of one group.
        prefetch: rows of global loads in flight ahead of the computed row.
        nontemporal: 1 = stream activations with the non-temporal hint (loads only where no
            two channel blocks share lines).
        halo_cached: 1 = load rows shared with neighbouring row blocks with the default
            cache policy so the second reader can hit in L2.
        xcd_chunk: consecutive tiles that go to the same XCD (they share halo rows through its
            L2) before the next run of tiles goes to the next XCD; 0 = one contiguous range of
            tiles per XCD, 1 = tiles dealt round-robin.
        block_n_iters: whole-image kernel only: image blocks a workgroup processes one after
            the other with the same filter fragments.
        variant: "mfma" (row-streaming MFMA kernel), "image" (whole-image MFMA kernel: image
            blocks of block_n images move through LDS whole, `split` waves share a group by
            splitting its accumulators; prefetch = 2 means two LDS buffers each for input and
            output, prefetch = 1 one of each, which lets two workgroups share a CU; block_p and
            the cache/XCD policies do not apply) or "direct" (one thread per output
            pixel-group; any shape).
        movers: whole-image kernel only: extra waves that move the image blocks between global
            memory and LDS for the whole workgroup while the other waves only multiply (0: every
            wave does both).
        block_p2: row-streaming kernel only: a second tile height.  The row blocks of an image
            then alternate between block_p and block_p2 rows, the first half of the grid takes
            the block_p tiles and the second half the block_p2 tiles.  For grids of two
            workgroups per compute unit, which the device starts as two cohorts of which the
            second trails the first by the first's prefetch burst (0: one height).
        block_q: row-streaming kernel only: output columns per workgroup (0: the whole width).
            A workgroup then stages block_q + S - 1 source columns of its rows, so rows of any
            width fit (reference: block_q and block_w, spio/kernels/conv2d_gw8_kernel.py:92-108).
        prefetch_start, prefetch_rate: row-streaming kernel only: rows requested before the
            first step and per step until the requests run `prefetch` rows ahead
            (prefetch_start = 0: all `prefetch` rows at once).
    """

    groups: int = 8
    block_p: int = 16
    block_n: int = 1
    split: int = 1
    prefetch: int = 2
    variant: str = "mfma"
    nontemporal: int = 1
    halo_cached: int = 1
    xcd_chunk: int = 4
    block_n_iters: int = 1
    movers: int = 0
    block_p2: int = 0
    prefetch_start: int = 0
    prefetch_rate: int = 1
    block_q: int = 0


def direction_geometry(params: Conv2dGw8Params, igrad: bool) -> Dict[str, int]:
    """Source/destination extents and effective padding of one direction."""
    if igrad:
        return dict(SH=params.p, SW=params.q, DH=params.h, DW=params.w,
                    EPY=params.transpose_padding_h, EPX=params.transpose_padding_w)  # fmt: skip
    return dict(SH=params.h, SW=params.w, DH=params.p, DW=params.q,
                EPY=params.padding_h, EPX=params.padding_w)  # fmt: skip


def stage_pitch(groups: int) -> int:
    """Bytes from pixel to pixel of a finished row in LDS: an odd number of 16-byte units (spio_conv_common.h)."""
    return 16 * (groups + 1 + groups % 2)


def mfma_geometry(params: Conv2dGw8Params, config: Conv2dGw8Config, igrad: bool) -> Dict[str, int]:
    """Host mirror of the compile-time constants of conv2d_gw8_mfma.hip."""
    d = direction_geometry(params, igrad)
    r, s = params.r, params.s
    gb, bp, nb, ts = config.groups, config.block_p, config.block_n, config.split
    bp2 = config.block_p2
    bq = config.block_q or d["DW"]
    kb = (s + 4) // 4
    wpi = bq + s - 1
    f = nb * wpi
    tiles = divup(f - s + 1, 32)  # a product takes 16 pairs of pixels
    tpw = divup(tiles, ts)
    fp = 32 * tpw * ts + 4 * kb - 2
    plane = fp // 2 + (8 - fp // 2) % 16
    gs = plane + fp // 2 + (9 - (plane + fp // 2)) % 16
    threads = 64 * gb * ts
    ostride = stage_pitch(gb)
    # ring rows (+ dump cell) and two output-stage rows
    lds = 2 * (gb * gs + 1) * 16 + 4 * (16 * tpw * ts * ostride + 128)
    if igrad:  # the data gradient stages its groups' filters in the same block first
        lds = max(lds, gb * 8 * r * s * 16)
    d.update(
        KB=kb, WPI=wpi, F=f, WT=2 * tiles, TPW=tpw, GS=gs,  # WT in 16 pixels, as the image kernel's; the kernel's own is tiles
        THREADS=threads, LDS_BYTES=lds, LPT=divup(f * gb, threads),
        SPT=divup(nb * bq * gb, threads), BQ=bq, QBLKS=divup(d["DW"], bq),
        GBLKS=divup(params.groups, gb), NBLKS=divup(params.n, nb),
        # two tile heights: PBLKS (block_p, block_p2) pairs per image, one workgroup per tile
        PBLKS=divup(d["DH"], bp + bp2) if bp2 else divup(d["DH"], bp),
        STEPS=max(bp, bp2) + r - 1,
    )  # fmt: skip
    d["NUM_BLOCKS"] = (2 if bp2 else 1) * d["GBLKS"] * d["PBLKS"] * d["QBLKS"] * d["NBLKS"]
    return d


def lane_registers(waves: int) -> int:
    """Registers a lane has where `waves` waves share a compute unit's four SIMDs (512 a lane and SIMD, dealt in
    eights).  A kernel that needs more keeps the rest in memory."""
    return {1: 512, 2: 256, 3: 168, 4: 128}.get(divup(waves, 4), 0)


def _mfma_fits(params, config, igrad) -> bool:
    """Whether a lane's registers hold what the row-streaming kernel keeps in them, or all but a few: filter fragments,
    accumulators and rows in flight.  Against what the compiler reports for 5370 kernels of 207 shapes, 1x1 to 7x7: of
    318 that used memory 13 pass, 12 of them with 76 bytes or less, of 5052 others 124 do not.  (Fitted again, with terms for
    a step's operands and for addresses, 12 and 95.)"""
    g = mfma_geometry(params, config, igrad)
    fragments, accumulators = 4 * params.r * g["KB"], 4 * g["TPW"] * params.r
    rows = 4 * min(config.prefetch, g["STEPS"]) * g["LPT"]
    needed = fragments + 1.6 * accumulators + 1.3 * rows + 6
    return needed <= 1.05 * lane_registers(config.groups * config.split)


def image_geometry(params: Conv2dGw8Params, config: Conv2dGw8Config, igrad: bool) -> Dict[str, int]:
    """Host mirror of the compile-time constants of conv2d_gw8_image_mfma.hip."""
    d = direction_geometry(params, igrad)
    r, s = params.r, params.s
    gb, nb, ts, iters = config.groups, config.block_n, config.split, config.block_n_iters
    ns = 2 * ((r + 1) // 2)
    nacc = ns // 2
    kb = (s + 3) // 4
    wpi = d["DW"] + s - 1
    f = nb * wpi
    wt = divup(f - s + 1, 16)
    fp = 16 * wt + 4 * kb - 1
    gs = fp + ((9 - fp % 16) + 16) % 16
    threads = 64 * (gb * ts + config.movers)
    mthreads = 64 * config.movers if config.movers else threads  # threads that move image blocks
    nbuf = 2 if config.prefetch >= 2 else 1  # prefetch = 1: single buffers (SPIO_DB = 0)
    in_units = d["SH"] * gb * gs
    out_bytes = d["DH"] * 16 * wt * (gb * 16 + 16)
    # input buffers, dump cells, output buffers (which first hold the groups' filters)
    lds = (nbuf * in_units + 32) * 16 + max(nbuf * out_bytes, gb * 8 * r * s * 16)
    lpt = divup(d["SH"] * nb * d["SW"] * gb, mthreads)
    spt = divup(d["DH"] * nb * d["DW"] * gb, mthreads)
    wlpt = divup(gb * 8 * r * s, 64 * gb * ts)  # the multiplying waves fetch the filters
    apw = max(nacc // max(ts, 1), 1)
    # registers per lane.  Multiplying: filter fragments, accumulators, two sets of source
    # fragments; moving: two blocks in flight and their LDS addresses; both: the filter share on
    # its way to LDS and the rest.  Without mover waves every wave holds both sets.
    multiplying = 4 * ns * kb + 4 * wt * apw + 8 * wt * kb
    moving = 8 * lpt + lpt + spt
    if config.movers:
        registers = max(multiplying + 4 * wlpt, moving) + 14
    else:
        registers = multiplying + 4 * max(2 * lpt, lpt + wlpt) + lpt + spt + 14
    # the same with fp32 source, destination and weights, by the number of blocks in flight
    wide = [16 * lpt * sets + 2 * (lpt + spt) for sets in (1, 2)]
    if config.movers:
        wide_registers = [max(multiplying + 8 * wlpt, w) + 14 for w in wide]
    else:
        wide_registers = [multiplying + max(w, 16 * lpt + 8 * wlpt + 2 * (lpt + spt)) + 14 for w in wide]
    d.update(
        WIDE_REGISTERS=wide_registers,
        NS=ns, NACC=nacc, APW=apw, KB=kb, WPI=wpi, F=f, WT=wt, GS=gs, THREADS=threads,
        MTHREADS=mthreads, LDS_BYTES=lds, LPT=lpt, SPT=spt, STEPS=d["DH"] + r - 1,
        GBLKS=divup(params.groups, gb), NBLKS=divup(params.n, nb),
        REGISTERS=registers, NBUF=nbuf,
    )  # fmt: skip
    d["WGBLKS"] = divup(d["NBLKS"], iters)
    d["NUM_BLOCKS"] = d["GBLKS"] * d["WGBLKS"]
    return d


def _register_budget(config) -> int:
    """Registers per lane that leave room for the workgroup's waves on a SIMD (512 in all)."""
    return {1: 232, 2: 232, 3: 160, 4: 128}.get(divup(config.groups * config.split + config.movers, 4), 0)


def float32_block_sets(params, config, igrad) -> int:
    """Image blocks in flight of the whole-image kernel where they are float32: two if the registers allow it,
    one, or none (no such version)."""
    registers = image_geometry(params, config, igrad)["WIDE_REGISTERS"]
    return sum(r <= _register_budget(config) for r in registers)


def _float32_config(params, config, igrad):
    """The configuration a version that reads float32 runs in: without mover waves where the registers allow it.
    Rounding and keeping a block is work that all waves share then (128n 384c 14x14 forward with mover waves
    22.3 us, without 20.4; of float16 blocks 8.6 and 10.4)."""
    without = replace(config, movers=0)
    if config.variant == "image" and config.movers and float32_block_sets(params, without, igrad):
        if _image_config_is_legal(params, without, igrad):
            return without
    return config


def _image_config_is_legal(params, config, igrad) -> bool:
    g = image_geometry(params, config, igrad)
    waves = config.groups * config.split + config.movers
    return (
        waves <= MAX_WAVES
        and config.movers >= 0
        and (config.movers == 0 or (config.prefetch >= 2 and g["MTHREADS"] % config.groups == 0))
        and g["THREADS"] % config.groups == 0
        and config.split >= 1
        and g["NACC"] % config.split == 0
        and config.block_n <= max(params.n, 1)
        and config.block_n_iters >= 1
        and g["LDS_BYTES"] <= DEVICE_LDS_BYTES
        and g["LPT"] <= MAX_LOADS_PER_THREAD
        and g["SPT"] <= MAX_LOADS_PER_THREAD
        and g["STEPS"] <= MAX_UNROLLED_STEPS
        and g["REGISTERS"] <= _register_budget(config)
        and config.block_n * params.c * max(params.h * params.w, params.p * params.q) * 2 < 2**31
    )


def _image_score(params, config, igrad, num_cus: int) -> float:
    """Relative cost of a whole-image configuration; lower is better.  Prices idle compute units
    (grid quantisation; LDS decides how many workgroups a CU holds), wasted MFMA columns, partial
    128-byte lines, the set-up a workgroup pays before its first block (filters through LDS,
    pipeline fill: about two blocks' worth, measured) and, weakly, split accumulators."""
    g = image_geometry(params, config, igrad)
    per_cu = max(1, min(DEVICE_LDS_BYTES // g["LDS_BYTES"], 2048 // g["THREADS"]))
    slots = num_cus * per_cu
    rounds = divup(g["NUM_BLOCKS"], slots)
    quant = rounds * slots / g["NUM_BLOCKS"]
    tile_eff = config.block_n * g["DW"] / (16.0 * g["WT"])
    group_eff = params.groups / (g["GBLKS"] * config.groups)
    split_line = 1.0 if (config.groups * 16) % 128 == 0 or config.groups == params.groups else 1.2
    setup = 1.0 + 2.0 / config.block_n_iters
    split = 1.0 + 0.05 * (config.split - 1)
    single = 1.0 if config.prefetch >= 2 else 1.03
    # mover waves pay where moving a block takes longer than multiplying it (measured: 3x3 on
    # 14x14 0.73x, 5x5 on 9x9 and 14x14 0.97x, 7x7 on 14x14 1.05x; first use of seven 5x5 shapes with them ahead:
    # 128n 1392c 9x9 20.5 -> 19.9 us, the others equal)
    movers = 1.0 if not config.movers else (0.9 if params.r * params.s <= 25 else 1.05)
    ragged = g["WGBLKS"] * config.block_n_iters * config.block_n / params.n
    return quant * ragged * split_line * setup * split * single * movers / (tile_eff * group_eff)


def _whole_round_iters(params, config, igrad, num_cus: int) -> List[int]:
    """Image blocks per workgroup with which the grid is one or two whole rounds of the device.

    A workgroup's set-up (filters through LDS, pipeline fill) costs about two image blocks, so fewer and
    longer workgroups are better until they leave compute units idle.  128n 1392c 9x9 5x5: 22 channel blocks
    leave 11 workgroups each, 12 images a workgroup; forward 21.3 us with 4 images (704 workgroups, 2.75
    rounds) and 21.7 with 16 (176, 0.7 rounds) -> 19.1, data gradient 21.2 -> 18.6."""
    g = image_geometry(params, replace(config, block_n_iters=1), igrad)
    per_cu = max(1, min(DEVICE_LDS_BYTES // g["LDS_BYTES"], 2048 // g["THREADS"]))
    return [divup(g["NBLKS"], max(1, num_cus * per_cu * rounds // g["GBLKS"])) for rounds in (1, 2)]


def _image_configs(params: Conv2dGw8Params, igrad: bool, num_cus: int) -> List[Conv2dGw8Config]:
    """Legal whole-image configurations, most promising first (none for large images)."""
    G = params.groups
    found = []
    for gb in sorted({g for g in (4, 8, 16, G) if g <= min(G, MAX_WAVES)}):
        for nb in (1, 2, 4, 8):
            for ts in (1, 2, 4):
                for buffers, movers in ((2, 0), (1, 0), (2, MOVER_WAVES)):
                    base = Conv2dGw8Config(groups=gb, block_p=direction_geometry(params, igrad)["DH"],
                                           block_n=nb, split=ts, prefetch=buffers, variant="image",
                                           halo_cached=0, xcd_chunk=0, movers=movers)  # fmt: skip
                    if not _image_config_is_legal(params, base, igrad):
                        continue
                    for iters in sorted({1, 2, 4, 8, 16, *_whole_round_iters(params, base, igrad, num_cus)}):
                        if nb * iters > max(params.n, 1) and iters > 1:
                            continue
                        cfg = replace(base, block_n_iters=iters)
                        found.append((_image_score(params, cfg, igrad, num_cus), cfg))
    found.sort(key=lambda sc: sc[0])
    return [cfg for _, cfg in found[:MAX_IMAGE_CONFIGS]]


def _mfma_config_is_legal(params, config, igrad) -> bool:
    g = mfma_geometry(params, config, igrad)
    return (
        config.groups * config.split <= MAX_WAVES
        and config.split <= g["WT"]
        and config.block_n <= max(params.n, 1)
        and config.block_p <= g["DH"]
        and config.block_p2 >= 0
        and (config.block_p2 == 0 or config.block_p + config.block_p2 <= g["DH"])
        and 0 <= config.prefetch_start <= config.prefetch
        and config.prefetch_start != 1
        and config.prefetch_rate >= 1
        and 0 <= config.block_q <= g["DW"]
        and g["LDS_BYTES"] <= MAX_LDS_BYTES
        and g["LPT"] <= MAX_LOADS_PER_THREAD
        and g["TPW"] * params.r <= MAX_ACCUMULATORS
        and config.prefetch >= 2
        # the step loop is always unrolled completely (exact counts of outstanding loads/stores)
        and g["STEPS"] <= MAX_UNROLLED_STEPS
        # 32-bit buffer offsets inside a workgroup's image block
        and config.block_n * params.c * max(params.h * params.w, params.p * params.q) * 2 < 2**31
        and g["LPT"] * config.prefetch <= 24
    )


def _policies_are_legal(config) -> bool:
    return config.nontemporal in (0, 1) and config.halo_cached in (0, 1) and config.xcd_chunk >= 0


def _config_is_legal(params, config, igrad: bool = False) -> bool:
    """Whether the row-streaming or the whole-image kernel can run a configuration."""
    if min(config.groups, config.block_p, config.block_n, config.split, config.prefetch) < 1:
        return False
    if config.variant == "image":
        return _policies_are_legal(config) and _image_config_is_legal(params, config, igrad)
    return (config.variant == "mfma" and config.prefetch % 2 == 0 and _policies_are_legal(config)
            and _mfma_config_is_legal(params, config, igrad))  # fmt: skip


def _resident_workgroups(lds_bytes: int, threads: int) -> int:
    """Workgroups of one kernel a CU can hold (LDS and thread limits)."""
    return max(1, min(160 * 1024 // max(lds_bytes, 1), 2048 // threads, 8))


def _mfma_score(params, config, igrad, num_cus: int) -> float:
    """Rough relative cost used only to order (and cap) the sweep; lower is better.

    The kernel is HBM-bound, so the model prices extra traffic (halo rows),
    idle compute units (grid quantisation), too few bytes in flight (prefetch
    depth x resident workgroups) and, weakly, wasted MFMA columns.
    """
    g = mfma_geometry(params, config, igrad)
    halo = (config.block_p + params.r - 1) / config.block_p * (g["BQ"] + params.s - 1) / g["BQ"]
    traffic = 1.0 + 0.5 * (halo - 1.0)
    useful = config.block_n * g["BQ"]
    tile_eff = useful / (16.0 * g["WT"])
    group_eff = params.groups / (g["GBLKS"] * config.groups)
    per_cu = _resident_workgroups(g["LDS_BYTES"], g["THREADS"])
    # compute units idle in the last round of workgroups
    quant = divup(g["NUM_BLOCKS"], num_cus) * num_cus / g["NUM_BLOCKS"]
    resident = min(per_cu, max(1, g["NUM_BLOCKS"] // num_cus))
    row_bytes = g["F"] * config.groups * 16
    in_flight = resident * min(config.prefetch, g["STEPS"]) * row_bytes
    starve = 1.0 + 0.6 * max(0.0, (64 * 1024 - in_flight) / (64 * 1024))
    few_waves = 1.15 if resident * g["THREADS"] < 512 else 1.0
    # one workgroup on a CU has nothing to run while it waits at its barrier (measured at N=128,
    # C=64, 56x56: 28-row tiles, one per CU, 20.6 us; 14-row tiles, two per CU, 18.8 us)
    alone = 1.04 if resident == 1 else 1.0
    big_block = 1.08 if g["THREADS"] > 512 else 1.0
    # a workgroup that covers only part of a 128-byte line of a pixel shares it with another one
    split_line = 1.0 if (config.groups * 16) % 128 == 0 or config.groups == params.groups else 1.12
    # every row block runs block_p steps, also the last, partly empty one
    ragged = g["PBLKS"] * (config.block_p + config.block_p2) / g["DH"] * g["QBLKS"] * g["BQ"] / g["DW"]
    return traffic * quant * ragged * starve * few_waves * alone * big_block * split_line / (tile_eff ** 0.3 * group_eff)


def _two_height_configs(params, configs, igrad, num_cus) -> List[Conv2dGw8Config]:
    """Variants of the leading geometries with two tile heights, for grids that put exactly two
    workgroups on every compute unit in one round: the device starts such a grid as two cohorts
    and the second trails the first by the first's prefetch burst, so the first half of the
    grid gets taller tiles and the second half shorter ones (measured at N=128, C=64, 56x56:
    14+14 rows 18.8 us, 19+9 rows 18.3 us).  The sweep decides; they rank behind the uniform
    tiles so that a capped sweep is not spent on them."""
    out = []
    seen = set()
    for cfg in configs:
        shape = (cfg.groups, cfg.block_p, cfg.block_n, cfg.split)
        if len(seen) == 2 or shape in seen:
            continue
        g = mfma_geometry(params, cfg, igrad)
        if cfg.variant != "mfma" or cfg.block_p2 or g["NUM_BLOCKS"] != 2 * num_cus:
            continue
        if g["PBLKS"] % 2 or g["DH"] % (2 * cfg.block_p) or cfg.block_p < 4:
            continue
        seen.add(shape)
        for frac in (0.29, 0.36, 0.43):
            delta = max(1, round(cfg.block_p * frac))
            for pf in sorted({cfg.prefetch, 10, 12}):
                cand = replace(cfg, block_p=cfg.block_p + delta, block_p2=cfg.block_p - delta, prefetch=pf)
                if cand not in out and _mfma_config_is_legal(params, cand, igrad):
                    out.append(cand)
    return out


def _get_configs(params: Conv2dGw8Params, device_attr=None, igrad: bool = False) -> List[Conv2dGw8Config]:
    """Legal configurations, most promising first; the direct kernel is always last."""
    d = direction_geometry(params, igrad)
    num_cus = getattr(device_attr, "multiprocessor_count", 256) or 256
    G = params.groups
    # Where a pixel is not whole lines also the groups in the fewest blocks of 12 or of 16 at most (one and a half lines
    # of 128 bytes, or two), all of one size: fewer boundaries lie inside lines, and the last block is not nearly empty.
    even_blocks = {divup(G, divup(G, most)) for most in (12, 16)} if G % 8 else set()
    group_choices = sorted({g for g in {4, 8, 16, G} | even_blocks if g <= min(G, MAX_WAVES)}) or [min(G, MAX_WAVES)]
    row_choices = balanced(d["DH"], (2, 4, 7, 8, 14, 16, 28, 32, 56, d["DH"]))
    # column blocks for wide rows only: narrower ones fit whole and pay no column halo
    col_choices = [bq for bq in COLUMN_BLOCK_CHOICES if d["DW"] >= 2 * bq and d["DW"] > 128]
    col_choices = [0] + sorted({*col_choices, *balanced(d["DW"], col_choices)})
    found = []
    for bq in col_choices:
        for gb in group_choices:
            for nb in (1, 2, 4, 8) if bq == 0 else (1,):
                for ts in (1, 2, 4):
                    if nb * ((bq or d["DW"]) + params.s - 1) - params.s + 1 <= 32 * (ts // 2):
                        continue  # half of the waves or more without a tile (one of four may be: 3 tiles, 1 a wave)
                    for bp in row_choices:
                        steps = bp + params.r - 1
                        for pf in PREFETCH_CHOICES:
                            if pf > 2 and pf > steps:
                                continue
                            cfg = Conv2dGw8Config(groups=gb, block_p=bp, block_n=nb, split=ts, prefetch=pf, block_q=bq)
                            if _mfma_config_is_legal(params, cfg, igrad):
                                found.append((_mfma_score(params, cfg, igrad, num_cus), cfg))
    # Those that keep part of their registers in memory (12 and 16 waves with 5x5 and 7x7 filters) after all others:
    # they are among the slowest (32n 64c 112x112 5x5, the eight that a first use tries: 31 to 114 us, without them
    # 31 to 46; 64n 96c 56x56 7x7 32 to 106, 31 to 40; of all configurations of these and three other shapes none of
    # the best 14 is one)
    found.sort(key=lambda sc: (not _mfma_fits(params, sc[1], igrad), sc[0]))
    # Two prefetch distances of a geometry first, then the others: a capped sweep sees more geometries.  (A geometry
    # that comes up again after 16 others may take two more; without that 49n 264c 34x34 19.8 us, with it 17.9.)
    head, rest = [], []
    for _, cfg in found:
        shape = replace(cfg, prefetch=0)
        (head if sum(replace(h, prefetch=0) == shape for h in head[-16:]) < 2 else rest).append(cfg)
        if len(head) >= MAX_GEOMETRIES:
            break
    rank = {cfg: i for i, (_, cfg) in enumerate(found)}
    if G % 8:
        # Which number of groups is best depends on how lines are shared, which the score does not see: the best geometry
        # of each whose registers fit first (of 16 no more than the others: it was the best of none).  First use of 8, before -> after:
        # 59n 456c 60x60 110 -> 88 us, 64n 144c 56x56 36.5 -> 28.2, 50n 152c 41x41 16.5 -> 13.1, 60n 200c 33x33 17.2 -> 14.7,
        # 7n 168c 159x159 33.2 -> 30.0, 4n 424c 84x84 5x5 20.7 -> 16.7, 2n 600c 147x147 7x7 47 -> 38; 8n 88c 61x40, 48c
        # 224x224, 648c 56x97 5x5 equal.
        # (A number of groups whose registers do not fit gives nothing there, and is left where the order above puts it: with
        # its best first 4n 424c 84x84 5x5 17.3, without 17.1, 2n 600c 147x147 7x7 32.7 and 32.3, 60n 216c 56x56 7x7 53.8 and 54.2.)
        tried = dict.fromkeys(cfg.groups for _, cfg in found if cfg.groups in even_blocks or cfg.groups != 16)
        leaders = [next((cfg for _, cfg in found if cfg.groups == g and _mfma_fits(params, cfg, igrad)), None) for g in tried]
        leaders = [cfg for cfg in leaders if cfg]
        head = leaders + [cfg for cfg in head if cfg not in leaders]
        rest = [cfg for cfg in rest if cfg not in leaders]
    configs = [*head[:8], *sorted(head[8:] + rest, key=rank.get)][:MAX_GEOMETRIES]
    # the memory-system policies, which the score cannot rank: halo rows with or without the
    # non-temporal hint, and how tiles are dealt to the XCDs
    leading = []  # the first four tile geometries, whatever their prefetch depth
    for cfg in configs:
        shape = (cfg.groups, cfg.block_p, cfg.block_n, cfg.split)
        if shape not in leading:
            if len(leading) == 4:
                break
            leading.append(shape)
    for cfg in list(configs):
        if (cfg.groups, cfg.block_p, cfg.block_n, cfg.split) in leading:
            for hc, ch in ((0, 4), (1, 0), (0, 0)):
                configs.append(replace(cfg, halo_cached=hc, xcd_chunk=ch))
    configs += _two_height_configs(params, configs, igrad, num_cus)
    configs = with_joined_stores(params, configs)
    # small images: the whole-image kernel; its two best candidates go first, so that the capped
    # sweep an operator runs on an unrecorded shape sees both kernels
    image = _image_configs(params, igrad, num_cus)
    if image and image_geometry(params, image[0], igrad)["NUM_BLOCKS"] >= num_cus:
        configs = image[:2] + configs + image[2:]
    else:  # too few image blocks to fill the device with workgroups that each pay the set-up
        configs = configs[:2] + image[:2] + configs[2:] + image[2:]
    configs.append(Conv2dGw8Config(groups=1, block_p=1, block_n=1, split=1, variant="direct"))
    return configs


def with_joined_stores(params: Conv2dGw8Params, configs: list) -> list:
    """`configs` with a second version of the leading eight, right behind each, that stores through L2.

    With an odd number of groups the boundary between two channel blocks is not even 32-byte aligned and
    memory has to merge the parts of a sector that two blocks store, unless L2 does it first.  Measured, best
    of the pairs, non-temporal -> default stores: 60n 216c 56x56 61 -> 48 us, 94n 296c 43x47 83 -> 66 (fused
    backward 110 -> 94); on smaller tensors it costs instead (30n 184c 60x60 20.4 -> 21.8, 32n 808c 20x20
    11.0 -> 11.5), so the sweep decides; a capped one
    does not count the second versions, whose geometry it tries anyway.  With an even number the hint is
    the better one or equal (128n 96c 56x56 29.1 against 35.0)."""
    out = []
    for i, cfg in enumerate(configs):
        out.append(cfg)
        if i < 8 and params.groups % 2 and cfg.groups < params.groups:
            out.append(replace(cfg, nontemporal=0))
    return out


def _shape_defines(params: Conv2dGw8Params) -> Dict[str, object]:
    return {
        "SPIO_N": params.n, "SPIO_C": params.c, "SPIO_H": params.h, "SPIO_W": params.w,
        "SPIO_R": params.r, "SPIO_S": params.s,
        "SPIO_PY": params.padding_h, "SPIO_PX": params.padding_w,
    }  # fmt: skip


def fits_float32_output(params: Conv2dGw8Params, config) -> bool:
    """Whether a configuration can store its activations as float32: an image block of four bytes an
    element has to stay within the 32-bit buffer offsets, as one of two bytes does."""
    block_n = getattr(config, "block_n", 1)
    return block_n * params.c * max(params.h * params.w, params.p * params.q) * 4 < 2**30


def reads_float32(params: Conv2dGw8Params, config, igrad: bool = False, src_f32: bool = False,
                  w_f32: bool = False, keep: bool = False) -> bool:  # fmt: skip
    """Whether a configuration has a version that reads float32 tensors.  The float16 copy it can leave is
    whole only if every source pixel is staged by the workgroup that owns it: padding below the filter size."""
    return (
        config.variant in ("mfma", "image")
        and fits_float32_output(params, config)
        and not (config.variant == "image" and src_f32
                 and not float32_block_sets(params, _float32_config(params, config, igrad), igrad))
        and not (igrad and w_f32)
        and not (keep and src_f32 and (params.padding_h >= params.r or params.padding_w >= params.s))
    )


def _get_kernel_spec(params: Conv2dGw8Params, config: Conv2dGw8Config, _device_attr=None,
                     igrad: bool = False, out_f32: bool = False, src_f32: bool = False,
                     w_f32: bool = False, keep: bool = False) -> KernelSpec:  # fmt: skip
    """Macros and launch geometry for one (params, config, direction); `out_f32`: the destination is a
    float32 tensor (the same values, widened when they are stored); `src_f32`, `w_f32`: source, weights are
    (rounded to float16 as they are read); `keep`: two more arguments, float16 tensors that receive what was
    rounded of the two."""
    params.validate()
    defines = _shape_defines(params)
    if out_f32:
        assert fits_float32_output(params, config), f"no float32 output for {config} and {params}"
        defines["SPIO_DST_F32"] = 1
    if src_f32:
        config = _float32_config(params, config, igrad)
    if src_f32 or w_f32:
        assert reads_float32(params, config, igrad, src_f32, w_f32, keep), f"no float32 input for {config} and {params}"
        defines.update(SPIO_SRC_F32=int(src_f32), SPIO_W_F32=int(w_f32), SPIO_KEEP=int(keep))
    defines["SPIO_IGRAD"] = int(igrad)
    defines["SPIO_HAS_BIAS"] = int(params.has_bias and not igrad)
    if config.variant == "direct":
        d = direction_geometry(params, igrad)
        threads = 256
        defines["SPIO_BLOCK_THREADS"] = threads
        total = params.n * d["DH"] * d["DW"] * params.groups
        return KernelSpec(defines, LaunchParams(grid=divup(total, threads), block=threads), DIRECT_SOURCE)
    if config.variant == "image":
        assert _image_config_is_legal(params, config, igrad), f"illegal configuration {config} for {params}"
        g = image_geometry(params, config, igrad)
        if src_f32:
            defines["SPIO_SETS"] = float32_block_sets(params, config, igrad)
        defines.update(
            SPIO_GB=config.groups, SPIO_NB=config.block_n, SPIO_TS=config.split,
            SPIO_ITERS=config.block_n_iters, SPIO_NT=config.nontemporal,
            SPIO_DB=int(config.prefetch >= 2), SPIO_MV=config.movers,
        )  # fmt: skip
        return KernelSpec(
            defines, LaunchParams(grid=g["NUM_BLOCKS"], block=g["THREADS"]), IMAGE_SOURCE, notes=g
        )
    if config.variant != "mfma":
        raise ValueError(f"unknown kernel variant {config.variant!r}")
    assert _mfma_config_is_legal(params, config, igrad), f"illegal configuration {config} for {params}"
    g = mfma_geometry(params, config, igrad)
    # float32 rows: half as many in flight, which are as many bytes (and registers)
    prefetch = max(2, config.prefetch // 2) if src_f32 else config.prefetch
    defines.update(
        SPIO_GB=config.groups, SPIO_BP=config.block_p, SPIO_NB=config.block_n,
        SPIO_TS=config.split, SPIO_PF=prefetch,
        SPIO_NT=config.nontemporal, SPIO_HALO_CACHED=config.halo_cached,
        SPIO_XCD_CHUNK=config.xcd_chunk,
    )  # fmt: skip
    if config.block_p2:
        defines["SPIO_BP2"] = config.block_p2
    if config.prefetch_start:
        defines["SPIO_PF0"] = max(2, config.prefetch_start // 2) if src_f32 else config.prefetch_start
    if config.prefetch_rate != 1:
        defines["SPIO_PF_RATE"] = config.prefetch_rate
    if config.block_q:
        defines["SPIO_BQ"] = config.block_q
    return KernelSpec(
        defines, LaunchParams(grid=g["NUM_BLOCKS"], block=g["THREADS"]), MFMA_SOURCE, notes=g
    )


def _get_kernel_name(igrad: bool = False, out_f32: bool = False, src_f32: bool = False, w_f32: bool = False,
                     keep: bool = False) -> str:  # fmt: skip
    name = ("spio_conv2d_gw8_dgrad" if igrad else "spio_conv2d_gw8_fprop") + ("_f32" if out_f32 else "")
    return name + ("_srcf32" if src_f32 else "") + ("_wf32" if w_f32 else "") + ("_keep" if keep else "")


def _make_test_args(params: Conv2dGw8Params, device, igrad: bool = False):
    """Synthetic (dst, src, weight, bias) for timing."""
    cl = torch.channels_last
    x = torch.randn(params.input_shape, device=device, dtype=torch.float16).contiguous(memory_format=cl)
    y = torch.randn(params.output_shape, device=device, dtype=torch.float16).contiguous(memory_format=cl)
    w = (torch.randn(params.weight_shape, device=device, dtype=torch.float16) * 0.1).contiguous(memory_format=cl)
    if igrad:
        return (x, y, w, None)
    bias = torch.randn(params.bias_shape, device=device, dtype=torch.float32) if params.has_bias else None
    return (y, x, w, bias)


conv2d_gw8_kernel_factory = KernelFactory(
    Conv2dGw8Params,
    Conv2dGw8Config,
    Conv2dStats,
    kernel_name=_get_kernel_name,
    configs=_get_configs,
    kernel_spec=_get_kernel_spec,
    make_test_args=_make_test_args,
    is_legal=_config_is_legal,
)
