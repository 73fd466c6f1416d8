"""Host-side kernel infrastructure without a GPU: configuration spaces, launch
geometry, JIT specialisation of every kernel family, caches and the tuner's
record store.  CPU only."""

import json
import os
from dataclasses import replace

import pytest

from helpers import reference_test_params, scratch_bytes
from spio_amd.compiler.compile import compile_hip
from spio_amd.compiler.compile_kernel import kernel_headers, read_source
from spio_amd.hip import DeviceAttributes
from spio_amd.kernels import (
    Conv2dGw8BgradConfig,
    Conv2dGw8Config,
    Conv2dGw8Params,
    Conv2dGw8WgradConfig,
    KernelCache,
    KernelFactory,
    KernelKey,
    KernelParamsLogger,
    LaunchParams,
    conv2d_gw8_bgrad_kernel_factory,
    conv2d_gw8_kernel_factory,
    conv2d_gw8_wgrad_kernel_factory,
    kernel_params_logging_is_enabled,
)
from spio_amd.kernels.conv2d_gw8_kernel import MAX_LDS_BYTES, image_geometry, mfma_geometry
from spio_amd.kernels.tuner import Tuner, config_to_dict, device_key

ATTR = DeviceAttributes()


def test_launch_params_normalisation():
    lp = LaunchParams(grid=7, block=(64, 2))
    assert lp.grid == (7, 1, 1) and lp.block == (64, 2, 1)
    with pytest.raises(AssertionError):
        LaunchParams(grid=0, block=64)
    with pytest.raises(ValueError):
        LaunchParams(grid=(1, 1, 1, 1), block=64)


@pytest.mark.parametrize("igrad", [False, True])
def test_every_shape_has_legal_configs(igrad):
    """Every shape of the reference's test list gets configurations whose derived
    geometry respects the device limits, and the direct kernel closes the list."""
    for params in reference_test_params(False):
        configs = conv2d_gw8_kernel_factory.configs(params, ATTR, igrad=igrad)
        assert configs and configs[-1].variant == "direct"
        assert len(set(configs)) == len(configs)
        for cfg in configs[:-1]:
            if cfg.variant == "image":  # the whole-image kernel has its own geometry
                g = image_geometry(params, cfg, igrad)
                assert g["THREADS"] <= 1024 and g["LDS_BYTES"] <= 160 * 1024 and g["NACC"] % cfg.split == 0
                spec = conv2d_gw8_kernel_factory.get_kernel_spec(params, cfg, ATTR, igrad=igrad)
                assert spec.launch_params.grid[0] == g["NUM_BLOCKS"] == g["GBLKS"] * g["WGBLKS"]
                assert spec.launch_params.block[0] == g["THREADS"]
                assert g["WGBLKS"] * cfg.block_n_iters * cfg.block_n >= params.n
                # data-mover waves come on top of the multiplying waves, need the second pair of
                # buffers, and a moving thread stays with one group
                assert g["THREADS"] == 64 * (cfg.groups * cfg.split + cfg.movers)
                assert g["MTHREADS"] == (64 * cfg.movers if cfg.movers else g["THREADS"])
                assert g["MTHREADS"] % cfg.groups == 0
                assert spec.defines["SPIO_MV"] == cfg.movers
                if cfg.movers:
                    assert cfg.prefetch >= 2 and spec.defines["SPIO_DB"] == 1
                continue
            g = mfma_geometry(params, cfg, igrad)
            assert g["THREADS"] <= 1024 and g["LDS_BYTES"] <= MAX_LDS_BYTES
            assert g["NUM_BLOCKS"] >= 1 and g["WT"] * 16 >= g["F"] - params.s + 1
            assert g["GS"] % 16 == 9 and g["GS"] >= 16 * g["WT"] + 4 * g["KB"] - 1
            spec = conv2d_gw8_kernel_factory.get_kernel_spec(params, cfg, ATTR, igrad=igrad)
            assert spec.launch_params.grid[0] == g["NUM_BLOCKS"]
            assert spec.launch_params.block[0] == g["THREADS"]


def test_model_shapes_and_wide_rows_get_mfma_kernels(capsys):
    """No performance cliff onto the any-shape kernel: every model-derived shape (at its full
    batch) and rows of any width (column blocks: 224, 384, 512, 1024 and 4000 pixels) have an
    MFMA configuration in every family, the fused backward kernel included for 3x3 and 5x5
    filters; a request that has only the any-shape kernel says so on first use."""
    from helpers import GOLDEN

    with open(os.path.join(GOLDEN, "conv2d_gw8_model_shapes.json"), encoding="utf-8") as f:
        rows = json.load(f)
    shapes = [Conv2dGw8Params(n=d["n"], c=d["c"], h=d["h"], w=d["w"], padding=(d["py"], d["px"]),
                              r=d["r"], s=d["s"], has_bias=d["has_bias"]) for d in rows]  # fmt: skip
    shapes += [Conv2dGw8Params(n=8, c=c, h=64, w=w) for c in (64, 256) for w in (64, 96, 128)]
    shapes += [Conv2dGw8Params(n=8, c=256, h=64, w=64, r=7, s=7, padding=3)]
    wide = [Conv2dGw8Params(n=2, c=c, h=20, w=w, r=r, s=r, padding=r // 2, has_bias=b)
            for w in (224, 384, 512, 1024, 4000) for c, r, b in ((64, 3, False), (32, 5, True), (256, 3, True))]  # fmt: skip
    wide += [Conv2dGw8Params(n=2, c=64, h=20, w=w, r=7, s=7, padding=3) for w in (224, 512, 1024)]
    for params in shapes + wide:
        for factory, kw in ((conv2d_gw8_kernel_factory, {}), (conv2d_gw8_kernel_factory, {"igrad": True}),
                            (conv2d_gw8_wgrad_kernel_factory, {})):  # fmt: skip
            configs = factory.configs(params, ATTR, **kw)
            assert any(c.variant == "mfma" for c in configs), f"{factory.get_full_kernel_name(params, **kw)}: direct only"
    for params in wide:
        if params.r <= 5:
            configs = list(conv2d_gw8_bgrad_kernel_factory.configs(params, ATTR))
            assert configs and all(c.block_q % 32 == 0 for c in configs), f"fused backward: none for {params.encode()}"
            if params.w >= 512:
                assert all(c.block_q > 0 for c in configs)

    # the cliff is announced where a request has nothing but the any-shape kernel
    huge = Conv2dGw8Params(n=1, c=64, h=8, w=4000)
    direct_only = KernelFactory(Conv2dGw8Params, Conv2dGw8Config, None, kernel_name="spio_conv2d_gw8_fprop",
                                configs=lambda p, a: [Conv2dGw8Config(variant="direct")],
                                kernel_spec=None)  # fmt: skip

    class Stop(Exception):
        pass

    def no_compile(*a, **k):
        raise Stop

    import spio_amd.kernels.kernel_cache as kernel_cache

    saved = kernel_cache.compile_and_load_kernel
    kernel_cache.compile_and_load_kernel = no_compile
    try:
        with pytest.raises(Stop):
            Tuner().best_kernel(direct_only, huge, 0, ATTR)
    finally:
        kernel_cache.compile_and_load_kernel = saved
    assert "no MFMA configuration fits" in capsys.readouterr().err


def test_kernel_names_follow_the_reference_convention():
    p = Conv2dGw8Params(n=4, c=64, h=16, w=32, has_bias=True)
    f = conv2d_gw8_kernel_factory
    assert f.get_full_kernel_name(p) == "spio_conv2d_gw8_fprop__4n_64c_16h_32w_1py_1px_3r_3s_b"
    assert f.get_full_kernel_name(p, igrad=True).startswith("spio_conv2d_gw8_dgrad__")
    assert conv2d_gw8_wgrad_kernel_factory.get_full_kernel_name(p).startswith("spio_conv2d_gw8_wgrad__")
    assert f.get_kernel_cache() is f.get_kernel_cache()
    assert f.get_kernel_cache() is not f.get_kernel_cache(igrad=True)


@pytest.mark.parametrize(
    "params",
    [
        Conv2dGw8Params(n=4, c=64, h=16, w=32, has_bias=True),
        Conv2dGw8Params(n=3, c=24, h=20, w=19, padding=(2, 0), r=4, s=1),
        Conv2dGw8Params(n=2, c=32, h=14, w=14, padding=3, r=7, s=7),
        Conv2dGw8Params(n=3, c=24, h=20, w=19, padding=(0, 2)),
    ],
    ids=lambda p: p.encode(),
)
def test_jit_specialisation_of_every_family(params):
    """hipRTC compiles first/last configuration of each family for gfx950 (no GPU needed)."""
    for factory, kw in ((conv2d_gw8_kernel_factory, {}), (conv2d_gw8_kernel_factory, {"igrad": True}),
                        (conv2d_gw8_wgrad_kernel_factory, {}), (conv2d_gw8_bgrad_kernel_factory, {})):  # fmt: skip
        configs = list(factory.configs(params, ATTR, **kw))
        if not configs:  # the fused backward kernel has no configuration for 7x7 (registers)
            assert factory is conv2d_gw8_bgrad_kernel_factory
            continue
        for cfg in {configs[0], configs[-1]}:
            kernel = factory.make_kernel(params, cfg, ATTR, **kw)
            kernel.compile()
            assert kernel.code[:4] == b"\x7fELF"
            assert kernel.kernel_name.encode() in kernel.code
            with pytest.raises(ValueError):
                kernel.launch()  # not loaded


def test_packaged_tuning_records_name_configurations_that_still_exist():
    """A packaged record whose configuration is no longer a candidate would be ignored and
    trigger a sweep on first use; keep the records in step with the configuration spaces."""
    import dataclasses
    import os

    import spio_amd.kernels as kernels_pkg

    from spio_amd.kernels import LayerNorm2dParams, layernorm_2d_bwd_kernel_factory, layernorm_2d_kernel_factory

    families = {
        "spio_conv2d_gw8_fprop": (conv2d_gw8_kernel_factory, {}),
        "spio_conv2d_gw8_dgrad": (conv2d_gw8_kernel_factory, {"igrad": True}),
        "spio_conv2d_gw8_wgrad": (conv2d_gw8_wgrad_kernel_factory, {}),
        "spio_conv2d_gw8_bgrad": (conv2d_gw8_bgrad_kernel_factory, {}),
        "spio_layernorm_2d": (layernorm_2d_kernel_factory, {}),
        "spio_layernorm_2d_bwd": (layernorm_2d_bwd_kernel_factory, {}),
    }
    tuned = os.path.join(os.path.dirname(kernels_pkg.__file__), "tuned")
    checked = 0
    for fname in os.listdir(tuned):
        arch, cus = fname[: -len(".json")].rsplit("_", 1)
        attr = dataclasses.replace(DeviceAttributes(), arch=arch, multiprocessor_count=int(cus[:-2]))
        with open(os.path.join(tuned, fname), encoding="utf-8") as f:
            records = json.load(f)
        for key, record in records.items():
            name, encoded = key.split("__")
            factory, kw = families[name]
            params = (LayerNorm2dParams if name.startswith("spio_layernorm_2d") else Conv2dGw8Params).decode(encoded)
            config = factory.config_cls(**record["config"])
            assert config in list(factory.configs(params, attr, **kw)), f"stale record {key}: {config}"
            assert record["us"] > 0
            checked += 1
    assert checked > 0


def test_illegal_config_is_rejected():
    p = Conv2dGw8Params(n=1, c=64, h=8, w=16)
    with pytest.raises(AssertionError):
        conv2d_gw8_kernel_factory.get_kernel_spec(p, Conv2dGw8Config(groups=16, split=4), ATTR)
    with pytest.raises(ValueError):
        conv2d_gw8_kernel_factory.get_kernel_spec(p, Conv2dGw8Config(variant="nope"), ATTR)


def test_overlay_cache_semantics():
    """A non-empty overlay must contain the key (reference: kernel_cache.py:62-68)."""
    import torch

    cache = KernelCache()
    p = Conv2dGw8Params(n=1, c=8, h=4, w=4)
    sentinel = object()
    cache.update_overlay({KernelKey(device_ordinal=0, params=p): sentinel})
    dev = torch.device("cuda", 0)
    assert cache.get(conv2d_gw8_kernel_factory, p, dev) is sentinel
    with pytest.raises(ValueError, match="overlay"):
        cache.get(conv2d_gw8_kernel_factory, Conv2dGw8Params(n=2, c=8, h=4, w=4), dev)
    cache.clear_overlay()


def test_params_logger_records_requests():
    import torch

    cache = KernelCache()
    p = Conv2dGw8Params(n=1, c=8, h=4, w=4)
    cache.update_overlay({KernelKey(device_ordinal=0, params=p): object()})
    assert not kernel_params_logging_is_enabled()
    with KernelParamsLogger() as logger:
        assert kernel_params_logging_is_enabled()
        cache.get(conv2d_gw8_kernel_factory, p, torch.device("cuda", 0), igrad=True)
    assert not kernel_params_logging_is_enabled()
    (rec,) = logger.get_logged_params()
    assert rec.params == p and rec.kernel_kwargs == (("igrad", True),)
    assert rec.key == KernelKey(device_ordinal=0, params=p)


def test_tuner_record_store(tmp_path, monkeypatch):
    monkeypatch.setenv("SPIO_TUNE_DB", str(tmp_path / "db.json"))
    t = Tuner()
    assert t.lookup(ATTR, "k__x") is None
    t._store(ATTR, "k__x", {"config": {"groups": 8}, "us": 12.5})
    assert Tuner().lookup(ATTR, "k__x")["us"] == 12.5
    assert device_key(ATTR) == "gfx950_256cu"
    assert json.load(open(tmp_path / "db.json"))["k__x"]["config"] == {"groups": 8}


@pytest.mark.parametrize("factory,mode,config,used", [
    # tiles of an earlier list: heights that do not divide 56 rows evenly
    (conv2d_gw8_kernel_factory, {}, Conv2dGw8Config(groups=8, block_p=16, prefetch=4), True),
    (conv2d_gw8_kernel_factory, {"igrad": True}, Conv2dGw8Config(groups=8, block_p=16, prefetch=4), True),
    (conv2d_gw8_wgrad_kernel_factory, {}, Conv2dGw8WgradConfig(groups=8, block_h=16), True),
    (conv2d_gw8_bgrad_kernel_factory, {}, Conv2dGw8BgradConfig(groups=8, block_h=16), True),
    # not a configuration of this kernel, or not one it can run
    (conv2d_gw8_kernel_factory, {}, Conv2dGw8Config(groups=8, block_p=64, prefetch=4), False),
    (conv2d_gw8_kernel_factory, {}, Conv2dGw8Config(groups=8, block_p=16, prefetch=4, halo_cached=2), False),
    (conv2d_gw8_kernel_factory, {}, Conv2dGw8Config(groups=0, block_p=16, prefetch=4), False),
    (conv2d_gw8_kernel_factory, {}, Conv2dGw8Config(groups=8, block_p=16, prefetch=None), False),
    (conv2d_gw8_wgrad_kernel_factory, {}, Conv2dGw8WgradConfig(groups=8, block_h=16, block_n_iters=0), False),
    (conv2d_gw8_bgrad_kernel_factory, {}, Conv2dGw8BgradConfig(groups=8, block_h=16, block_q=40), False),
    (conv2d_gw8_wgrad_kernel_factory, {}, Conv2dGw8WgradConfig(variant="direct", chunks=0), False),
])  # fmt: skip
def test_a_recorded_choice_is_used_while_the_kernel_can_run_it(factory, mode, config, used, tmp_path, monkeypatch):
    """Records are kept longer than the lists of candidates they were chosen from."""
    from spio_amd.kernels import kernel_cache

    monkeypatch.setenv("SPIO_TUNE_DB", str(tmp_path / "db.json"))
    monkeypatch.setenv("SPIO_TUNE", "0")
    params = Conv2dGw8Params(n=37, c=64, h=56, w=56)
    tuner = Tuner()
    tuner._store(ATTR, factory.get_full_kernel_name(params, **mode), {"config": config_to_dict(config), "us": 1.0})
    monkeypatch.setattr(kernel_cache, "compile_and_load_kernel", lambda f, p, c, *a, **kw: c)
    first = list(factory.configs(params, ATTR, **mode))[0]
    assert config not in factory.configs(params, ATTR, **mode) and config != first
    assert tuner.best_kernel(factory, params, 0, ATTR, **mode) == (config if used else first)


def test_small_image_shapes_offer_mover_wave_configurations():
    """The whole-image kernel is offered with and without data-mover waves for the small-image
    shapes; for 3x3 filters both are among the first candidates (a sweep cut short sees both)."""
    for shape in ("128n_384c_14h_14w_1py_1px_3r_3s_b", "256n_256c_14h_14w_3py_3px_7r_7s_nb"):
        params = Conv2dGw8Params.decode(shape)
        configs = conv2d_gw8_kernel_factory.configs(params, ATTR)
        image = [c for c in configs if c.variant == "image"]
        assert any(c.movers for c in image) and any(not c.movers for c in image)
        if params.r == 3:  # where moving a block takes longer than multiplying it
            assert {bool(c.movers) for c in configs[:4] if c.variant == "image"} == {False, True}
    # illegal: mover waves with single buffers, or more waves than a workgroup holds
    params = Conv2dGw8Params.decode("128n_384c_14h_14w_1py_1px_3r_3s_b")
    for bad in (Conv2dGw8Config(groups=8, block_p=14, variant="image", prefetch=1, movers=4, block_n_iters=2),
                Conv2dGw8Config(groups=8, block_p=14, variant="image", prefetch=2, movers=12, block_n_iters=2)):
        with pytest.raises(AssertionError):
            conv2d_gw8_kernel_factory.get_kernel_spec(params, bad, ATTR)


def test_layernorm_lane_choices():
    """Lanes per pixel: one unit per lane by default; where C/8 is not a power of two also the
    largest power of two dividing it, both among the first candidates."""
    from spio_amd.kernels import LayerNorm2dParams, layernorm_2d_kernel_factory

    expected = {96: 4, 192: 8, 384: 16, 768: 32, 64: None, 40: None, 2048: None}
    for c, exact in expected.items():
        params = LayerNorm2dParams(n=2, c=c, h=3, w=5)
        configs = layernorm_2d_kernel_factory.configs(params, ATTR)
        assert len(set(configs)) == len(configs)
        lanes = {cfg.lanes for cfg in configs}
        assert lanes == ({0, exact} if exact else {0})
        if exact:
            assert {cfg.lanes for cfg in configs[:2]} == {0, exact}
        for cfg in configs:
            spec = layernorm_2d_kernel_factory.get_kernel_spec(params, cfg, ATTR)
            lpp = spec.defines["SPIO_LN_LPP"]
            upl = -(-(c // 8) // lpp)
            assert lpp & (lpp - 1) == 0 and lpp * upl >= c // 8 and cfg.unroll * upl <= 8


def test_layernorm_eps_encodes_to_identifier_characters_and_round_trips():
    """The encoded parameters become part of the kernel's extern "C" symbol: every eps must give
    identifier characters only, decode back to the same value, and compile."""
    import re

    from spio_amd.kernels import LayerNorm2dParams, layernorm_2d_bwd_kernel_factory, layernorm_2d_kernel_factory

    assert LayerNorm2dParams(n=2, c=96, h=7, w=7).encode() == "2n_96c_7h_7w_1em06eps_wb"  # recorded names
    for eps in (1e-3, 1e-4, 0.1, 1.5e-5, 1e-12, 1e-5, 1e-6, 1.0, 2.5, 1e20):
        params = LayerNorm2dParams(n=2, c=96, h=7, w=7, eps=eps, has_bias=False)
        name = params.encode()
        assert re.fullmatch(r"[A-Za-z0-9_]+", name), name
        assert LayerNorm2dParams.decode(name) == params
    for factory in (layernorm_2d_kernel_factory, layernorm_2d_bwd_kernel_factory):
        for eps in (1e-3, 1.0):
            params = LayerNorm2dParams(n=2, c=96, h=7, w=7, eps=eps)
            kernel = factory.make_kernel(params, factory.configs(params, ATTR)[0], ATTR)
            kernel.compile()
            assert kernel.code


def test_fused_backward_works_on_the_larger_of_input_and_output():
    """The fused backward kernel's grid and loads per thread follow the domain both tensors sit in:
    the input's size where the output is smaller, the output's where it is larger; with an even
    filter size the two are offset by half a pixel and the domain holds both."""
    from spio_amd.kernels import Conv2dGw8BgradConfig, bgrad_is_supported
    from spio_amd.kernels.conv2d_gw8_bgrad_kernel import bgrad_domain, bgrad_geometry

    cfg = Conv2dGw8BgradConfig(groups=4, block_h=7, block_n=1)
    same = Conv2dGw8Params(n=4, c=32, h=28, w=28, padding=1)
    small = Conv2dGw8Params(n=4, c=32, h=28, w=28, padding=0)  # 26 x 26 output
    large = Conv2dGw8Params(n=4, c=32, h=28, w=28, padding=(3, 1))  # 32 x 28 output
    assert bgrad_domain(same) == bgrad_domain(small) == (28, 28) and bgrad_domain(large) == (32, 28)
    assert bgrad_geometry(small, cfg) == bgrad_geometry(same, cfg)
    assert bgrad_geometry(large, cfg)["PBLKS"] == 5 and bgrad_geometry(large, cfg)["STEPS"] == 7 + 3
    even = Conv2dGw8Params(n=4, c=32, h=28, w=28, r=4, s=1, padding=(2, 0))  # 29 x 28 output
    assert bgrad_domain(even) == (29, 28) and bgrad_geometry(even, cfg)["STEPS"] == 7 + 1 + 3
    assert bgrad_domain(Conv2dGw8Params(n=4, c=32, h=28, w=28, r=4, s=4, padding=(0, 3))) == (28, 31)
    assert all(bgrad_is_supported(p) for p in (same, small, large, even))


def test_weight_gradient_image_placement_reads_the_right_pixels():
    """The staged-row layout of the weight-gradient kernel (images sharing halo columns, chunks
    that hold their own images), restated from its constants: for every grad_output pixel and
    column tap, the x cell the contraction reads is that image's own column, or a cell no image
    ever writes (zero) where the column lies in the padding."""
    from spio_amd.kernels.conv2d_gw8_wgrad_kernel import image_placement

    cases = [(14, 7, 3, (1, 2, 3, 4, 5, 6, 8)), (14, 3, 1, (2, 4, 8)), (7, 3, 1, (4, 7, 8)), (10, 3, 1, (3, 6)),
             (15, 5, 2, (2, 4)), (13, 6, 4, (2, 4)), (28, 3, 1, (1, 2)), (9, 5, 0, (3, 5)), (12, 4, 3, (2, 4))]
    packed_seen = False
    for w, s, px, counts in cases:
        params = Conv2dGw8Params(n=8, c=16, h=w, w=w, r=1, s=s, padding=(0, px))
        q_width = params.q
        for nb in counts:
            g = image_placement(params, nb)
            ip, ipc, kc, xcp = g["IP"], g["IPC"], g["KC"], g["XCP"]
            packed_seen |= bool(g["PACKED"])
            d_off = [(i // ipc) * 32 + (i % ipc) * ip for i in range(nb)]
            x_off = [(i // ipc) * xcp + (i % ipc) * ip for i in range(nb)]
            assert max(d_off) + q_width <= 32 * kc
            assert kc <= (((nb - 1) * (q_width + s - 1) + q_width) + 31) // 32  # never more chunks than before
            owner = {}  # x cell -> (image, column) of the data it holds
            for i in range(nb):
                for col in range(params.w):
                    cell = x_off[i] + col + px
                    assert cell not in owner and cell < g["FPX"]
                    owner[cell] = (i, col)
            for i in range(nb):
                for q in range(q_width):
                    pos = d_off[i] + q
                    chunk, local = divmod(pos, 32)
                    for tap in range(s):
                        cell = chunk * xcp + local + tap  # what the B fragment of this tap reads
                        col = q + tap - px
                        if 0 <= col < params.w:
                            assert owner.get(cell) == (i, col), (w, s, px, nb, i, q, tap)
                        else:
                            assert cell not in owner, (w, s, px, nb, i, q, tap)
    assert packed_seen


def test_counter_figures_in_profiles_were_measured_with_the_committed_kernel_sources():
    """bench.py reads roofline.traffic and mfma_util from profiles/*.md; every such line names the
    kernel source and the digest of the text it was measured with.  A kernel edited after its
    profile was taken would make bench.py report traffic_stale: the committed state has none."""
    import importlib.util
    import re

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    spec = importlib.util.spec_from_file_location("bench_module", os.path.join(root, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    seen = 0
    for workload in ("target", "cfg1", "cfg2", "cfg3"):
        for kernel in ("fprop", "dgrad", "wgrad", "bgrad"):
            for kind in ("traffic_bytes", "mfma_util"):
                value, stale = bench.profile_figure(kind, workload, kernel)
                if value is None:
                    assert (workload, kernel) == ("cfg3", "bgrad")  # 7x7 has no fused backward kernel
                    continue
                assert stale is False, (kind, workload, kernel)
                seen += 1
    assert seen == 30
    # the model bench.py prices every kernel against: launch floor + bytes at the copy's marginal rate
    m = bench.stream_model(18.3, 102769664)
    assert abs(m["stream_model_us"] - (2.2 + 102769664 / 6.2e6)) < 0.01 and 0.9 < m["frac_of_stream_model"] < 1.1
    assert re.fullmatch(r"[0-9a-f]{12}", bench.source_digest("conv2d_gw8_mfma.hip"))


def test_weight_gradient_mfma_kernel_is_not_offered_past_its_32_bit_indices():
    """The MFMA weight-gradient kernel indexes its tensors in 16-byte units with 32-bit integers:
    up to 32 GiB per tensor.  Beyond that only the general kernel (64-bit arithmetic) is offered;
    the forward and fused backward kernels rebase their descriptors per image block and stay."""
    from spio_amd.hip.driver import DeviceAttributes
    from spio_amd.kernels import (
        Conv2dGw8Params,
        conv2d_gw8_bgrad_kernel_factory,
        conv2d_gw8_kernel_factory,
        conv2d_gw8_wgrad_kernel_factory,
    )

    attr = DeviceAttributes()
    fits = Conv2dGw8Params(n=11000, c=64, h=56, w=56)  # 4.4 GB per tensor
    past = Conv2dGw8Params(n=90000, c=64, h=56, w=56)  # 36 GB per tensor
    assert {c.variant for c in conv2d_gw8_wgrad_kernel_factory.configs(fits, attr)} >= {"mfma"}
    assert {c.variant for c in conv2d_gw8_wgrad_kernel_factory.configs(past, attr)} == {"direct"}
    assert conv2d_gw8_kernel_factory.configs(past, attr)[0].variant == "mfma"
    assert conv2d_gw8_bgrad_kernel_factory.configs(past, attr)


def test_second_store_policies_do_not_shorten_a_capped_sweep(monkeypatch):
    """With an odd number of groups in several channel blocks the leading configurations come in two store
    policies; the first `count` geometries of a capped sweep are the same as without them."""
    from spio_amd.kernels.tuner import _leading, _on_miss_limit

    for factory in (conv2d_gw8_kernel_factory, conv2d_gw8_bgrad_kernel_factory):
        odd = list(factory.configs(Conv2dGw8Params(n=50, c=152, h=21, w=41, padding=1), DeviceAttributes()))
        both = odd[:_leading(odd, 8)]
        assert sum(c.nontemporal for c in both) == 8 and any(not c.nontemporal for c in both)
        for before, c in zip(both, both[1:]):
            assert c.nontemporal or replace(c, nontemporal=1) == before
        even = list(factory.configs(Conv2dGw8Params(n=50, c=160, h=21, w=41, padding=1), DeviceAttributes()))
        assert all(c.nontemporal for c in even) and _leading(even, 8) == 8 and _leading(even, 10**6) == len(even)
        monkeypatch.delenv("SPIO_TUNE_MAX_CONFIGS", raising=False)
        assert _on_miss_limit(odd) == len(both) and _on_miss_limit(even) == 8
        monkeypatch.setenv("SPIO_TUNE_MAX_CONFIGS", "4")  # a bound that the caller states counts every version
        assert _on_miss_limit(odd) == 4 and _on_miss_limit(even) == 4


def test_whole_image_configurations_offer_whole_rounds():
    """Among the whole-image configurations is one whose workgroups are one round of the device at most and
    would not be one with fewer image blocks each; every one covers the batch."""
    from types import SimpleNamespace

    from spio_amd.kernels import conv2d_gw8_kernel as ck

    for n, c, h, k in ((128, 1392, 9, 5), (100, 400, 14, 5), (37, 256, 7, 3)):
        params = Conv2dGw8Params(n=n, c=c, h=h, w=h, r=k, s=k, padding=k // 2)
        configs = [q for q in ck._get_configs(params, SimpleNamespace(multiprocessor_count=256)) if q.variant == "image"]
        geometries = [(q, ck.image_geometry(params, q, False)) for q in configs]
        assert all(g["WGBLKS"] * q.block_n_iters >= g["NBLKS"] for q, g in geometries)
        first, g = geometries[0]
        resident = max(1, min(ck.DEVICE_LDS_BYTES // g["LDS_BYTES"], 2048 // g["THREADS"]))
        shorter = ck.image_geometry(params, replace(first, block_n_iters=max(1, first.block_n_iters - 1)), False)
        assert g["NUM_BLOCKS"] <= 2 * 256 * resident
        assert first.block_n_iters == 1 or shorter["NUM_BLOCKS"] > g["NUM_BLOCKS"]


def test_balanced_blocks_and_runs_of_image_blocks():
    """Tiles cut an extent into as many blocks as the sizes asked for, nearly equal ones; runs of image blocks
    leave no workgroup with a share much shorter than another's."""
    from spio_amd.kernels.conv2d_gw8_wgrad_kernel import conv2d_gw8_wgrad_kernel_factory, image_block_runs
    from spio_amd.util.math import balanced

    assert balanced(57, (4, 14, 28, 57, 64)) == [4, 12, 19, 57] and balanced(56, (4, 14, 28)) == [4, 14, 28]
    for extent in range(1, 80):
        for size in range(1, extent + 1):
            (block,) = balanced(extent, (size,))
            assert block <= size and -(-extent // block) == -(-extent // size)
    for blocks in (1, 2, 5, 10, 63, 500):
        for tiles in (1, 32, 300):
            runs = image_block_runs(blocks, tiles, 256, (1, 2, 4, 8))
            assert 1 in runs or blocks == 1 and runs == [1]
            assert all(1 <= r <= 16 for r in runs)
    params = Conv2dGw8Params(n=20, c=1024, h=27, w=27, padding=2, r=5, s=5)
    first = conv2d_gw8_wgrad_kernel_factory.configs(params, ATTR)[0]
    images = first.block_n * first.block_n_iters
    assert -(-params.n // images) * images <= params.n + 2  # runs of 8 of two images: 16 and 4


def test_row_offsets_stay_within_32_bits():
    """Rows in the padding and slots without a row have offsets without signed overflow: an image of almost 2 GiB,
    where the rows a step or two behind it would overflow."""
    params = Conv2dGw8Params(n=1, c=8, h=32748, w=4096, padding=1, r=3, s=3)
    config = Conv2dGw8WgradConfig(groups=1, block_h=14, block_n=1, block_n_iters=1, prefetch=4, block_q=64)
    defines = dict(conv2d_gw8_wgrad_kernel_factory.get_kernel_spec(params, config, ATTR).defines, SPIO_KERNEL_NAME="k")
    source = read_source("conv2d_gw8_wgrad_mfma.hip") + """
    static_assert(!kRowDescriptors, "offsets from the first row of an image");
    constexpr int IDLE_ROW = kP + ROWS + BH;  // the row that a slot without a step asks for, behind the last block
    static_assert(IDLE_ROW * X_ROW_BYTES >= (1ll << 31), "a row behind the image overflows");
    static_assert(ROW_OFFSET(IDLE_ROW, X_ROW_BYTES) == (unsigned)(IDLE_ROW * X_ROW_BYTES));
    static_assert(ROW_OFFSET(-kPadY, X_ROW_BYTES) == (unsigned)(-kPadY * X_ROW_BYTES));
    // rows that exist: lanes with data stay below 2 GiB, lanes without above every descriptor
    static_assert(ROW_OFFSET(kH - 1, X_ROW_BYTES) == (kH - 1) * X_ROW_BYTES && NB * X_IMAGE_BYTES < (1ll << 31));
    static_assert((unsigned)OUT_OF_RANGE + ROW_OFFSET(kH - 1, X_ROW_BYTES) >= (1u << 31));
    """
    assert compile_hip(source, "row_offsets.hip", headers=kernel_headers(), defines=defines)


@pytest.mark.parametrize("groups,prefetch,iters", [(4, 4, 1), (4, 4, 2)])
def test_weight_gradient_of_whole_images_keeps_its_sums_in_registers(groups, prefetch, iters):
    """Unrolled over 56 rows the step loop is long; left rolled it indexes the sums in memory."""
    params = Conv2dGw8Params(n=64, c=96, h=56, w=56, padding=2, r=5, s=5, has_bias=True)
    config = Conv2dGw8WgradConfig(groups=groups, block_h=56, prefetch=prefetch, block_n_iters=iters)
    assert scratch_bytes(conv2d_gw8_wgrad_kernel_factory, params, config) == 0


@pytest.mark.parametrize("config,kernel_size", [
    (Conv2dGw8WgradConfig(groups=4, block_h=56, prefetch=2, two_stage=1), 7),
    (Conv2dGw8WgradConfig(groups=8, block_h=56, block_n=2, prefetch=2), 3),
    (Conv2dGw8Config(groups=8, block_p=56, block_n=2, prefetch=8), 3),
])  # fmt: skip
def test_long_loops_are_unrolled(config, kernel_size):
    factory = conv2d_gw8_kernel_factory if isinstance(config, Conv2dGw8Config) else conv2d_gw8_wgrad_kernel_factory
    params = Conv2dGw8Params(n=64, c=64 if kernel_size == 3 else 96, h=56, w=56, padding=kernel_size // 2,
                             r=kernel_size, s=kernel_size, has_bias=True)  # fmt: skip
    assert scratch_bytes(factory, params, config) == 0


def test_chunks_of_twelve_steps_are_unrolled():
    """Left rolled they index the accumulators, 720 bytes a lane, in memory; unrolled a few registers are short."""
    params = Conv2dGw8Params.decode("62n_56c_46h_46w_2py_2px_5r_5s_b")
    config = Conv2dGw8BgradConfig(groups=4, split=2, prefetch=4)
    assert scratch_bytes(conv2d_gw8_bgrad_kernel_factory, params, config) <= 96


@pytest.mark.parametrize("shape,family,mode", [
    ("32n_64c_112h_112w_2py_2px_5r_5s_b", "fprop", {}),
    ("64n_96c_56h_56w_3py_3px_7r_7s_b", "fprop", {}),
    ("64n_96c_56h_56w_3py_3px_7r_7s_b", "fprop", {"igrad": True}),
    ("128n_1392c_9h_9w_2py_2px_5r_5s_nb", "wgrad", {}),
    ("64n_96c_56h_56w_3py_3px_7r_7s_b", "wgrad", {}),
    ("128n_1392c_9h_9w_2py_2px_5r_5s_nb", "bgrad", {}),
], ids=str)  # fmt: skip
def test_the_first_candidates_fit_the_registers(shape, family, mode):
    """The eight that a first use tries: all but a few of their registers (bytes a lane of memory) are registers."""
    factory = {"fprop": conv2d_gw8_kernel_factory, "wgrad": conv2d_gw8_wgrad_kernel_factory,
               "bgrad": conv2d_gw8_bgrad_kernel_factory}[family]  # fmt: skip
    params = Conv2dGw8Params.decode(shape)
    for config in factory.configs(params, ATTR, **mode)[:8]:
        assert scratch_bytes(factory, params, config, **mode) <= (140 if family == "bgrad" else 100), config


def test_weight_gradient_candidates_of_few_groups_are_not_all_split():
    """Three waves are fewer than a compute unit has SIMDs, and still the fastest (128n 24c 144x144)."""
    params = Conv2dGw8Params.decode("128n_24c_144h_144w_1py_1px_3r_3s_nb")
    assert any(c.split == 1 for c in conv2d_gw8_wgrad_kernel_factory.configs(params, ATTR)[:8])


@pytest.mark.parametrize("groups", [9, 13, 19, 25, 53, 71])
def test_capped_sweeps_try_every_number_of_groups_where_lines_are_shared(groups):
    """Pixels that are not whole lines: among the first eight row-streaming geometries is one of every block of groups
    that is offered, up to sixteen groups, blocks of one size among them; where a pixel is whole lines there are no others
    than 4, 8, 16 and all."""
    from spio_amd.kernels.tuner import _leading

    def row_streaming(c):
        configs = list(conv2d_gw8_kernel_factory.configs(Conv2dGw8Params(n=16, c=c, h=40, w=40, padding=1), DeviceAttributes()))
        return [cfg for cfg in configs if cfg.variant == "mfma"]

    configs = row_streaming(8 * groups)
    first = configs[:_leading(configs, 8)]
    even = {-(-groups // -(-groups // most)) for most in (12, 16)}
    assert even <= {cfg.groups for cfg in configs}
    assert {cfg.groups for cfg in configs} - {16} <= {cfg.groups for cfg in first}
    assert {cfg.groups for cfg in row_streaming(8 * 24)} <= {4, 8, 16, 24}



@pytest.mark.parametrize("groups", [1, 2, 3, 4, 5, 7, 8, 11, 12, 15])
def test_a_tile_stages_its_pixels_in_different_banks(groups):
    """16 lanes store 8 bytes each for as many pixels of a finished row: their 16-byte columns of the 256 bytes that the
    banks span are all different, in both kernels whose lanes all convert."""
    params = Conv2dGw8Params(n=2, c=8 * groups, h=9, w=40)
    for source, factory, config in (
        ("conv2d_gw8_mfma.hip", conv2d_gw8_kernel_factory, Conv2dGw8Config(groups=groups, block_p=4, prefetch=2)),
        ("conv2d_gw8_bgrad_mfma.hip", conv2d_gw8_bgrad_kernel_factory, Conv2dGw8BgradConfig(groups=groups, block_h=4, prefetch=2)),
    ):
        spec = factory.get_kernel_spec(params, config, ATTR)
        pixels = """
        constexpr bool distinct() {
            bool taken[16] = {};
            for (int i = 0; i < 16; ++i) {
                if (taken[i * OSTRIDE / 16 % 16]) return false;
                taken[i * OSTRIDE / 16 % 16] = true;
            }
            return OSTRIDE % 16 == 0 && OSTRIDE > GB * 16;
        }
        static_assert(distinct());
        """ + f"static_assert(LDS_UNITS * 16 == {spec.notes['LDS_BYTES']});"
        assert compile_hip(read_source(source) + pixels, source, headers=kernel_headers(), defines=dict(spec.defines, SPIO_KERNEL_NAME="k"))



@pytest.mark.parametrize("shape", ["3n_24c_9h_32w_1py_1px_3r_3s_nb", "2n_64c_9h_64w_3py_3px_7r_7s_b"])
@pytest.mark.parametrize("igrad", [False, True])
def test_rows_of_whole_tiles_have_no_slack_cells(shape, igrad):
    """Where the pixels that fragment reads touch end with the row there is nothing behind it to zero, and nothing divides
    by how many cells that is."""
    params = Conv2dGw8Params.decode(shape)
    spec = conv2d_gw8_kernel_factory.get_kernel_spec(params, Conv2dGw8Config(groups=3, block_p=4), ATTR, igrad=igrad)
    source = read_source("conv2d_gw8_mfma.hip") + "static_assert(FP == F);"
    assert compile_hip(source, "slack.hip", headers=kernel_headers(), defines=dict(spec.defines, SPIO_KERNEL_NAME="k"),
                       extra_options=["-Werror=division-by-zero"])  # fmt: skip



@pytest.mark.parametrize("megabytes", [0.1, 4, 8, 13, 25.7, 38.6, 77, 150, 500, 1023, 1024, 20000])
def test_sweeps_time_from_memory(megabytes):
    """Launches rotate over four times the memory-side cache, whatever the size of a set (very small ones excepted), and
    over no more than one set beyond that."""
    from spio_amd.kernels.tuner import _rotation_sets

    size, cache = int(megabytes * 2**20), 256 * 2**20
    sets = _rotation_sets(size)
    assert 1 <= sets <= 128
    assert sets * size >= 4 * cache or sets == 128 and megabytes < 8
    assert (sets - 1) * size < 4 * cache



@pytest.mark.parametrize("igrad", [False, True])
@pytest.mark.parametrize("filter_size", [3, 5, 7])
@pytest.mark.parametrize("n,c,hw", [(60, 216, 56), (16, 72, 112), (4, 424, 84), (16, 200, 33), (64, 104, 28), (8, 600, 49)])
def test_capped_sweeps_leave_out_what_keeps_registers_in_memory(n, c, hw, filter_size, igrad):
    """Also where the best geometry of every number of groups comes first: a number of groups whose registers do not fit
    has none there."""
    from spio_amd.kernels.conv2d_gw8_kernel import _mfma_fits
    from spio_amd.kernels.tuner import _leading

    params = Conv2dGw8Params(n=n, c=c, h=hw, w=hw, r=filter_size, s=filter_size, padding=filter_size // 2)
    configs = list(conv2d_gw8_kernel_factory.configs(params, DeviceAttributes(), igrad=igrad))
    rows = [cfg for cfg in configs if cfg.variant == "mfma"]
    assert len({replace(cfg, prefetch=0) for cfg in rows if _mfma_fits(params, cfg, igrad)}) >= 8
    first = configs[:_leading(configs, 8)]
    assert all(_mfma_fits(params, cfg, igrad) for cfg in first if cfg.variant == "mfma")



@pytest.mark.parametrize("two_stage,fused", [((False, False), True), ((False, True), False), ((True, True), True), ((True, False), True)])
def test_the_launch_that_clears_the_sums_counts_in_the_choice_of_backward_kernels(two_stage, fused, monkeypatch):
    """Recorded times hold both stages of a kernel that stores its sums, and not the launch before one that adds them."""
    import types

    import torch

    from spio_amd.functional import conv2d_gw8_function as op

    times = {"bgrad": 43.7, "dgrad": 19.3, "wgrad": 22.6}  # less than 2.2 us apart with the launch between the two

    class Factory:
        def __init__(self, name, overwrites=False):
            self.name, self.overwrites = name, overwrites

        def configs(self, *_args):
            return [None]

        def get_kernel(self, *_args, **_kw):
            return types.SimpleNamespace(kernel_spec=types.SimpleNamespace(overwrites_output=self.overwrites), name=self.name)

        def get_full_kernel_name(self, _params, **_kw):
            return self.name

    monkeypatch.setenv("SPIO_FUSED_BACKWARD", "auto")
    monkeypatch.setattr(op, "get_device_attributes", lambda _ordinal: ATTR)
    monkeypatch.setattr(op, "conv2d_gw8_bgrad_kernel_factory", Factory("bgrad", two_stage[0]))
    monkeypatch.setattr(op, "conv2d_gw8_kernel_factory", Factory("dgrad"))
    monkeypatch.setattr(op, "conv2d_gw8_wgrad_kernel_factory", Factory("wgrad", two_stage[1]))
    monkeypatch.setattr(op.tuner, "lookup", lambda _attr, name: {"us": times[name]})
    monkeypatch.setattr(op, "_fused_choice", {})
    params = Conv2dGw8Params(n=128, c=1392, h=9, w=9, r=5, s=5, padding=2)
    chosen = op.fused_backward_kernel(params, torch.device("cuda", 0))
    assert (chosen is not None) == fused


def test_finalists_of_a_sweep_are_timed_in_turn(tmp_path, monkeypatch):
    """A device that is slow for a while after the first pass: the leader, timed first, does not bear it alone."""
    import sys
    import types

    module = sys.modules[Tuner.__module__]
    timings = []

    class FakeKernel:
        kernel_name, code = "k__x", b""

        def __init__(self, groups, us):
            self.config, self.us = Conv2dGw8Config(groups=groups), us

        def load(self, **_kw):
            pass

        def unload(self):
            pass

        def time(self, _sets, warmup, iters):
            timings.append(self.us * (1.06 if 2 <= len(timings) < 7 else 1.0))  # (two are the first pass)
            return 1e-3 * timings[-1]

    kernels = [FakeKernel(4, 10.0), FakeKernel(8, 10.4)]
    monkeypatch.setattr(module, "compile_kernel_configs", lambda *_a, **_kw: kernels)
    monkeypatch.setattr(module, "_rotation_sets", lambda _bytes: 1, raising=False)
    monkeypatch.setattr(Tuner, "_first_valid", lambda _self, _f, _p, timed, *_a: timed[0])
    factory = types.SimpleNamespace(get_full_kernel_name=lambda *_a, **_kw: "k__x", make_test_args=lambda *_a, **_kw: ())
    record = str(tmp_path / "db.json")
    best = Tuner().sweep(factory, None, 0, ATTR, configs=[k.config for k in kernels], record_path=record)
    assert best.config.groups == 4 and json.load(open(record))["k__x"]["us"] == pytest.approx(10.0)


@pytest.mark.parametrize("n,c,h,w,filter_size", [(32, 64, 224, 224, 3), (16, 64, 128, 512, 3), (8, 64, 64, 1024, 3), (4, 96, 100, 300, 5)])
def test_wide_rows_get_column_blocks_of_whole_chunks(n, c, h, w, filter_size):
    """Among the first configurations are column blocks that take the weight gradient no more 32-pixel chunks than the data
    gradient 32-pixel tiles; a block is one column narrower only where rows are split."""
    from spio_amd.kernels.conv2d_gw8_bgrad_kernel import bgrad_geometry

    params = Conv2dGw8Params(n=n, c=c, h=h, w=w, r=filter_size, s=filter_size, padding=filter_size // 2)
    first = list(conv2d_gw8_bgrad_kernel_factory.configs(params, ATTR))[:8]
    geometries = [bgrad_geometry(params, cfg) for cfg in first if cfg.block_q]
    assert any(g["KC"] <= g["WT"] for g in geometries)
    narrow = next(cfg for cfg in first if cfg.narrow)
    g = bgrad_geometry(params, narrow)
    assert g["BQ"] == narrow.block_q - 1 and g["QBLKS"] * g["BQ"] >= w > (g["QBLKS"] - 1) * g["BQ"]
    assert conv2d_gw8_bgrad_kernel_factory.get_kernel_spec(params, narrow, ATTR).defines["SPIO_BQ"] == g["BQ"]
    for other in (replace(narrow, block_q=0), replace(narrow, narrow=2), replace(narrow, narrow=-1)):
        assert not conv2d_gw8_bgrad_kernel_factory.is_legal(params, other)


@pytest.mark.parametrize("fitting", [1, 2, 3, 9, 40])
def test_sweeps_leave_memory_where_little_is_left(fitting, tmp_path, monkeypatch):
    """Where fewer sets fit than a sweep rotates over it does with half of them: kernels allocate workspaces while they are
    timed.  The check of the winner comes when all but the first are given back."""
    import sys
    import types
    import weakref

    import torch

    module = sys.modules[Tuner.__module__]
    live, seen = weakref.WeakSet(), []

    class FakeTensor:
        def numel(self):
            return 10**6

        def element_size(self):
            return 1

    class FakeKernel:
        kernel_name, code, config = "k__x", b"", Conv2dGw8Config(groups=4)

        def load(self, **_kw):
            pass

        def unload(self):
            pass

        def time(self, sets, warmup, iters):
            seen.append((len(sets), len(live)))
            return 1e-3

    def make_test_args(*_args, **_kw):
        if len(live) == fitting:
            raise torch.OutOfMemoryError
        tensor = FakeTensor()
        live.add(tensor)
        return (tensor,)

    def first_valid(_self, _factory, _params, timed, *_args):
        seen.append((1, len(live)))
        return timed[0]

    monkeypatch.setattr(module, "compile_kernel_configs", lambda *_a, **_kw: [FakeKernel()])
    monkeypatch.setattr(Tuner, "_first_valid", first_valid)
    factory = types.SimpleNamespace(get_full_kernel_name=lambda *_a, **_kw: "k__x", make_test_args=make_test_args)
    Tuner().sweep(factory, None, 0, ATTR, configs=[FakeKernel.config], record_path=str(tmp_path / "db.json"))
    assert seen == [(max(1, fitting // 2),) * 2, (1, 1)]


@pytest.mark.parametrize("sets,workspace,free,expected", [(4, 1000, 100, 4), (128, 10**6, 10**9, 128), (128, 20 << 20, 10**9, 52),
                                                          (8, 3 << 30, 10**9, 1), (128, 20 << 20, 5, 5), (3, 1000, 0, None)])  # fmt: skip
def test_timed_two_stage_kernels_share_workspaces(sets, workspace, free, expected, monkeypatch):
    """One for each set of arguments up to 1 GB together, or as many as there is memory for: one at least."""
    import sys
    import types

    import torch

    params = Conv2dGw8Params(n=4, c=16, h=14, w=14)
    config = Conv2dGw8WgradConfig(groups=2, block_h=14, prefetch=2, two_stage=1)
    kernel = conv2d_gw8_wgrad_kernel_factory.make_kernel(params, config=config, device_attr=ATTR)
    module = sys.modules[type(kernel).__module__]
    kernel.function = kernel.epilogue_function = object()
    kernel.kernel_spec = replace(kernel.kernel_spec, workspace_bytes=workspace)
    made, launched = [], []

    def make_workspace(_self, _device):
        if len(made) == free:
            raise torch.OutOfMemoryError
        made.append(object())
        return made[-1]

    monkeypatch.setattr(type(kernel), "_workspace", make_workspace)
    monkeypatch.setattr(type(kernel), "_prepare", lambda _self, _args: None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda _device: types.SimpleNamespace(cuda_stream=0))
    monkeypatch.setattr(module, "launch_sequence_timed", lambda s, *_args: launched.extend(s) or 1.0)
    args = [("grad_weight%d" % i, "x", "grad_output") for i in range(sets)]
    if expected is None:
        with pytest.raises(torch.OutOfMemoryError):
            kernel.time(args)
        return
    assert kernel.time(args) == 1.0
    assert len(made) == expected and len(launched) == sets
    for i, ((*_, main), (*_, second)) in enumerate(launched):
        assert made[i % expected] in main and made[i % expected] in second and args[i][0] in second
