"""Lifetime of the kernels that the native call path's launch plans point into.  CPU only: the kernels
are stand-ins that note when their code object would be unloaded."""

import gc
import threading

import pytest

from spio_amd import native
from spio_amd.hip import DeviceAttributes
from spio_amd.kernels import Conv2dGw8Config, KernelParamsLogger, KernelSpec, LaunchParams, conv2d_gw8_kernel_factory, kernel_cache
from spio_amd.kernels.kernel import Kernel, LaunchTimer

WIDE_FORWARD = (0, 0, 2, 64, 8, 8, 3, 3, 1, 1, 0, native.WIDE)  # a key: float32-storing forward kernel on device 0


class _Module:
    def __init__(self, loaded):
        self._loaded = loaded
        loaded.append(id(self))

    def unload(self):
        if id(self) in self._loaded:
            self._loaded.remove(id(self))

    __del__ = unload


class _Kernel(Kernel):
    """A loaded kernel whose module goes when nothing refers to it any more, as hip.driver.Module does."""

    def __init__(self, loaded):
        super().__init__("k", KernelSpec({}, LaunchParams(grid=1, block=64), "x.hip"), config=Conv2dGw8Config())
        self.module = _Module(loaded)
        self.function = type("Function", (), {"handle": 1})()


@pytest.fixture
def made(monkeypatch):
    """(kernels made, modules loaded) with compiling and loading replaced."""
    kernels, loaded = [], []

    def compile_and_load(factory, params, config, ordinal, device_attr, **kwargs):
        kernels.append(kwargs)
        return _Kernel(loaded)

    monkeypatch.setattr(kernel_cache, "compile_and_load_kernel", compile_and_load)
    monkeypatch.setattr(kernel_cache, "get_device_attributes", lambda ordinal: DeviceAttributes())
    monkeypatch.setattr("spio_amd.hip.driver.get_device_attributes", lambda ordinal: DeviceAttributes())
    monkeypatch.setattr(conv2d_gw8_kernel_factory, "_kernel_caches", {})
    monkeypatch.setenv("SPIO_TUNE", "0")
    yield kernels, loaded
    native.forget_plans()


def test_forgotten_plans_leave_their_kernels_loaded(made):
    """A HIP graph, a queued launch or another thread may still use a kernel whose plan is dropped."""
    kernels, loaded = made
    native._make_plan(WIDE_FORWARD)
    handed_out = list(loaded)
    assert len(handed_out) == 2  # the float16 kernel, in whose configuration the float32 one is made, and that
    native.forget_plans()
    native.Bypass().release()
    gc.collect()
    assert loaded == handed_out
    native._make_plan(WIDE_FORWARD)
    gc.collect()
    assert loaded == handed_out and len(kernels) == 2  # the same kernels again, nothing is compiled twice


def test_concurrent_plans_share_one_kernel(made):
    kernels, loaded = made
    threads = [threading.Thread(target=native._make_plan, args=(WIDE_FORWARD,)) for _ in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    gc.collect()
    assert len(kernels) == 2 and len(loaded) == 2


def test_a_plan_owns_its_kernel(made):
    """Clearing the kernel cache drops the plans, but not a kernel that a plan in use still holds."""
    _, loaded = made
    plan = native._make_plan(WIDE_FORWARD)
    conv2d_gw8_kernel_factory.get_kernel_cache().clear_cache()
    conv2d_gw8_kernel_factory.get_kernel_cache(out_f32=True).clear_cache()
    gc.collect()
    assert len(loaded) == 1 and id(plan[3].module) == loaded[0]


def test_unloading_a_kernel_outside_the_plans_forgets_none(made, monkeypatch):
    """A sweep unloads its candidates: the plan it is part of, and those of other shapes, stay."""
    _, loaded = made
    calls = []
    monkeypatch.setattr(native, "forget_plans", lambda: calls.append(1))
    _Kernel(loaded).unload()
    assert not calls
    native._make_plan(WIDE_FORWARD)[3].unload()
    assert calls


@pytest.mark.parametrize("recorder", [KernelParamsLogger, LaunchTimer])
def test_recorders_may_be_entered_again(recorder, monkeypatch):
    """One instance, inside itself: the native path stays off until the outer block ends."""
    held = []
    monkeypatch.setattr(native._native, "bypass", held.append)
    with recorder() as outer:
        with outer:
            assert sum(held) == 2
        assert sum(held) == 1
    assert sum(held) == 0


def test_versions_that_read_float32_with_registers_in_memory_are_not_used(made, monkeypatch):
    """They are slower than a conversion and the plain kernel, in whose configuration they run."""
    kernels, loaded = made
    spilled = []

    def compile_and_load(factory, params, config, ordinal, device_attr, **kwargs):
        kernel = _Kernel(loaded)
        kernel.scratch_bytes = 68 if kwargs.get("src_f32") or kwargs.get("w_f32") else 0
        spilled.append(kernel.scratch_bytes)
        return kernel

    monkeypatch.setattr(kernel_cache, "compile_and_load_kernel", compile_and_load)
    kind, device, *shape, mode = WIDE_FORWARD
    for reads in (native.READ_F32, native.WEIGHT_F32, native.READ_F32 | native.WEIGHT_F32 | native.KEEP):
        assert native._make_plan((kind, device, *shape, mode | reads)) is None
    assert spilled == [0, 68, 68, 68]  # the plain kernel, then a version each
    assert native._make_plan(WIDE_FORWARD) is not None
