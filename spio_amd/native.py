"""The operators' native call path: loading it, its launch plans, and when it stands aside.

`_native.so` (csrc/spio_torch.cpp) runs a call of `conv2d_gw8` or `layernorm_2d` on plain GPU tensors
without going through the Python definition of the operator, which costs several times what the
kernels take at ordinary sizes.  It asks `_make_plan` once per shape for the kernels to launch
(tuner, compiler and caches are the Python side's) and keeps the answer until `forget_plans()`.
Where the file cannot be built or loaded the Python definitions run every call.
Whoever wants to see or choose every launch (overlay caches, KernelParamsLogger, LaunchTimer)
holds a `Bypass` meanwhile: all calls then take the Python path.
"""

import importlib
import struct
import warnings

import torch
from torch._library.custom_ops import CustomOpDef

from .build import build_extension, extension_is_current

try:
    if not extension_is_current():
        build_extension()
    _native = importlib.import_module(f"{__package__}._native")
except (ImportError, OSError, RuntimeError) as error:
    _native = None
    warnings.warn(f"spio_amd._native could not be built or loaded; every call pays for the Python path: {error}",
                  RuntimeWarning, stacklevel=2)  # fmt: skip


def forget_plans():
    """Drop every launch plan (a kernel of one was unloaded, caches or choices cleared).  The kernels stay
    with their caches: graphs, queued work and other threads may still launch them."""
    if _native is not None:
        _native.forget()


class Bypass:
    """While one of these is held, the native path declines every call."""

    def __init__(self):
        self._held = _native is not None
        if self._held:
            _native.bypass(1)
            forget_plans()

    def release(self):
        """Let calls take the native path again (idempotent)."""
        if self._held:
            self._held = False
            _native.bypass(-1)

    __del__ = release


def _stage(function, launch_params):
    return [function.handle, *launch_params.grid, *launch_params.block, launch_params.shared_mem_bytes]


# bits of a key's mode: which tensors are float32 (results, source, weights), whether the kernel keeps what it
# rounds, and that the weights are float16 (and so is their gradient)
WIDE = 0 if _native is None else _native.WIDE
HALF_WEIGHT = 0 if _native is None else _native.HALF_WEIGHT
READ_F32 = 0 if _native is None else _native.READ_F32
WEIGHT_F32 = 0 if _native is None else _native.WEIGHT_F32
KEEP = 0 if _native is None else _native.KEEP


def _adapted(kernel, factory, params, device, mode, **kwargs):
    """`kernel` or the version of it for the caller's types, in the configuration chosen for the plain one (it
    reads and multiplies the same); None where that has no such version."""
    from . import kernels

    config = kernels.stored_sums(factory, params, kernel.config) if mode & HALF_WEIGHT else kernel.config
    if mode & WIDE:
        if not kernels.fits_float32_output(params, config):
            return None
        kwargs["out_f32"] = True
    if mode & (READ_F32 | WEIGHT_F32):
        if factory is kernels.conv2d_gw8_bgrad_kernel_factory:
            kwargs["src_f32"] = True
            if not kernels.bgrad_reads_float32(params, config):
                return None
        else:
            reads = dict(src_f32=bool(mode & READ_F32), w_f32=bool(mode & WEIGHT_F32), keep=bool(mode & KEEP))
            if not kernels.reads_float32(params, config, kwargs.get("igrad", False), **reads):
                return None
            kwargs.update(reads)
    if config == kernel.config and not mode & (WIDE | READ_F32 | WEIGHT_F32):
        return kernel
    adapted = factory.get_kernel_in_config(params, device, config, **kwargs)
    # Float32 rows and filters take twice the registers.  What then has to keep some in memory is slower than
    # conversions and the plain kernel: 64n 96c 56x56 5x5 by 16 waves, forward 124 us (144 bytes a lane) and 70 with
    # conversions, data gradient 107 (68) and 60; 117n 48c 39x39 7x7 57 (72) and 49; 49n 264c 34x34 55 (8) and 46; 24 of
    # 27 such versions were, the others 10 per cent faster.  (Not the fused backward: 57 (68) and 73 at 128n 64c
    # 56x56, 9 of 10 faster.)
    if "w_f32" in kwargs and adapted.scratch_bytes > kernel.scratch_bytes:
        return None
    return adapted


def _make_plan(values):
    """(stages, workspace bytes, overwrites, kernel) for a key of csrc/spio_torch.cpp; the plan owns the kernel."""
    from . import kernels
    from .functional.conv2d_gw8_function import fused_backward_kernel

    kind, ordinal = values[:2]
    device = torch.device("cuda", ordinal)
    if kind < 4:
        n, c, h, w, r, s, py, px, bias, mode = values[2:]
        params = kernels.Conv2dGw8Params(n=n, c=c, h=h, w=w, r=r, s=s, padding=(py, px), has_bias=bool(bias))
        params.validate()
        factory, direction = kernels.conv2d_gw8_kernel_factory, {"igrad": True} if kind == 1 else {}
        if kind == 3:
            factory = kernels.conv2d_gw8_bgrad_kernel_factory
            kernel = fused_backward_kernel(params, device)
        elif kind == 2:
            factory = kernels.conv2d_gw8_wgrad_kernel_factory
            kernel = factory.get_kernel(params, device)
        else:
            kernel = factory.get_kernel(params, device, **direction)
        if kernel is not None:
            kernel = _adapted(kernel, factory, params, device, mode, **direction)
    else:
        n, c, h, w, eps, weight, bias = values[2:9]
        params = kernels.LayerNorm2dParams(n=n, c=c, h=h, w=w, eps=struct.unpack("<d", struct.pack("<q", eps))[0],
                                           has_weight=bool(weight), has_bias=bool(bias))  # fmt: skip
        factory = kernels.layernorm_2d_kernel_factory if kind == 4 else kernels.layernorm_2d_bwd_kernel_factory
        kernel = factory.get_kernel(params, device)
    if kernel is None:
        return None
    kernel.in_plans = True
    spec = kernel.kernel_spec
    stages = [_stage(kernel.function, spec.launch_params)]
    if kernel.epilogue_function is not None:
        stages.append(_stage(kernel.epilogue_function, spec.epilogue_launch_params))
    if kernel.epilogue_half_function is not None:
        stages.append(_stage(kernel.epilogue_half_function, spec.epilogue_half_launch_params))
    return stages, spec.workspace_bytes, spec.overwrites_output, kernel


class NativeOp(CustomOpDef):
    """A custom operator whose plain calls take the native path."""

    def __call__(self, *args, **kwargs):
        if torch.compiler.is_compiling():  # the graph records the operator
            return self._opoverload(*args, **kwargs)
        result = self.native(*args, **kwargs)
        return super().__call__(*args, **kwargs) if result is NotImplemented else result


def adopt(op, native_name):
    """Give the custom operator `op` the native path `native_name`."""
    if _native is None:
        return
    op.__class__ = NativeOp
    op.native = getattr(_native, native_name)


def configure(backward_op, norm_gradients):
    """Switch the native path on; what its backward passes hand over to where they stand aside."""
    if _native is None:
        return
    _native.configure(_make_plan, backward_op, norm_gradients)
    _native.bypass(-1)
