"""The operators' native call path (csrc/spio_torch.cpp) against the Python definition of the same
operators: same results whatever is differentiated, laid out or cast, and it stands aside where a
tracer, a transform or a recorder has to see the call."""

import pytest
import torch

from helpers import scratch_bytes
from spio_amd import native
from spio_amd.functional import conv2d_gw8, layernorm_2d
from spio_amd.hip import get_device_attributes
from spio_amd.kernels import Conv2dGw8Config, Conv2dGw8Params, KernelParamsLogger, conv2d_gw8_kernel_factory
from spio_amd.kernels.tuner import config_to_dict, tuner

pytestmark = pytest.mark.gpu
CL = torch.channels_last


def _both(call, inputs):
    """Results and gradients of `call` on the native path and on the Python path."""
    results = []
    for python in (False, True):
        held = native.Bypass() if python else None
        before = native._native.plans()
        leaves = [t if t is None else t.detach().clone(memory_format=torch.preserve_format).requires_grad_(t.requires_grad)
                  for t in inputs]  # fmt: skip
        y = call(*leaves)
        wanted = [t for t in leaves if t is not None and t.requires_grad]
        torch.manual_seed(7)
        grads = torch.autograd.grad(y, wanted, torch.randn_like(y)) if wanted else ()
        results.append([y, *grads])
        assert (native._native.plans() == 0) if python else (native._native.plans() >= max(before, 1))
        if held is not None:
            held.release()
    return results


def _check(call, inputs, tol=2e-3):
    native_results, python_results = _both(call, inputs)
    for a, b in zip(native_results, python_results):
        assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
        torch.testing.assert_close(a.float(), b.float(), rtol=tol, atol=tol * float(b.detach().float().abs().max()))


def _conv_args(p, dtype=torch.float16, layout=CL, grads=(True, True, True), bias_dtype=torch.float32):
    torch.manual_seed(3)
    x = torch.randn(p.input_shape, device="cuda").to(dtype).contiguous(memory_format=layout)
    w = (torch.randn(p.weight_shape, device="cuda") * 0.1).to(dtype).contiguous(memory_format=layout)
    b = torch.randn(p.c, device="cuda").to(bias_dtype) if p.has_bias else None
    args = [x.requires_grad_(grads[0]), w.requires_grad_(grads[1]), b if b is None else b.requires_grad_(grads[2])]
    return args, lambda x, w, b: conv2d_gw8(x, w, b, padding_y=p.padding_h, padding_x=p.padding_w, groups=p.groups)


@pytest.mark.parametrize("grads", [(False,) * 3, (True,) * 3, (True, False, False), (False, True, False),
                                   (False, False, True), (False, True, True)])  # fmt: skip
@pytest.mark.parametrize("p", [Conv2dGw8Params(2, 64, 14, 14, has_bias=True), Conv2dGw8Params(3, 24, 9, 7, (0, 2), 5, 3)])
def test_conv_matches_the_python_operator(p, grads):
    args, call = _conv_args(p, grads=grads)
    if not p.has_bias and grads == (False, False, True):
        return  # nothing is differentiated
    _check(call, args)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("layout", [CL, torch.contiguous_format])
def test_conv_under_autocast_and_in_any_layout(dtype, layout):
    args, call = _conv_args(Conv2dGw8Params(2, 40, 13, 11, has_bias=True), dtype, layout)

    def under_autocast(*a):
        with torch.autocast("cuda", dtype=torch.float16):
            return call(*a)

    _check(under_autocast, args)
    if dtype == torch.float16:
        _check(call, args)


@pytest.mark.parametrize("fused", ["0", "1"])
@pytest.mark.parametrize("p", [Conv2dGw8Params(2, 40, 13, 11, has_bias=True), Conv2dGw8Params(2, 16, 9, 9, 3),
                               Conv2dGw8Params(9, 64, 7, 7, 2, 5, 5)], ids=lambda p: p.encode())  # fmt: skip
def test_float32_tensors_that_kernels_read(p, fused, monkeypatch):
    """Under autocast the kernels read float32 tensors themselves: whichever of input and weight is float32 and
    wants a gradient, an input that is not 16-byte aligned, and one that is written to after the forward
    pass, which used a copy of it (weights likewise)."""
    monkeypatch.setenv("SPIO_FUSED_BACKWARD", fused)

    def check(args, call):
        def under_autocast(x, w, b):
            with torch.autocast("cuda", dtype=torch.float16):
                y = call(x, w, b)
            with torch.no_grad():
                for t in (x, w):
                    if t.dtype == torch.float32:
                        t.add_(1.0)
            return y

        _check(under_autocast, args)

    for grads in ((True,) * 3, (True, False, False), (False, True, True), (False, False, True), (False,) * 3):
        args, call = _conv_args(p, torch.float32, grads=grads)
        if any(t is not None and t.requires_grad for t in args) or not any(grads):
            check(args, call)
    args, call = _conv_args(p, torch.float32)
    check([args[0], args[1].detach().half().requires_grad_(), args[2]], call)
    check([args[0].detach().half().requires_grad_(), *args[1:]], call)
    storage = torch.randn(args[0].numel() + 1, device="cuda")
    shifted = storage[1:].as_strided(args[0].shape, args[0].stride())
    assert shifted.data_ptr() % 16 == 4
    with torch.autocast("cuda", dtype=torch.float16):
        y, expected = [call(t, args[1].detach(), args[2]) for t in (shifted, shifted.clone(memory_format=CL))]
    assert torch.equal(y, expected)


@pytest.mark.parametrize("weight,bias", [(True, True), (True, False), (False, True), (False, False)])
def test_norm_matches_the_python_operator(weight, bias):
    torch.manual_seed(5)
    x = torch.randn(3, 48, 6, 5, device="cuda", dtype=torch.float16).contiguous(memory_format=CL).requires_grad_()
    w = torch.randn(48, device="cuda").requires_grad_() if weight else None
    b = torch.randn(48, device="cuda").requires_grad_() if bias else None
    _check(lambda x, w, b: layernorm_2d(x, w, b, 1e-5), [x, w, b])


def test_float32_is_converted_where_a_version_that_reads_it_is_short_of_registers(tmp_path, monkeypatch):
    """In a configuration of 16 waves whose float16 kernel fits the registers and whose float32 one does not."""
    monkeypatch.setenv("SPIO_TUNE_DB", str(tmp_path / "db.json"))
    factory, config = conv2d_gw8_kernel_factory, Conv2dGw8Config(groups=4, block_p=14, split=4, prefetch=10)
    p = Conv2dGw8Params(2, 64, 28, 56, padding=2, r=5, s=5, has_bias=True)
    tuner._store(get_device_attributes(0), factory.get_full_kernel_name(p), {"config": config_to_dict(config), "us": 1.0})
    reads = dict(out_f32=True, src_f32=True, w_f32=True, keep=True)
    for kwargs in ({}, reads):
        kernel = factory.get_kernel_in_config(p, torch.device("cuda", 0), config, **kwargs)
        assert kernel.scratch_bytes == scratch_bytes(factory, p, config, **kwargs)
        assert (kernel.scratch_bytes > 0) == bool(kwargs)
    args, call = _conv_args(p, torch.float32)

    def under_autocast(*a):
        with torch.autocast("cuda", dtype=torch.float16):
            return call(*a)

    assert factory.get_kernel(p, torch.device("cuda", 0)).config == config
    _check(under_autocast, args)


def test_gradients_accumulate_and_graphs_are_kept():
    args, call = _conv_args(Conv2dGw8Params(2, 16, 8, 8, has_bias=True))
    y = call(*args)
    dy = torch.randn_like(y)
    y.backward(dy, retain_graph=True)
    once = [t.grad.clone() for t in args]
    y.backward(dy)
    for t, g in zip(args, once):
        torch.testing.assert_close(t.grad.float(), 2 * g.float(), rtol=2e-3, atol=2e-3 * float(g.abs().max()))
    with pytest.raises(RuntimeError, match="second time"):
        y.backward(dy)


def test_it_stands_aside():
    args, call = _conv_args(Conv2dGw8Params(2, 16, 8, 8))
    expected = call(*args)
    compiled = torch.compile(lambda *a: call(*a) * 2, fullgraph=True)
    torch.testing.assert_close(compiled(*args), expected * 2)
    with KernelParamsLogger() as logger:
        call(*args)
    assert len(logger.get_logged_params()) == 1
    with pytest.raises(AssertionError):  # the operator's own checks
        conv2d_gw8(args[0].float(), args[1], None, padding_y=1, padding_x=1, groups=2)
    with pytest.raises(RuntimeError):  # no second derivatives
        y = call(*args)
        (g,) = torch.autograd.grad(y.float().square().sum(), args[0], create_graph=True)
        torch.autograd.grad(g.float().square().sum(), args[0])


@pytest.mark.parametrize("padding", [2**63 - 1, 2**62, 2**40])
@pytest.mark.parametrize("side", ["padding_y", "padding_x"])
def test_paddings_without_a_possible_output_are_refused(side, padding):
    """The Python operator raises when it allocates the output; a size that wraps around is never launched."""
    args, _ = _conv_args(Conv2dGw8Params(2, 16, 8, 8), grads=(False,) * 3)
    native.forget_plans()
    with pytest.raises((TypeError, RuntimeError)):
        conv2d_gw8(args[0], args[1], None, groups=2, **{side: padding})
    assert native._native.plans() == 0
