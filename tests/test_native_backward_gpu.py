"""Gradients recorded by the operators' native call path (csrc/spio_torch.cpp): what they do when something
between the forward and the backward pass changes the saved tensors, asks for second derivatives or wants to see
the launches."""

import gc

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from spio_amd import native
from spio_amd.functional import conv2d_gw8, conv2d_gw8_backward_op, layernorm_2d, layernorm_2d_gradients
from spio_amd.kernels import KernelParamsLogger
from spio_amd.kernels.kernel import LaunchTimer

pytestmark = pytest.mark.gpu
CL = torch.channels_last


def _leaves(op, dtype=torch.float16, layout=CL, affine=True):
    """Leaves and a call of a small convolution ("conv", "autocast") or norm ("norm")."""
    torch.manual_seed(11)
    x = torch.randn(3, 24, 9, 7, device="cuda").to(dtype).contiguous(memory_format=layout).requires_grad_()
    if op == "norm":
        vectors = [torch.randn(24, device="cuda").requires_grad_() for _ in range(2 if affine else 0)]
        return [x, *vectors], lambda x, *v: layernorm_2d(x, *v, eps=1e-5) if v else layernorm_2d(x, eps=1e-5)
    w = (torch.randn(24, 8, 3, 3, device="cuda") * 0.1).to(dtype).contiguous(memory_format=layout).requires_grad_()
    b = [torch.randn(24, device="cuda").requires_grad_()] if affine else []

    def call(x, w, b=None):
        with torch.autocast("cuda", dtype=torch.float16, enabled=op == "autocast"):
            return conv2d_gw8(x, w, b, padding_y=1, padding_x=1, groups=3)

    return [x, w, *b], call


def _assert_near(got, expected, tol=2e-3):
    for a, e in zip(got, expected):
        assert a.dtype == e.dtype and a.shape == e.shape
        torch.testing.assert_close(a.float(), e.float(), rtol=tol, atol=tol * float(e.detach().float().abs().max()))


def _repack(t):
    return t.detach().clone(memory_format=torch.contiguous_format)


_HOOKS = {
    "relaid": lambda: torch.autograd.graph.saved_tensors_hooks(_repack, lambda t: t),
    "pinned": lambda: torch.autograd.graph.save_on_cpu(pin_memory=True),
    "transposed": lambda: torch.autograd.graph.saved_tensors_hooks(
        lambda t: t.detach().transpose(0, -1).contiguous(), lambda t: t.transpose(0, -1)),
}  # fmt: skip


@pytest.mark.parametrize("hooks", list(_HOOKS))
@pytest.mark.parametrize("op,dtype,fused", [("conv", torch.float16, "0"), ("conv", torch.float16, "1"),
                                            ("autocast", torch.float32, "0"), ("autocast", torch.float32, "1"),
                                            ("norm", torch.float16, "auto")])  # fmt: skip
def test_saved_tensors_may_come_back_in_another_layout(op, dtype, fused, hooks, monkeypatch):
    """Hooks on saved tensors keep values and sizes, not strides: the gradients are those without hooks."""
    monkeypatch.setenv("SPIO_FUSED_BACKWARD", fused)
    leaves, call = _leaves(op, dtype)
    plain = call(*leaves)
    dy = torch.randn_like(plain)
    expected = torch.autograd.grad(plain, leaves, dy)
    with _HOOKS[hooks]():
        y = call(*leaves)
    _assert_near(torch.autograd.grad(y, leaves, dy), expected)


def test_a_captured_graph_outlives_the_launch_plans():
    """A graph captured over a call on float32 activations replays whatever drops the plans meanwhile."""
    leaves, call = _leaves("autocast", torch.float32)
    dy = torch.randn(3, 24, 9, 7, device="cuda").contiguous(memory_format=CL)

    def step():
        y = call(*leaves)
        return [y.detach(), *torch.autograd.grad(y, leaves, dy)]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step()
    for seed in range(3):
        native.Bypass().release()
        native.forget_plans()
        gc.collect()
        torch.manual_seed(seed)
        with torch.no_grad():
            leaves[0].copy_(torch.randn(3, 24, 9, 7, device="cuda"))
        graph.replay()
        torch.cuda.synchronize()
        _assert_near(captured, step())


@pytest.mark.parametrize("op,dtype,layout,affine", [
    ("conv", torch.float16, CL, True), ("conv", torch.float16, torch.contiguous_format, True),
    ("autocast", torch.float32, CL, True), ("autocast", torch.float32, torch.contiguous_format, False),
    ("norm", torch.float16, CL, False), ("norm", torch.float16, torch.contiguous_format, False),
    ("norm", torch.float16, torch.contiguous_format, True),
])  # fmt: skip
def test_second_derivatives_are_refused(op, dtype, layout, affine):
    """A gradient made with create_graph=True depends on the inputs whatever was cast or laid out anew on the
    way, and differentiating it raises: a penalty on it is never dropped from a sum."""
    leaves, call = _leaves(op, dtype, layout, affine)
    for wanted in leaves:
        y = call(*leaves)
        (g,) = torch.autograd.grad(y.sum(), wanted, create_graph=True)  # a grad_output that needs no gradient
        assert g.requires_grad
        loss = g.float().square().sum() + y.float().sum()
        with pytest.raises(RuntimeError, match="autograd formula"):
            loss.backward(retain_graph=True)
        for leaf in leaves[: 2 if op == "norm" else 3]:  # no gradient of the norm depends on its bias
            with pytest.raises(RuntimeError, match="autograd formula"):
                loss.backward(inputs=[leaf], retain_graph=True)


@pytest.mark.parametrize("op,dtype", [("conv", torch.float16), ("autocast", torch.float32), ("norm", torch.float16)])
def test_backward_stands_aside(op, dtype):
    """A backward pass whose forward ran natively takes the Python operator where a timer, a logger or a
    dispatch mode was entered in between, with the same gradients."""
    leaves, call = _leaves(op, dtype)
    y = call(*leaves)
    dy = torch.randn_like(y)
    expected = torch.autograd.grad(y, leaves, dy, retain_graph=True)
    plans = native._native.plans()
    assert plans > 0

    with LaunchTimer() as timer:
        _assert_near(torch.autograd.grad(y, leaves, dy, retain_graph=True), expected)
    assert any("grad" in str(k) or "_bwd" in str(k) for k in timer.events)

    with KernelParamsLogger() as logger:
        _assert_near(torch.autograd.grad(y, leaves, dy, retain_graph=True), expected)
    assert logger.get_logged_params() and native._native.plans() == 0

    seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Mode():
        _assert_near(torch.autograd.grad(y, leaves, dy, retain_graph=True), expected)
    assert any("_backward" in f and f.startswith("spio") for f in seen)


@pytest.mark.parametrize("op,dtype", [("conv", torch.float16), ("autocast", torch.float32), ("norm", torch.float16)])
def test_batched_gradients(op, dtype):
    """Several gradients of one output at once, as jacobian(vectorize=True) asks for them."""
    leaves, call = _leaves(op, dtype)
    y = call(*leaves)
    dys = torch.randn(3, *y.shape, device="cuda", dtype=y.dtype)
    expected = [torch.stack(g) for g in zip(*[torch.autograd.grad(y, leaves, dy, retain_graph=True) for dy in dys])]
    _assert_near(torch.autograd.grad(y, leaves, dys, is_grads_batched=True), expected)


@pytest.mark.parametrize("op,dtype,layout,which", [
    ("conv", torch.float16, CL, 0), ("conv", torch.float16, torch.contiguous_format, 0),
    ("conv", torch.float16, torch.contiguous_format, 1), ("conv", torch.float16, CL, 2),
    ("autocast", torch.float16, torch.contiguous_format, 0), ("autocast", torch.float32, CL, 2),
    ("norm", torch.float16, torch.contiguous_format, 0), ("norm", torch.float16, CL, 1),
])  # fmt: skip
def test_saved_inputs_must_not_change(op, dtype, layout, which):
    """The operators save their own arguments: writing to one before the backward pass is an error, in any layout."""
    leaves, call = _leaves(op, dtype, layout)
    y = call(*leaves)
    with torch.no_grad():
        leaves[which].add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()


def test_norm_backward_choice_is_read_in_the_backward_pass(monkeypatch):
    """SPIO_LAYERNORM_BACKWARD=torch set behind the forward pass: no plan of the backward kernel is made, and
    the gradients can be differentiated, with the results of the Python operator."""
    leaves, call = _leaves("norm")
    y = call(*leaves)
    dy = torch.randn_like(y)
    expected = torch.autograd.grad(y, leaves, dy, retain_graph=True)
    native.forget_plans()
    monkeypatch.setenv("SPIO_LAYERNORM_BACKWARD", "torch")
    _assert_near(torch.autograd.grad(y, leaves, dy, retain_graph=True), expected)
    assert native._native.plans() == 0

    def second(y):
        (g,) = torch.autograd.grad(y, leaves[0], dy, create_graph=True)
        return torch.autograd.grad(g.float().square().sum(), leaves[:2])

    results = second(call(*leaves))
    held = native.Bypass()
    _assert_near(results, second(call(*leaves)))
    held.release()


@pytest.mark.parametrize("in_backward", [False, True])
def test_a_launch_that_fails_raises_value_error(in_backward):
    """The error of the kernels' Python launch; here the library refuses a plan without a function."""
    leaves, call = _leaves("conv")
    y = call(*leaves)
    native.forget_plans()
    native._native.configure(lambda values: ([[0, 1, 1, 1, 64, 1, 1, 0]], 0, False, None), conv2d_gw8_backward_op, None)
    try:
        with pytest.raises(ValueError, match="launch"):
            y.sum().backward() if in_backward else call(*leaves)
    finally:
        native.forget_plans()
        native._native.configure(native._make_plan, conv2d_gw8_backward_op, layernorm_2d_gradients)


def _profiled(op, dtype):
    """{operator: shapes of its tensor arguments} of a pass as torch's profiler sees it."""
    leaves, call = _leaves(op, dtype)
    y = call(*leaves)
    torch.autograd.grad(y, leaves, torch.randn_like(y))
    with torch.autograd.profiler.profile(record_shapes=True, use_device=None) as profile:
        y = call(*leaves)
        torch.autograd.grad(y, leaves, torch.randn_like(y))
    return {e.name: [s for s in e.input_shapes if s] for e in profile.function_events if e.name.startswith("spio::")}


@pytest.mark.parametrize("op,dtype", [("conv", torch.float16), ("autocast", torch.float32), ("norm", torch.float16)])
def test_profiles_show_the_operators(op, dtype):
    """Forward and backward operators appear under their names with the shapes of their tensors."""
    seen = _profiled(op, dtype)
    held = native.Bypass()
    expected = _profiled(op, dtype)
    held.release()
    assert len(expected) == 2 and seen == expected
