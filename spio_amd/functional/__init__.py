"""Functional interface: the `spio::conv2d_gw8` custom operators."""

from .conv2d_gw8_function import (
    conv2d_gw8,
    conv2d_gw8_backward_op,
    fused_backward_kernel,
    reset_fused_backward_choices,
)
from .layernorm_2d_function import layernorm_2d, layernorm_2d_backward, layernorm_2d_gradients
from .. import native as _native_path

_native_path.adopt(conv2d_gw8, "conv2d_gw8")
_native_path.adopt(layernorm_2d, "layernorm_2d")
_native_path.configure(conv2d_gw8_backward_op, layernorm_2d_gradients)
