"""``mcoplib.custom_ops`` wrappers of the fused norm/quant path (reference
mcoplib/custom_ops.py:7-45): allocate the outputs the way the reference does and call the
``op`` entry point, both in the _torch_ops extension."""

from __future__ import annotations

from typing import Optional, Tuple

import torch

from . import op as ops  # noqa: F401  (loads the library, then the extension)
from . import _torch_ops


def fused_add_rms_norm_dynamic_per_token_quant_padding_output(
        input: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, pad_size: int,
        epsilon: float):
    """Allocates the padded output as bf16 [..., pad_size] (2*pad_size bytes per row, viewed as
    int8 for the kernel), output_rms like input, the unpacked int8 codes and scales [T, 1], and
    returns (output, residual, output_rms, output_quant_int8, scales); ``residual`` is updated
    in place (reference mcoplib/custom_ops.py:7-27)."""
    assert input.is_contiguous()
    assert weight.is_contiguous()
    return _torch_ops.padded_new(input, residual, weight, pad_size, epsilon)


def rms_norm_dynamic_per_token_quant(input: torch.Tensor, weight: torch.Tensor, epsilon: float,
                                     quant_dtype: torch.dtype,
                                     scale_ub: Optional[torch.Tensor] = None,
                                     residual: Optional[torch.Tensor] = None
                                     ) -> Tuple[torch.Tensor, torch.Tensor]:
    """Returns (codes like input in quant_dtype, scales [T, 1] fp32); updates ``residual`` in
    place when given.  ``quant_dtype`` must be int8, as for the reference custom op."""
    return _torch_ops.custom_new(input, weight, epsilon, quant_dtype, scale_ub, residual)
