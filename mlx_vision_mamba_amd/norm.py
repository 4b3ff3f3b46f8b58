"""LayerNorm over the last axis on the GPU (HIP kernels behind include/mvm_norm.h).

Replaces the reference's ``nn.LayerNorm(d_model)`` (MLX, eps 1e-5, affine):
the pre-norm of ResidualMambaBlock / BidirectionalMambaBlock /
MultiDirectionalMambaBlock (reference mamba_block.py:201-205, :222-227,
:401, :548) and the encoder's final norm (vision_mamba.py:192, :223).  The
modules keep their ``nn.LayerNorm`` children (same parameters and state_dict
keys); only the computation runs here.

``layer_norm(x, norm, residual=True)`` also returns x itself as a second
output for the block's residual branch ``x + f(norm(x))``.  The gradient
that reaches x through that branch then arrives in this function's backward
together with the normalised branch's, and the backward kernel adds the two
in its store, so no separate accumulation pass runs.
"""

from __future__ import annotations

import torch

from . import _lib


def _norm(x, weight, bias, eps, residual):
    out = _lib.native().norm(x, weight, bias, eps, residual)
    return tuple(out) if residual else out[0]


class _LayerNormFn:
    """The LayerNorm's autograd Function (csrc/torch_ext.cpp)."""

    @staticmethod
    def apply(x, weight, bias, eps, residual):
        if _lib.is_tracing():
            return _lib.traced(_norm, x, weight, bias, eps, residual)
        return _norm(x, weight, bias, eps, residual)


def layer_norm(x, norm, residual=False):
    """``norm(x)`` for an ``nn.LayerNorm`` over the last axis, computed by the
    HIP kernels.  With ``residual=True`` returns ``(norm(x), x_alias)``;
    use ``x_alias`` (it is x) for the block's residual sum so that both
    gradients of x are combined by the norm's backward kernel."""
    if not isinstance(norm, torch.nn.LayerNorm):
        raise TypeError(f"layer_norm needs an nn.LayerNorm, got {type(norm).__name__}")
    if len(norm.normalized_shape) != 1 or not norm.elementwise_affine or norm.bias is None:
        raise ValueError("layer_norm supports an affine LayerNorm over the last axis with bias")
    return _LayerNormFn.apply(x, norm.weight, norm.bias, norm.eps, residual)
