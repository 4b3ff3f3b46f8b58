"""The block's projections as float32 products on the bf16 matrix units (HIP
kernels behind include/mvm_gemm.h; their autograd Functions are in
csrc/torch_ext.cpp).

Replaces the reference's ``nn.Linear`` in_proj and out_proj
(mamba_block.py:125, :153, :165, :191) for all K directions of a block:

  in_proj   xz (M, K*2*Din) = h (M, E) @ W_in (K*2*Din, E)^T
  out_proj  out (M, E) = sum_k y[:, k] (M, Din) @ W_out[k] (E, Din)^T

The out_proj reads the K stacked weight matrices where they lie, as one
product over K*Din, and its weight gradient comes out in the same (K, E, Din)
layout, so no reordered copy of either is made.  ``batched`` runs the
direction-batched products of x_proj and dt_proj (:137-140, :174-180) and their
gradients.
"""

from __future__ import annotations

from . import _lib


def in_proj(h, W):
    """h (..., E) @ W (O, E)^T."""
    return _lib.native().in_proj(h, W)


def out_proj(y, W):
    """Sum over k of y (..., K, D)[k] @ W (K, E, D)[k]^T: (..., E)."""
    return _lib.native().out_proj(y, W)


def batched(A, B, out=None, ta=False, tb=False, accumulate=False, stream=False):
    """out[q] (+)= op(A[q]) @ op(B[q]) for float32 (batch, rows, cols) views;
    ta / tb transpose an operand.  The kernels take contiguous columns, and
    16-byte rows of an operand whose summed index is the contiguous one (from
    32 summed values up); for other operands, and for a ``stream`` product that
    reads 12 Mi values of A or more, torch computes it."""
    return _lib.native().batched(A, B, out, ta, tb, accumulate, stream)
