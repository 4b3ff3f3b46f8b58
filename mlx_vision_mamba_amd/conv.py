"""Causal depthwise conv1d + SiLU along scan orders, on the GPU.

Replaces MambaBlock's ``conv1d`` + ``[:, :L]`` + ``silu``
(reference mamba_block.py:129-132, :170-171) for all K directions of a
block at once: x is (B, N, K, D) in token order and position s of direction
k reads token row ``seq_to_tok[k, s]``, so no permuted copy is built.
"""

from __future__ import annotations

import torch

from . import _lib


def _conv_silu(x, weight, bias, tok):
    return _lib.native().conv_silu(x, weight, bias, tok)


def causal_conv_silu(x, weight, bias, seq_to_tok=None):
    """silu(causal depthwise conv) per direction.

    x: (B, N, K, D) float32 (channel stride 1, any other strides);
    weight: (K, D, d_conv); bias: (K, D); seq_to_tok: (K, N) int32 GPU
    tensor or None (identity order).  Returns (B, N, K, D) contiguous.
    """
    if weight.dim() != 3 or weight.shape[:2] != (x.shape[2], x.shape[3]):
        raise ValueError(f"weight must be (K, D, d_conv); got {tuple(weight.shape)}")
    if bias.shape != (x.shape[2], x.shape[3]):
        raise ValueError(f"bias must be (K, D); got {tuple(bias.shape)}")
    if seq_to_tok is not None:
        if seq_to_tok.dtype != torch.int32 or seq_to_tok.shape != (x.shape[2], x.shape[1]):
            raise ValueError("seq_to_tok must be int32 of shape (K, N)")
        seq_to_tok = seq_to_tok.to(x.device).contiguous()
    if _lib.is_tracing():
        return _lib.traced(_conv_silu, x, weight, bias, seq_to_tok)
    return _conv_silu(x, weight, bias, seq_to_tok)
