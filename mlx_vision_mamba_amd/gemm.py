"""The block's projections as float32 products on the bf16 matrix units (HIP
kernels behind include/mvm_gemm.h).

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

import ctypes

import torch
import torch.nn.functional as F

from . import _lib
from .scan import _ptr, _stream_ptr

_SEG = 32  # out_proj: Din is a multiple of this, or there is one direction


def _aligned(t):
    return t.data_ptr() % 16 == 0


def _launch(A, B, C, m, n, k, lda, ldb, ldc, a_km, b_km, batch=1, sa=0, sb=0, sc=0, seg=0, seg_stride=0,
            accumulate=False):
    d = _lib.GemmDesc(m, n, k, batch, lda, ldb, ldc, sa, sb, sc, seg, seg_stride, a_km, b_km,
                      int(accumulate), 0)
    lib = _lib.lib()
    dev = C.device
    with torch.cuda.device(dev):
        nbytes = _lib.check(lib.mvm_gemm_workspace_bytes(ctypes.byref(d)))
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev) if nbytes else None
        _lib.check(lib.mvm_gemm_f32(ctypes.byref(d), _ptr(A), _ptr(B), _ptr(C), _ptr(ws), nbytes,
                                    ctypes.c_void_p(_stream_ptr(dev))))


def _dense(g):
    """g with the layout and alignment the products take."""
    g = g.contiguous()
    return g if _aligned(g) else g.clone()


def _usable(x, W, *widths):
    """Whether the products take (x, W): float32 on the GPU outside autocast
    (whose casts F.linear applies), row lengths that are multiples of 4 (16-byte
    rows) and below the kernels' limit of 2^21, aligned weights."""
    return (x.is_cuda and x.device == W.device and x.dtype == torch.float32 and W.dtype == torch.float32
            and not torch.is_autocast_enabled("cuda") and W.is_contiguous() and _aligned(W)
            and all(w % 4 == 0 and 0 < w < 1 << 21 for w in widths))


class _InProjFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, h, W):
        O, E = W.shape
        h2 = _dense(h.reshape(-1, E))
        M = h2.shape[0]
        out = torch.empty((M, O), dtype=torch.float32, device=h.device)
        _launch(h2, W, out, M, O, E, E, E, O, 1, 1)
        ctx.save_for_backward(h2, W)
        ctx.hshape = h.shape
        return out.view(*h.shape[:-1], O)

    @staticmethod
    def backward(ctx, g):
        h2, W = ctx.saved_tensors
        O, E = W.shape
        M = h2.shape[0]
        g2 = _dense(g.reshape(M, O))
        dh = dW = None
        if ctx.needs_input_grad[0]:
            dh = torch.empty((M, E), dtype=torch.float32, device=g.device)
            _launch(g2, W, dh, M, E, O, O, E, E, 1, 0)
            dh = dh.view(ctx.hshape)
        if ctx.needs_input_grad[1]:
            dW = torch.empty((O, E), dtype=torch.float32, device=g.device)
            _launch(g2, h2, dW, O, E, M, O, E, E, 0, 0)
        return dh, dW


class _OutProjFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, y, W):
        K, E, D = W.shape
        y2 = _dense(y.reshape(-1, K * D))
        M = y2.shape[0]
        out = torch.empty((M, E), dtype=torch.float32, device=y.device)
        _launch(y2, W, out, M, E, K * D, K * D, D, E, 1, 1, seg=D if K > 1 else 0, seg_stride=E * D)
        ctx.save_for_backward(y2, W)
        ctx.yshape = y.shape
        return out.view(*y.shape[:-2], E)

    @staticmethod
    def backward(ctx, g):
        y2, W = ctx.saved_tensors
        K, E, D = W.shape
        M = y2.shape[0]
        g2 = _dense(g.reshape(M, E))
        dy = dW = None
        if ctx.needs_input_grad[0]:
            dy = torch.empty((M, K, D), dtype=torch.float32, device=g.device)
            _launch(g2, W, dy, M, D, E, E, D, K * D, 1, 0, batch=K, sb=E * D, sc=D)
            dy = dy.view(ctx.yshape)
        if ctx.needs_input_grad[1]:
            dW = torch.empty((K, E, D), dtype=torch.float32, device=g.device)
            _launch(g2, y2, dW, E, D, M, E, K * D, D, 0, 0, batch=K, sb=D, sc=E * D)
        return dy, dW


def in_proj(h, W):
    """h (..., E) @ W (O, E)^T."""
    O, E = W.shape
    if _usable(h, W, O, E):
        return _InProjFn.apply(h, W)
    return F.linear(h, W)


def out_proj(y, W):
    """Sum over k of y (..., K, D)[k] @ W (K, E, D)[k]^T: (..., E)."""
    K, E, D = W.shape
    if _usable(y, W, E, D, K * D) and (K == 1 or D % _SEG == 0):
        return _OutProjFn.apply(y, W)
    # one product over the concatenated directions (a reordered copy of W)
    return F.linear(y.reshape(*y.shape[:-2], K * D), W.permute(1, 0, 2).reshape(E, K * D))


# batch x rows from which dt_proj's two products over the rows (the delta_raw
# and its gradient's) are left to the BLAS library: they stream 77 MB at 4 x
# 6272 rows of 768 channels, with almost no arithmetic, and the library's picks
# take 25.6 and 22.3 us there, the kernels here 31.4 and 27.3; at 8 x 1024 rows
# it is 21 and 20 us against 12.1 and 13.7.
STREAM_ROWS = 16384


def _rowmajor(t):
    """Whether (batch, rows, cols) t has contiguous columns and 16-byte rows."""
    return (t.stride(2) == 1 and t.stride(1) % 4 == 0 and t.stride(0) % 4 == 0 and _aligned(t)
            and t.stride(1) < 1 << 21)


def batched(A, B, out=None, ta=False, tb=False, accumulate=False, stream=False):
    """out[q] (+)= op(A[q]) @ op(B[q]) for float32 (batch, rows, cols) views
    with contiguous columns; ta / tb transpose an operand.  An operand whose
    summed index is its contiguous one (A without ta, B with tb) needs 16-byte
    rows from 32 summed values up, and out columns that are contiguous; where
    the kernels do not take the operands, and for a ``stream`` product of many
    rows, torch computes it."""
    Av, Bv = (A.transpose(1, 2) if ta else A), (B.transpose(1, 2) if tb else B)
    q, m, k = Av.shape
    n = Bv.shape[2]
    if out is None:
        out = torch.empty((q, m, n), dtype=torch.float32, device=A.device)
    ok = (A.stride(2) == 1 and B.stride(2) == 1 and max(A.stride(1), B.stride(1)) < 1 << 21
          and (k < 32 or ((ta or _rowmajor(A)) and (not tb or _rowmajor(B))))
          and not (stream and q * m > STREAM_ROWS))
    if ok:
        _launch(A, B, out, m, n, k, A.stride(1), B.stride(1), out.stride(1), int(not ta), int(tb),
                batch=q, sa=A.stride(0), sb=B.stride(0), sc=out.stride(0), accumulate=accumulate)
        return out
    return out.baddbmm_(Av, Bv) if accumulate else torch.bmm(Av, Bv, out=out)
