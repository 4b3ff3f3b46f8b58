"""Selective scan on MI355X: the scan entry points over the HIP C ABI (their
autograd Function and launches are in csrc/torch_ext.cpp).

Drop-in for the reference's scan entry points (paths relative to the
reference repository root):

* ``selective_scan(x, delta, A, B, C, D) -> y``   mamba_block.py:20-74
* ``selective_scan_chunked`` / ``selective_scan_parallel``   mamba_fast.py:17, :165
* ``selective_scan_metal`` (forward only, no autograd)       mamba_metal.py:230
* ``selective_scan_metal_trainable``                         mamba_metal.py:275
* ``selective_scan_metal_fused``                             mamba_metal_fused.py:253

All of them compute the same function with the same six gradients; they run
the HIP kernels of libmvm_scan.so and differ only in how the sequence is cut
into time chunks.  CPU tensors raise: there is no CPU fallback.

``selective_scan_directions`` is the index-remapped multi-direction form
used by the direction blocks: K scans over (B, L, K, D) token-order tensors,
where scan position s of direction k reads and writes token row
``seq_to_tok[k, s]`` (replacing the permuted copies of
mamba_block.py:254-338, :443-533).
"""

from __future__ import annotations

import ctypes

import torch

from . import _lib

_DT_CODE = {torch.float32: _lib.MVM_F32, torch.bfloat16: _lib.MVM_BF16}

#: scan_mode names accepted by MambaBlock (mamba_block.py:104-122) plus "hip".
SCAN_MODES = ("sequential", "chunked", "parallel", "metal", "metal_train", "metal_fused", "hip")


# Optional per-call timing: when a list, every forward / backward launch
# appends (kind, start_event, end_event, algorithmic_bytes), the events being
# recorded on the stream the kernels run on.
_timing = None


def set_scan_timing(records):
    """Start (pass a list) or stop (pass None) recording scan launches."""
    global _timing
    _timing = records
    if records is None:
        _lib.native().set_timer(None, None)
    else:
        _lib.native().set_timer(_timer_start, _timer_stop)


def _timer_start():
    """(records, start event) when launch timing is on, else (None, None).
    The records list is read once per call, so a call that starts recording
    also finishes it."""
    rec = _timing
    if rec is None:
        return None, None
    ev = torch.cuda.Event(enable_timing=True)
    ev.record()
    return rec, ev


def _timer_stop(started, kind, nbytes):
    rec, ev0 = started
    if rec is not None:
        ev1 = torch.cuda.Event(enable_timing=True)
        ev1.record()
        rec.append((kind, ev0, ev1, nbytes))


def algorithmic_bytes(bsz, L, D, N, in_size, out_size, ndir=1):
    """Bytes a scan forward / VJP must move if every tensor is read or
    written exactly once: (forward, vjp).  delta, ddelta, A, dA, D, dD are
    float32; u, B, C, dy use in_size and y, du, dB, dC use out_size bytes.
    ``bsz`` counts (batch, direction) rows; A and D exist once per direction."""
    fwd = (bsz * L * D * (in_size + 4 + out_size) + bsz * L * N * 2 * in_size
           + ndir * (D * N * 4 + D * 4))
    vjp = (bsz * L * D * (in_size + 4 + in_size + out_size + 4)
           + bsz * L * N * (2 * in_size + 2 * out_size) + ndir * (D * N * 8 + D * 8))
    return fwd, vjp


def algorithmic_bytes_fused(bsz, L, D, N, ndir=1, gate=True, bias=True):
    """(forward, vjp) bytes of the fused form (float32): the plain scan's
    tensors (delta_raw / ddelta_raw in place of delta / ddelta) plus, with a
    gate, z and y_raw (written by the forward; read by the VJP, which also
    writes dz), plus the dt bias and its gradient."""
    fwd, vjp = algorithmic_bytes(bsz, L, D, N, 4, 4, ndir)
    if gate:
        fwd += bsz * L * D * (4 + 4)
        vjp += bsz * L * D * (4 + 4 + 4)
    if bias:
        fwd += ndir * D * 4
        vjp += ndir * D * 8
    return fwd, vjp


def _stream_ptr(device) -> int:
    return torch.cuda.current_stream(device).cuda_stream


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else ctypes.c_void_p(0)


def _make_desc(u, Bm, in_dt, out_dt, tok, chunk_len):
    bsz, L, K, D = u.shape
    N = Bm.shape[-1]
    d = _lib.ScanDesc()
    d.batch, d.seqlen, d.dim, d.dstate, d.ndir = bsz, L, D, N, K
    d.x_stride_b, d.x_stride_t, d.x_stride_k = u.stride(0), u.stride(1), u.stride(2)
    d.bc_stride_b, d.bc_stride_t, d.bc_stride_k = Bm.stride(0), Bm.stride(1), Bm.stride(2)
    d.seq_to_tok = tok.data_ptr() if tok is not None else None
    d.in_dtype = _DT_CODE[in_dt]
    d.out_dtype = _DT_CODE[out_dt]
    d.chunk_len = int(chunk_len)
    return d


def _resolve_chunk(L, chunk_len):
    """chunk_len: int >= 0 (0 = library heuristic) or 'whole' (one chunk)."""
    if chunk_len == "whole":
        return max(16, (L + 15) // 16 * 16)
    return int(chunk_len)


def scan_forward(u, delta, A, Bm, Cm, Dv, tok=None, chunk_len=0, out_dtype=None, save_ckpt=False):
    """Raw forward launch (no autograd).  Returns (y, ckpt or None).

    Shapes: u, delta (B,L,K,D); A (K,D,N); Bm, Cm (B,L,K,N); Dv (K,D);
    tok (K,L) int32 on the same device or None.
    """
    with torch.no_grad():
        return _lib.native().scan_forward(u, delta, A, Bm, Cm, Dv, tok, _resolve_chunk(u.shape[1], chunk_len),
                                          out_dtype, save_ckpt, False)


def scan_backward(u, delta, A, Bm, Cm, Dv, dy, ckpt=None, tok=None, chunk_len=0, out_dtype=None):
    """Raw VJP launch.  Returns float32/out-dtype (du, ddelta, dA, dB, dC, dD)."""
    with torch.no_grad():
        return tuple(_lib.native().scan_backward(u, delta, A, Bm, Cm, Dv, dy, ckpt, tok,
                                                 _resolve_chunk(u.shape[1], chunk_len), out_dtype))


# ------------------------------------------------------------- fused form

def scan_fused_forward(u, delta_raw, delta_bias, A, Bm, Cm, Dv, z, tok=None, chunk_len=0,
                       save=False, a_is_log=False):
    """y = scan(u, softplus(delta_raw + delta_bias), A, B, C, D) * silu(z)
    (mamba_block.py:180-190) in one launch sequence.  With ``a_is_log`` the
    A argument holds A_log and the kernels use A = -exp(A_log) (:184).

    u, delta_raw, z: (B, L, K, D) float32 views with channel stride 1 and any
    other strides (z may be None: no gate); delta_bias (K, D) or None;
    A (K, D, N); Bm, Cm (B, L, K, N) views; Dv (K, D).  Returns
    (y, y_raw, ckpt): y (B, L, K, D) contiguous; y_raw and ckpt are saved for
    the backward when ``save`` (else None).
    """
    return _lib.native().scan_fused_forward(u, delta_raw, delta_bias, A, Bm, Cm, Dv, z, tok,
                                            _resolve_chunk(u.shape[1], chunk_len), bool(save), bool(a_is_log))


def scan_fused_backward(u, delta_raw, delta_bias, A, Bm, Cm, Dv, z, y_raw, ckpt, dy, tok=None,
                        chunk_len=0, du=None, ddelta_raw=None, dB=None, dC=None, dz=None,
                        a_is_log=False):
    """VJP of scan_fused_forward for dy (gradient of the gated y).  With
    ``a_is_log`` (A holds A_log) the returned dA is the gradient with
    respect to A_log.

    Output views may be passed in (any strides with channel stride 1, e.g.
    slices of a larger gradient buffer); missing ones are allocated with
    the layout of their primal.  Returns (du, ddelta_raw, ddelta_bias, dA,
    dB, dC, dD, dz); ddelta_bias is None without a bias, dz None without a
    gate.
    """
    return _lib.native().scan_fused_backward(
        u, delta_raw, delta_bias, A, Bm, Cm, Dv, z, y_raw, ckpt, dy, tok, _resolve_chunk(u.shape[1], chunk_len),
        du, ddelta_raw, dB, dC, dz, bool(a_is_log))


def check_permutation_table(table):
    """Raises ValueError unless every row of the (K, L) table is a
    permutation of 0..L-1.  The kernels only clamp table entries into
    [0, L): a row that misses a token would leave that token's outputs
    unwritten and a repeated token would be written twice.  The check runs
    once per table tensor (and again after an in-place change)."""
    stamp = (table.data_ptr(), table._version)
    if getattr(table, "_mvm_perm_checked", None) == stamp:
        return
    K, L = table.shape
    ok = True
    if L > 0:
        srt = torch.sort(table.long(), dim=1).values
        ok = bool((srt == torch.arange(L, device=table.device)).all())
    if not ok:
        raise ValueError("seq_to_tok: every row must be a permutation of 0..L-1")
    table._mvm_perm_checked = stamp


def selective_scan_directions(u, delta, A, B, C, D, seq_to_tok=None, chunk_len=0, out_dtype=None,
                              forward_only=False):
    """K index-remapped scans in one launch.

    u, delta: (B, L, K, D) in token order; A: (K, D, N); B, C: (B, L, K, N);
    D: (K, D); seq_to_tok: (K, L) int32 tensor on the GPU (or None for the
    identity order).  Returns y (B, L, K, D) in token order.
    ``forward_only`` returns a detached y without saving checkpoints (the
    reference's inference-only ``metal`` mode).
    """
    if seq_to_tok is not None:
        if seq_to_tok.dtype != torch.int32 or seq_to_tok.shape != (u.shape[2], u.shape[1]):
            raise ValueError("seq_to_tok must be int32 of shape (K, L)")
        # checked on the caller's tensor, so that a table kept on the host is
        # checked once, not again for every fresh device copy
        check_permutation_table(seq_to_tok)
        seq_to_tok = seq_to_tok.to(u.device).contiguous()
    if forward_only:
        y, _ = scan_forward(u.detach(), delta.detach(), A.detach(), B.detach(), C.detach(),
                            D.detach(), seq_to_tok, _resolve_chunk(u.shape[1], chunk_len), out_dtype)
        return y
    return _apply_scan(u, delta, A, B, C, D, seq_to_tok, chunk_len, out_dtype, False)


def _apply_scan(*args):
    return _lib.traced(_scan, *args) if _lib.is_tracing() else _scan(*args)


def _scan(u, delta, A, B, C, D, tok, chunk_len, out_dtype, flat):
    return _lib.native().scan(u, delta, A, B, C, D, tok, _resolve_chunk(u.shape[1], chunk_len), out_dtype, flat)


def _scan3(x, delta, A, B, C, D, chunk_len, out_dtype=None):
    if x.dim() != 3:
        raise ValueError(f"x must be (B, L, D); got {tuple(x.shape)}")
    return _apply_scan(x, delta, A, B, C, D, None, chunk_len, out_dtype, True)


def selective_scan(x, delta, A, B, C, D, chunk_len=0, out_dtype=None):
    """Selective scan (S6), forward + VJP on the GPU.  mamba_block.py:20-74.

    x, delta: (B, L, D_inner); A: (D_inner, N); B, C: (B, L, N); D: (D_inner,).
    ``chunk_len`` = 0 lets the library cut long sequences into time chunks
    (two-pass carry); ``"whole"`` keeps one chunk per channel.
    """
    return _scan3(x, delta, A, B, C, D, chunk_len, out_dtype)


def selective_scan_sequential(x, delta, A, B, C, D):
    """Sequential in time: one chunk per channel (the ``sequential`` mode)."""
    return _scan3(x, delta, A, B, C, D, "whole")


def selective_scan_chunked(x, delta, A, B, C, D, chunk_size=32):
    """mamba_fast.py:17 ``chunked`` mode: time chunks of ``chunk_size``
    (rounded up to a multiple of 16) joined by the carry pass."""
    return _scan3(x, delta, A, B, C, D, max(16, (int(chunk_size) + 15) // 16 * 16))


def selective_scan_parallel(x, delta, A, B, C, D):
    """mamba_fast.py:165 ``parallel`` mode: chunk-parallel scan, chunk
    length chosen by the library."""
    return _scan3(x, delta, A, B, C, D, 0)


def selective_scan_metal(x, delta, A, B, C, D):
    """mamba_metal.py:230 ``metal`` mode: inference only, no autograd (the
    result is detached and no checkpoints are written)."""
    if x.dim() != 3:
        raise ValueError(f"x must be (B, L, D); got {tuple(x.shape)}")
    with torch.no_grad():
        return _lib.native().scan_forward(x, delta, A, B, C, D, None, 0, None, False, True)[0].detach()


def selective_scan_metal_trainable(x, delta, A, B, C, D):
    """mamba_metal.py:275 ``metal_train`` mode (same function and gradients)."""
    return _scan3(x, delta, A, B, C, D, 0)


def selective_scan_metal_fused(x, delta, A, B, C, D):
    """mamba_metal_fused.py:253 ``metal_fused`` mode."""
    return _scan3(x, delta, A, B, C, D, 0)


_MODE_FNS = {
    "sequential": selective_scan_sequential,
    "chunked": selective_scan_chunked,
    "parallel": selective_scan_parallel,
    "metal": selective_scan_metal,
    "metal_train": selective_scan_metal_trainable,
    "metal_fused": selective_scan_metal_fused,
    "hip": selective_scan,
}

# chunk_len used by the direction blocks for each mode
_MODE_CHUNK = {"sequential": "whole", "chunked": 32, "parallel": 0, "metal": 0,
               "metal_train": 0, "metal_fused": 0, "hip": 0}


def get_scan_fn(scan_mode: str):
    """Scan function for a scan_mode string (mamba_block.py:104-122).

    Unknown names raise ValueError (the reference silently fell back to the
    sequential scan, mamba_block.py:121-122).
    """
    try:
        return _MODE_FNS[scan_mode]
    except KeyError:
        raise ValueError(f"unknown scan_mode {scan_mode!r}; expected one of {SCAN_MODES}") from None


def chunk_len_for(rows, L, D, N=16, fused=False):
    """Time-chunk length the library picks for `rows` = batch x directions
    scans of length L over D channels (the whole sequence when it is one
    chunk); ``fused``: the one that the blocks pass to their fused scans."""
    d = _lib.ScanDesc()
    d.batch, d.seqlen, d.dim, d.dstate, d.ndir = rows, L, D, N, 1
    d.x_stride_b, d.x_stride_k, d.x_stride_t = L * D, 0, D
    d.bc_stride_b, d.bc_stride_k, d.bc_stride_t = L * N, 0, N
    d.in_dtype = d.out_dtype = _lib.MVM_F32
    if fused:
        return _lib.check(_lib.lib().mvm_scan_long_chunk_len(ctypes.byref(d)))
    return _lib.check(_lib.lib().mvm_scan_chunk_len(ctypes.byref(d)))


def mode_chunk_len(scan_mode: str):
    get_scan_fn(scan_mode)
    return _MODE_CHUNK[scan_mode]


def selftest_lanes(device="cuda"):
    """Runs the cross-lane layout check kernel; returns a (128,) float tensor."""
    out = torch.empty(128, dtype=torch.float32, device=device)
    with torch.cuda.device(out.device):
        _lib.check(_lib.lib().mvm_selftest_lanes(_ptr(out), ctypes.c_void_p(_stream_ptr(out.device))))
    return out
