"""Mamba blocks on MI355X (PyTorch modules over the HIP selective scan).

Mirrors the reference's module API (mlx_vision_mamba/mamba_block.py):
``MambaBlock`` (:77-192), ``ResidualMambaBlock`` (:195-205),
``BidirectionalMambaBlock`` (:208-237) and ``MultiDirectionalMambaBlock``
(:341-566), with the same constructor arguments, parameter names and
forward semantics, and with ``scan_mode`` passed down to every inner block
(the reference built the inner blocks with the default mode, :202, :223-224,
:403).

Direction blocks do not build permuted copies.  All K directions run as one
batch: one in_proj GEMM (E -> K*2*D_inner), a causal depthwise conv and the
selective scan that read and write through per-direction index tables, the
per-token projections batched over K, and one out_proj GEMM over the
concatenated K*D_inner features, which is also the (atomic-free) sum over
directions (:562-566).

Between the two GEMMs the block core (conv + SiLU, x_proj, dt_proj, and the
scan with the softplus of delta and the y * silu(z) gate fused into it,
:170-190) is one autograd Function whose backward writes the gradient of
the in_proj output in place: the conv's dx and the gate's dz land in the two
halves of one buffer, so no slice / cat / elementwise pass is materialised.
Activations between the projections are kept direction-major,
(K, B*N, features), so the x_proj / dt_proj GEMMs batch over K without
copies.

The direction blocks' per-direction parameters (in_proj, conv1d, x_proj,
dt_proj, A_log, D, out_proj) are slices of one (K, ...) buffer per kind owned
by the direction module, so the batched operands are views, not per-step
concatenations; each buffer's gradient returns to the K parameters as its K
slices.  The buffers are (re)built at the first forward and whenever a
parameter stops being its slice (after ``.to()``, or a replaced parameter).
"""

from __future__ import annotations

import math
from typing import Optional, Sequence

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _lib
from . import directions as _dirs
from .conv import causal_conv_silu
from .norm import layer_norm
from .scan import _resolve_chunk, check_permutation_table, get_scan_fn, mode_chunk_len


def _dt_bias_init(d_inner: int, dt_min: float = 1e-3, dt_max: float = 1e-1) -> torch.Tensor:
    """dt_proj bias with softplus(bias) log-uniform in [dt_min, dt_max]."""
    dt = torch.exp(torch.rand(d_inner) * (math.log(dt_max) - math.log(dt_min)) + math.log(dt_min))
    return dt + torch.log(-torch.expm1(-dt))


class MambaBlock(nn.Module):
    """in_proj -> causal depthwise conv1d -> SiLU -> selective scan -> gate ->
    out_proj (mamba_block.py:77-192).  Input / output (B, L, d_model).

    scan_mode: "sequential", "chunked", "parallel", "metal", "metal_train",
    "metal_fused" (the reference's names, mamba_block.py:104-120) or "hip";
    every mode runs the HIP scan.  Unknown names raise ValueError.

    ``self._scan_fn`` is the scan function the mode selects
    (mamba_block.py:104-122).  The library's modes run inside the fused
    block core; a caller that assigns another callable
    ``f(x, delta, A, B, C, D) -> y`` to ``_scan_fn`` gets the reference's op
    sequence with ``f`` called where the reference calls it (:187), in this
    block and in the direction blocks that contain it.
    """

    def __init__(self, d_model: int = 384, d_state: int = 16, d_conv: int = 4,
                 expand_factor: int = 2, scan_mode: str = "sequential"):
        super().__init__()
        self.d_model = d_model
        self.d_state = d_state
        self.d_inner = d_model * expand_factor
        self.d_conv = d_conv
        self.scan_mode = scan_mode
        self._scan_fn = get_scan_fn(scan_mode)
        self.dt_rank = math.ceil(d_model / 16)                                 # :136
        self.in_proj = nn.Linear(d_model, 2 * self.d_inner, bias=False)        # :125
        self.conv1d = nn.Conv1d(self.d_inner, self.d_inner, kernel_size=d_conv,
                                padding=d_conv - 1, groups=self.d_inner)        # :129-132
        self.x_proj = nn.Linear(self.d_inner, self.dt_rank + 2 * d_state, bias=False)  # :137
        self.dt_proj = nn.Linear(self.dt_rank, self.d_inner, bias=True)        # :140
        with torch.no_grad():
            self.dt_proj.bias.copy_(_dt_bias_init(self.d_inner))
        A = torch.arange(1, d_state + 1, dtype=torch.float32).repeat(self.d_inner, 1)
        self.A_log = nn.Parameter(torch.log(A))                                # :143-147
        self.D = nn.Parameter(torch.ones(self.d_inner))                        # :150
        self.out_proj = nn.Linear(self.d_inner, d_model, bias=False)           # :153

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if _custom_scan(self):
            return _scan_fn_forward(self, x)
        return _directional_forward([self], x, None, self.scan_mode)


class ResidualMambaBlock(nn.Module):
    """Pre-norm MambaBlock with a residual (mamba_block.py:195-205)."""

    def __init__(self, d_model: int = 384, d_state: int = 16, d_conv: int = 4,
                 expand_factor: int = 2, scan_mode: str = "sequential"):
        super().__init__()
        self.norm = nn.LayerNorm(d_model)
        self.mamba = MambaBlock(d_model, d_state, d_conv, expand_factor, scan_mode)

    def forward(self, x):
        h, xr = layer_norm(x, self.norm, residual=True)
        return xr + self.mamba(h)


class BidirectionalMambaBlock(nn.Module):
    """Forward + reversed-sequence MambaBlocks, summed with a residual
    (mamba_block.py:208-237)."""

    def __init__(self, d_model: int = 384, d_state: int = 16, d_conv: int = 4,
                 expand_factor: int = 2, scan_mode: str = "sequential"):
        super().__init__()
        self.norm = nn.LayerNorm(d_model)
        self.forward_mamba = MambaBlock(d_model, d_state, d_conv, expand_factor, scan_mode)
        self.backward_mamba = MambaBlock(d_model, d_state, d_conv, expand_factor, scan_mode)
        self.scan_mode = scan_mode
        self._tables = {}

    def forward(self, x):
        h, xr = layer_norm(x, self.norm, residual=True)                      # :227
        tok = _cached_table(self._tables, 2, x.shape[1], None, x.device)
        blocks = [self.forward_mamba, self.backward_mamba]
        if any(_custom_scan(b) for b in blocks):
            return xr + _per_direction_forward(blocks, h, tok)
        return _directional_forward(blocks, h, tok, self.scan_mode, self, blocks, residual=xr)


class MultiDirectionalMambaBlock(nn.Module):
    """K independent MambaBlocks, one per scan order, summed with a residual
    (mamba_block.py:341-566).  K = 2, 4 (2D grid), 6 (3D) or 8 (4D).

    When the token count differs from the grid size (a subset of patches),
    the block falls back to forward + backward scans with blocks 0 and 1
    (mamba_block.py:554-559).
    """

    def __init__(self, d_model: int = 384, d_state: int = 16, d_conv: int = 4,
                 expand_factor: int = 2, num_directions: int = 2,
                 grid_shape: Optional[Sequence[int]] = None, scan_mode: str = "sequential"):
        super().__init__()
        if num_directions not in (2, 4, 6, 8):
            raise ValueError(f"num_directions must be 2, 4, 6, or 8, got {num_directions}")
        need = {4: 2, 6: 3, 8: 4}.get(num_directions)
        if need is not None and (grid_shape is None or len(grid_shape) != need):
            raise ValueError(f"K={num_directions} requires a {need}-D grid_shape, got {grid_shape}")
        self.num_directions = num_directions
        self.grid_shape = tuple(grid_shape) if grid_shape is not None else None
        self.scan_mode = scan_mode
        self.norm = nn.LayerNorm(d_model)
        self.mamba_blocks = nn.ModuleList(
            [MambaBlock(d_model, d_state, d_conv, expand_factor, scan_mode)
             for _ in range(num_directions)])
        self._tables = {}

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        bsz, n, _ = x.shape
        h, xr = layer_norm(x, self.norm, residual=True)                      # :548
        expected = math.prod(self.grid_shape) if self.grid_shape is not None else n
        if n != expected and self.num_directions > 2:                         # :554-559
            tok = _cached_table(self._tables, 2, n, None, x.device)
            blocks = [self.mamba_blocks[0], self.mamba_blocks[1]]
        else:
            grid = self.grid_shape if self.num_directions > 2 else None
            tok = _cached_table(self._tables, self.num_directions, n, grid, x.device)
            blocks = list(self.mamba_blocks)
        if any(_custom_scan(b) for b in blocks):
            return xr + _per_direction_forward(blocks, h, tok)
        return _directional_forward(blocks, h, tok, self.scan_mode, self,
                                    list(self.mamba_blocks), residual=xr)         # :562-566


# per-direction parameters stored as slices of one (K, ...) buffer per kind
STACKED_PARAMS = ("in_proj.weight", "conv1d.weight", "conv1d.bias", "x_proj.weight",
                  "dt_proj.weight", "dt_proj.bias", "A_log", "D", "out_proj.weight")


_STACKED_PATHS = tuple((tuple(n.split(".")[:-1]), n.split(".")[-1]) for n in STACKED_PARAMS)


def _param(blk, path):
    """The parameter at dotted ``path`` of ``blk``, by direct registry lookups
    (the same objects attribute access returns, without Module.__getattr__)."""
    *mods, name = path.split(".")
    for m in mods:
        blk = blk._modules[m]
    return blk._parameters[name]


def _params_of(blocks):
    """STACKED_PARAMS of each block, kind-major: [[kind 0 of block 0, ...], ...]."""
    out = []
    for mods, name in _STACKED_PATHS:
        row = []
        for b in blocks:
            for m in mods:
                b = b._modules[m]
            row.append(b._parameters[name])
        out.append(row)
    return out


def _is_slice_of(p, buf, k):
    return (p.device == buf.device and p.dtype == buf.dtype and p.shape == buf.shape[1:]
            and p.is_contiguous()
            and p.data_ptr() == buf.data_ptr() + k * buf.stride(0) * buf.element_size())


def _direction_stacks(owner, blocks):
    """The (K, ...) buffers whose k-th slices are the parameters of blocks[k],
    one per name of STACKED_PARAMS, kept on ``owner``.  Rebuilt (values
    copied from the current parameters, which then become slices of the new
    buffers) when any parameter is not its slice.  The per-call check
    compares each parameter's data pointer, shape, strides, dtype and device
    with its slice's (the buffers are held here, so their memory is never
    reused while the pointers are compared)."""
    return _stacks_of(owner, _params_of(blocks))


def _stacks_of(owner, params):
    flat = [p for ps in params for p in ps]
    bufs = owner.__dict__.get("_param_stacks")
    # (a module pickled by an older version holds a tuple here)
    if isinstance(bufs, list) and _lib.native().stacks_match(bufs, flat):
        return bufs
    with torch.no_grad():
        bufs = [torch.stack([p.detach() for p in ps], 0) for ps in params]
        for buf, ps in zip(bufs, params):
            for k, p in enumerate(ps):
                p.data = buf[k]
    owner.__dict__["_param_stacks"] = bufs
    return bufs


class _DirectionParams:
    """(buffers..., parameters...) -> the buffers, differentiable w.r.t. the
    parameters that are their slices (csrc/torch_ext.cpp): the backward hands
    each buffer's gradient to its K parameters as K contiguous slices."""

    @staticmethod
    def apply(nbuf, *tensors):
        return tuple(_lib.native().direction_params(list(tensors[:nbuf]), list(tensors[nbuf:])))


def _cached_table(cache, K, n, grid, device):
    key = (K, n, grid, str(device))
    if key not in cache:
        table = _dirs.seq_to_tok_table(K, n, grid).to(device)
        check_permutation_table(table)
        cache[key] = table
    return cache[key]


def _custom_scan(blk):
    """True when the caller replaced ``blk._scan_fn`` with a function other
    than the one its ``scan_mode`` selects (mamba_block.py:104-122).  The
    library's own modes all compute the same scan, which the fused block
    core runs; any other callable is honoured by _scan_fn_forward."""
    return blk._scan_fn is not get_scan_fn(blk.scan_mode)


def _scan_fn_forward(blk, x):
    """MambaBlock.__call__ in the reference's op sequence
    (mamba_block.py:155-192), calling ``blk._scan_fn(x, delta, A, B, C, D)``
    at :187.  Used when a block's scan function was replaced; the conv +
    SiLU runs on the HIP conv kernel, the rest on torch ops."""
    din, ns, R = blk.d_inner, blk.d_state, blk.dt_rank
    xz = F.linear(x, blk.in_proj.weight)                                      # :165
    xb, z = xz[..., :din], xz[..., din:]                                       # :166-167
    conv_w = blk.conv1d.weight.reshape(1, din, blk.d_conv)
    xc = causal_conv_silu(xb.unsqueeze(2), conv_w, blk.conv1d.bias.unsqueeze(0)).squeeze(2)  # :170-171
    dbc = F.linear(xc, blk.x_proj.weight)                                      # :174
    dt, Bm, Cm = dbc[..., :R], dbc[..., R:R + ns], dbc[..., R + ns:]           # :175-177
    delta = F.softplus(F.linear(dt, blk.dt_proj.weight, blk.dt_proj.bias))     # :180-181
    A = -torch.exp(blk.A_log)                                                  # :184
    y = blk._scan_fn(xc, delta, A, Bm, Cm, blk.D)                              # :187
    y = y * F.silu(z)                                                          # :190
    return F.linear(y, blk.out_proj.weight)                                    # :191


def _per_direction_forward(blocks, h, tok):
    """Sum over directions of block k run on h in the scan order tok[k]
    (a gathered copy, as the reference builds, mamba_block.py:407-533), its
    output put back in token order.  Used when a block's scan function was
    replaced, so that each block's own ``__call__`` runs."""
    y = None
    for k, blk in enumerate(blocks):
        order = tok[k].long()
        out = blk(h[:, order])
        out = out[:, torch.argsort(order)]
        y = out if y is None else y + out
    return y


def _directional_forward(blocks, h, tok, scan_mode, owner=None, stacked=None, residual=None):
    """Run len(blocks) MambaBlocks on one (B, N, E) input, block k scanning
    in the order of tok[k], and return the sum of their outputs and of the
    ``residual``, which out_proj's product adds as it stores.  The
    parameters of ``stacked`` (all direction blocks of ``owner``, of which
    ``blocks`` are the first) are slices of one buffer per kind; without an
    owner there is one block, whose parameters are used as they are."""
    K = len(blocks)
    if owner is None:
        params, stacks = _params_of(blocks), []
    else:
        params = _params_of(stacked)
        stacks = _stacks_of(owner, params)
    flat = [p for ps in params for p in ps[:K]]
    # the reference's "metal" mode is inference only (mamba_metal.py:230)
    args = mode_chunk_len(scan_mode), scan_mode == "metal"
    if _lib.is_tracing():
        return _lib.traced(_directional_flat, h, residual, tok, K, *args, len(flat), *flat, *stacks)
    return _directional(h, residual, tok, K, *args, flat, stacks)


def _directional(h, residual, tok, K, chunk_len, detach, params, stacks):
    return _lib.native().directional(h, params, stacks, K, tok, _resolve_chunk(h.shape[1], chunk_len), detach,
                                     residual)


def _directional_flat(h, residual, tok, K, chunk_len, detach, nparam, *tensors):
    return _directional(h, residual, tok, K, chunk_len, detach, list(tensors[:nparam]), list(tensors[nparam:]))
