"""dt_proj inside the fused scan forward (mvm_scan_fused_dt_fwd) against the
fused forward fed with the float64 product rounded to float32.

delta_raw: |got - ref| <= (R + 2) * 2^-23 * S, S = sum_r |dt_r W_r| (one
rounding per term at most, each of a partial sum <= S).  y and the checkpoints
follow from it: a change e of delta_raw changes delta by at most e, and y by a
sum over earlier positions, held here to the scan's own bar 1e-5 + 1e-4 |ref|.
"""

import ctypes

import numpy as np
import pytest
import torch

import mlx_vision_mamba_amd as mvm
from mlx_vision_mamba_amd import _lib, scan
from oracle import torch_ref

pytestmark = pytest.mark.gpu


def _ptr(t):
    return t.data_ptr() if t is not None else None


@pytest.mark.parametrize("R,N,D,L,chunk", [
    (1, 1, 5, 1, 0), (7, 4, 64, 16, 0), (13, 8, 70, 33, 16), (16, 16, 64, 48, 0), (17, 16, 100, 50, 16),
    (24, 16, 130, 47, 0), (25, 16, 64, 31, 32), (40, 5, 96, 17, 0), (48, 16, 128, 200, 0), (24, 16, 64, 300, 16)])
@pytest.mark.parametrize("order,bias,gate", [("table", True, True), ("identity", False, False)])
def test_forward_matches_the_two_step_form(cuda, R, N, D, L, chunk, order, bias, gate):
    gen = torch.Generator().manual_seed(R * 100 + L)
    K, bsz = 2, 2
    rn = lambda *s: torch.randn(*s, generator=gen).cuda()  # noqa: E731
    P = -(-(R + 2 * N) // 4) * 4
    dbc = rn(K, bsz * L, P)
    v = lambda t: t.view(K, bsz, L, t.shape[-1]).permute(1, 2, 0, 3)  # noqa: E731
    W = rn(K, D, R) * R ** -0.5
    A = -torch.exp(rn(K, D, N) * 0.3)
    u, Dv, z = v(rn(K, bsz * L, D)), rn(K, D), rn(bsz, L, K, D) if gate else None
    b = rn(K, D) - 3 if bias else None
    tok = torch.stack([torch.randperm(L, generator=gen) for _ in range(K)]).int().cuda() if order == "table" else None
    dt, Bm, Cm = (v(dbc)[..., s] for s in (slice(0, R), slice(R, R + N), slice(R + N, R + 2 * N)))
    ref_raw = torch.einsum("blkr,kdr->blkd", dt.double().cpu(), W.double().cpu()).cuda()
    S = torch.einsum("blkr,kdr->blkd", dt.double().abs().cpu(), W.double().abs().cpu()).cuda()
    raw = torch.full((K, bsz * L, D), float("nan")).cuda()
    y = torch.empty(bsz, L, K, D).cuda()
    y_raw = torch.empty_like(y) if gate else None
    fd = _lib.FusedDesc()
    s = fd.scan
    s.batch, s.seqlen, s.dim, s.dstate, s.ndir = bsz, L, D, N, K
    s.x_stride_b, s.x_stride_t, s.x_stride_k = u.stride()[:3]
    s.bc_stride_b, s.bc_stride_t, s.bc_stride_k = Bm.stride()[:3]
    s.seq_to_tok, s.chunk_len = _ptr(tok), chunk
    fd.dt_stride_b, fd.dt_stride_t, fd.dt_stride_k = v(raw).stride()[:3]
    fd.y_stride_b, fd.y_stride_t, fd.y_stride_k = y.stride()[:3]
    if gate:
        fd.z_stride_b, fd.z_stride_t, fd.z_stride_k = z.stride()[:3]
    lib = _lib.lib()
    ck = torch.empty(_lib.check(lib.mvm_scan_ckpt_elems(ctypes.byref(fd.scan)))).cuda()
    nb = _lib.check(lib.mvm_scan_fused_workspace_bytes(ctypes.byref(fd), 0, int(gate)))
    ws = torch.empty(max(nb, 1), dtype=torch.uint8, device=cuda)
    st = torch.cuda.current_stream().cuda_stream

    def run(raw_out, ck_out):
        _lib.check(lib.mvm_scan_fused_dt_fwd(
            ctypes.byref(fd), _ptr(u), _ptr(dt), R, _ptr(W), _ptr(b), _ptr(A), _ptr(Bm), _ptr(Cm), _ptr(Dv), _ptr(z),
            _ptr(y), _ptr(y_raw), _ptr(raw_out), _ptr(ck_out), _ptr(ws), nb, st))

    run(raw, ck)
    assert ((v(raw).double() - ref_raw).abs() <= (R + 2) * 2.0 ** -23 * S + 1e-30).all()
    ry, ry_raw, rck = scan.scan_fused_forward(u, v(ref_raw.float().permute(2, 0, 1, 3).reshape(K, bsz * L, D)), b, A,
                                              Bm, Cm, Dv, z, tok, chunk, save=True)
    ckv = lambda t: t.view(bsz * K, -(-L // 8), D, 16)[:, :L // 8]  # noqa: E731  (after every whole 8 positions)
    for got, ref in ((y, ry), (y_raw, ry_raw), (ckv(ck), ckv(rck))):
        if got is None:
            continue
        assert ((got - ref).abs() <= 1e-5 + 1e-4 * ref.abs()).all()
    first = y.clone()
    run(None, None)  # forward only
    assert torch.equal(y, first)


def test_rank_limits(cuda):
    fd = _lib.FusedDesc()
    s = fd.scan
    s.batch, s.seqlen, s.dim, s.dstate, s.ndir = 0, 4, 8, 4, 1
    s.x_stride_b, s.x_stride_t, s.x_stride_k, s.bc_stride_b, s.bc_stride_t, s.bc_stride_k = 32, 8, 8, 64, 16, 16
    for k in ("dt", "y", "z"):
        for d, val in (("b", 32), ("k", 8), ("t", 8)):
            setattr(fd, f"{k}_stride_{d}", val)
    call = lambda r: _lib.lib().mvm_scan_fused_dt_fwd(ctypes.byref(fd), None, None, r, *[None] * 12, 0, None)  # noqa: E731
    assert call(1) == 0 and call(48) == 0
    assert call(0) == call(49) == _lib.MVM_ERR_UNSUPPORTED


@pytest.mark.parametrize("E", [24, 272, 400, 784])
def test_block_against_the_restatement(cuda, E):
    """Blocks on either side of the rank limit (dt_rank 2, 17, 25, 49): output
    and parameter gradients against the float64 restatement."""
    torch.manual_seed(E)
    m = mvm.MambaBlock(E, d_state=8, scan_mode="hip").to(cuda)
    x = torch.randn(1, 21, E, generator=torch.Generator().manual_seed(1))
    g = torch.randn(1, 21, E, generator=torch.Generator().manual_seed(2))
    y = m(x.to(cuda))
    grads = torch.autograd.grad(y, list(m.parameters()), g.to(cuda))
    with torch.no_grad():
        y0 = m(x.to(cuda))
    assert torch.equal(y0, y)
    params = torch_ref.params_from_module(m)
    ref = torch_ref.mamba_block(params, "", x.double(), d_state=8, d_conv=4)
    rg = torch.autograd.grad(ref, [params[n] for n, _ in m.named_parameters()], g.double())
    for name, a, r in zip(["y"] + [n for n, _ in m.named_parameters()], [y, *grads], [ref, *rg]):
        err = np.abs(a.detach().double().cpu().numpy() - r.detach().numpy())
        bound = 1e-4 * r.detach().abs().max().item() + 1e-4 * r.detach().abs().numpy()
        assert (err <= bound).all(), (name, err.max())


@pytest.mark.parametrize("E,N", [(400, 1), (400, 3), (432, 2), (480, 1), (512, 1)])
def test_rows_no_longer_than_the_last_column_group(cuda, E, N):
    """Ranks 25..32 with rows of x_proj's output of at most 34 values: the
    third group of 16 columns lies past the rank, and past most of the rows."""
    torch.manual_seed(E)
    m = mvm.MambaBlock(E, d_state=N, scan_mode="hip").to(cuda)
    x = torch.randn(2, 19, E, generator=torch.Generator().manual_seed(1))
    y = m(x.to(cuda))
    params = torch_ref.params_from_module(m)
    ref = torch_ref.mamba_block(params, "", x.double(), d_state=N, d_conv=4).detach()
    err = (y.detach().double().cpu() - ref).abs()
    assert (err <= 1e-4 * ref.abs().max() + 1e-4 * ref.abs()).all(), err.max()
