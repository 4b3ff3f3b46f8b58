"""GPU parity of the float32 products on the bf16 matrix units
(include/mvm_gemm.h) against float64.

Per element |got - ref| <= (6 * ceil(k / 16) + splits + 2) * 2^-23 * S with
S = sum_p |a_p b_p|: one rounding of a partial sum (at most S, a unit of at
most 2^-23) for each of the six MFMAs per 16 values of k, for each part of a
split and for the addition to C; the products left out of the split are below
2^-25 * S.  Over normal inputs the error in the 2-norm is also held to that of
torch's float32 product (the BLAS library's float32 matrix instructions).
"""

import ctypes

import pytest
import torch
import torch.nn.functional as F

from mlx_vision_mamba_amd import _lib, gemm

pytestmark = pytest.mark.gpu


def _operand(rows, k, kmajor, batch, pad, gen):
    """(logical (batch, rows, k) float64-free values, buffer, leading dim, batch stride)"""
    r, c = (rows, k) if kmajor else (k, rows)
    ld = -(-c // 4) * 4 + pad
    buf = torch.randn(batch, r, ld, generator=gen).cuda()
    v = buf[:, :, :c]
    return (v if kmajor else v.transpose(1, 2)), buf, ld, r * ld


def _run(desc, A, B, C, add=None):
    lib = _lib.lib()
    nbytes = _lib.check(lib.mvm_gemm_workspace_bytes(ctypes.byref(desc)))
    ws = torch.full((max(nbytes, 1),), 255, dtype=torch.uint8, device="cuda")  # NaN if read before written
    _lib.check(lib.mvm_gemm_f32(ctypes.byref(desc), A.data_ptr(), B.data_ptr(),
                                add.data_ptr() if add is not None else None, C.data_ptr(), ws.data_ptr(),
                                nbytes, torch.cuda.current_stream().cuda_stream))


CASES = [
    # m, n, k, batch, splits, pad
    (1, 1, 1, 1, 0, 0), (3, 5, 7, 2, 0, 4), (64, 64, 32, 1, 0, 0), (65, 63, 33, 1, 0, 0),
    (127, 129, 31, 1, 1, 0), (128, 128, 16, 1, 1, 0), (200, 131, 17, 3, 1, 4), (129, 257, 100, 1, 3, 0),
    (300, 200, 1655, 1, 0, 0), (1100, 1300, 48, 1, 0, 0), (1100, 1300, 75, 1, 1, 0), (64, 72, 50, 1, 24, 0),
    (70, 60, 40, 2, 64, 0), (5, 4, 0, 1, 0, 0), (2500, 1700, 36, 1, 2, 0),
]


@pytest.mark.parametrize("akm", [0, 1])
@pytest.mark.parametrize("bkm", [0, 1])
@pytest.mark.parametrize("m,n,k,batch,splits,pad", CASES)
def test_product(cuda, m, n, k, batch, splits, pad, akm, bkm):
    gen = torch.Generator().manual_seed(m * 7 + n * 3 + k)
    a, A, lda, sa = _operand(m, max(k, 1), akm, batch, pad, gen)
    b, B, ldb, sb = _operand(n, max(k, 1), bkm, batch, pad, gen)
    ldc = n + 3
    for acc in (0, 1, 2):  # nothing, C itself, another buffer is added
        C0 = torch.randn(batch, m, ldc, generator=gen).cuda()
        C = C0.clone() if acc < 2 else torch.randn(batch, m, ldc, generator=gen).cuda()
        keep = C.clone()
        d = _lib.GemmDesc(m, n, k, batch, lda, ldb, ldc, sa, sb, m * ldc, 0, 0, akm, bkm, 0, splits)
        _run(d, A, B, C, (None, C, C0)[acc])
        ad, bd = a.double()[:, :, :k], b.double()[:, :, :k].transpose(1, 2).contiguous()
        ref = ad @ bd + (C0.double()[:, :, :n] if acc else 0)
        S = ad.abs() @ bd.abs() + (C0.double()[:, :, :n].abs() if acc else 0)
        bound = (6 * -(-k // 16) + max(splits, 24) + 2) * 2.0 ** -23 * S
        assert ((C.double()[:, :, :n] - ref).abs() <= bound).all()
        assert torch.equal(C[:, :, n:], keep[:, :, n:])  # nothing outside the matrix
        again = keep.clone()
        _run(d, A, B, again, (None, again, C0)[acc])
        assert torch.equal(again, C)


@pytest.mark.parametrize("m,n,k", [(640, 768, 384), (392, 768, 3072), (1655, 200, 800), (384, 768, 6272)])
@pytest.mark.parametrize("shift", [0.0, 1.0])
def test_error_no_larger_than_float32(cuda, m, n, k, shift):
    """Unit normal inputs, and inputs of one sign (shift: |x|, no cancellation)."""
    gen = torch.Generator().manual_seed(k)
    A, B = torch.randn(m, k, generator=gen).cuda(), torch.randn(n, k, generator=gen).cuda()
    if shift:
        A, B = A.abs(), B.abs()
    C = torch.empty(m, n, device="cuda")
    _run(_lib.GemmDesc(m, n, k, 1, k, k, n, 0, 0, 0, 0, 0, 1, 1, 0, 0), A, B, C)
    ref = A.double() @ B.double().t().contiguous()
    err = lambda x: ((x.double() - ref).norm() / ref.norm()).item()  # noqa: E731
    assert err(C) <= err(F.linear(A, B)), (err(C), err(F.linear(A, B)))


@pytest.mark.parametrize("K,D", [(3, 32), (4, 96), (2, 160), (2, 16), (2, 400), (3, 48)])
def test_segments(cuda, K, D):
    """One product over K weight matrices that lie apart."""
    gen = torch.Generator().manual_seed(K)
    M, E = 150, 72
    y, W = torch.randn(M, K, D, generator=gen).cuda(), torch.randn(K, E, D, generator=gen).cuda()
    ref = torch.einsum("mkd,ked->me", y.double().cpu(), W.double().cpu())
    S = torch.einsum("mkd,ked->me", y.double().abs().cpu(), W.double().abs().cpu())
    for splits in (0, 1, 2, 5):
        C = torch.empty(M, E, device="cuda")
        _run(_lib.GemmDesc(M, E, K * D, 1, K * D, D, E, 0, 0, 0, D, E * D, 1, 1, 0, splits), y, W, C)
        assert ((C.double().cpu() - ref).abs() <= (6 * -(-K * D // 16) + 26) * 2.0 ** -23 * S).all()


@pytest.mark.parametrize("akm,bkm", [(1, 1), (1, 0), (0, 0)])
@pytest.mark.parametrize("k,splits", [(40, 1), (333, 3)])
def test_special_values_as_float32(cuda, akm, bkm, k, splits):
    """Infinities, NaN, values near the largest float32 and tiny inputs give
    what float32 arithmetic gives."""
    m, n = 140, 70
    gen = torch.Generator().manual_seed(k)
    a, A, lda, _ = _operand(m, k, akm, 1, 0, gen)
    b, B, ldb, _ = _operand(n, k, bkm, 1, 0, gen)
    a, b = a[0], b[0]
    inf = float("inf")
    a[3, 5], a[9, 7], a[20, 0] = inf, -inf, float("nan")
    a[70] = 0.0
    a[70, 1], b[:, 1] = 3.4028e38, 0.25  # rounds to infinity in bf16; the product is finite
    a[100, 2], a[100, 3], b[11, 2], b[11, 3] = inf, inf, 1.0, -1.0
    C = torch.empty(m, n, device="cuda")
    d = _lib.GemmDesc(m, n, k, 1, lda, ldb, n, 0, 0, 0, 0, 0, akm, bkm, 0, splits)
    _run(d, A, B, C)
    ref = (a.double() @ b.double().t().contiguous()).float()
    assert torch.equal(torch.isnan(C), torch.isnan(ref))
    assert torch.equal(torch.isinf(C), torch.isinf(ref)) and (C[torch.isinf(C)] == ref[torch.isinf(ref)]).all()
    ok = torch.isfinite(ref)
    S = a.abs().nan_to_num(0, 0, 0).double() @ b.abs().double().t().contiguous()
    assert ((C - ref).double().abs()[ok] <= ((k + 4) * 2.0 ** -23 * S)[ok]).all()
    # inputs so small that the split's low parts underflow
    A.copy_(torch.randn(A.shape, generator=gen) * 2.0 ** -118)
    B.copy_(torch.randn(B.shape, generator=gen))
    _run(d, A, B, C)
    ref = a.double() @ b.double().t().contiguous()
    S = a.abs().double() @ b.abs().double().t().contiguous()
    assert ((C.double() - ref).abs() <= (k + 4) * (2.0 ** -23 * S + 2.0 ** -149)).all()


@pytest.mark.parametrize("B,n,K,D,E", [(2, 37, 1, 24, 12), (3, 50, 4, 64, 40), (0, 5, 2, 32, 16), (1, 9, 2, 40, 20)])
def test_projections_match_autograd(cuda, B, n, K, D, E):
    """in_proj / out_proj (also where the kernels do not take the shape:
    Din = 40 in two directions, not a multiple of 16) against float64 autograd."""
    gen = torch.Generator().manual_seed(1)
    h = torch.randn(B, n, E, generator=gen).cuda().requires_grad_()
    Wi = torch.randn(K * 2 * D, E, generator=gen).cuda().requires_grad_()
    Wo = torch.randn(K, E, D, generator=gen).cuda().requires_grad_()
    xz = gemm.in_proj(h, Wi)
    out = gemm.out_proj(xz.view(B, n, K, 2 * D)[..., D:].contiguous(), Wo)
    g = torch.randn(B, n, E, generator=gen).cuda()
    got = [out, *torch.autograd.grad(out, (h, Wi, Wo), g)]
    hd, wi, wo = [t.detach().double().cpu().requires_grad_() for t in (h, Wi, Wo)]
    o64 = torch.einsum("bnkd,ked->bne", (hd @ wi.t()).view(B, n, K, 2 * D)[..., D:], wo)
    ref = [o64, *torch.autograd.grad(o64, (hd, wi, wo), g.double().cpu())]
    for x, r in zip(got, ref):
        assert x.shape == r.shape
        # two chained products of at most 6 * 60 roundings each
        assert (x.double().cpu() - r).norm() <= 800 * 2.0 ** -24 * r.norm() + 1e-30


@pytest.mark.parametrize("q,m,k,n", [(1, 196, 24, 96), (2, 331, 13, 40), (2, 90, 29, 33), (1, 70, 50, 30),
                                     (3, 64, 32, 24), (2, 9000, 24, 16), (2, 9000, 16, 24)])
def test_batched_matches_float64(cuda, q, m, k, n):
    """The direction-batched products in the forms of x_proj and dt_proj:
    plain and transposed operands, column slices of a wider buffer (rows of a
    multiple of 4 and not), accumulation, and the streamed ones."""
    gen = torch.Generator().manual_seed(m + k)
    rn = lambda *s: torch.randn(*s, generator=gen).cuda()  # noqa: E731
    for pad in (0, 3, 4):
        wide = rn(q, m, k + pad)
        a, at = wide[..., :k], rn(q, k, m + pad)[..., :m]
        b, bt = rn(q, k, n), rn(q, n, k + pad)[..., :k]
        for A, ta in ((a, False), (at, True)):
            for B, tb in ((b, False), (bt, True)):
                for stream in (False, True):
                    Ad = (A.transpose(1, 2) if ta else A).double()
                    Bd = (B.transpose(1, 2) if tb else B).contiguous().double()
                    ref, S = Ad @ Bd, Ad.abs() @ Bd.abs()
                    bound = (6 * -(-k // 16) + 26) * 2.0 ** -23
                    got = gemm.batched(A, B, ta=ta, tb=tb, stream=stream)
                    assert ((got.double() - ref).abs() <= bound * S).all()
                    out = rn(q, m, n + pad)
                    keep = out.clone()
                    gemm.batched(A, B, out=out[..., :n], ta=ta, tb=tb, accumulate=True)
                    r2, S2 = ref + keep[..., :n].double(), S + keep[..., :n].double().abs()
                    assert ((out[..., :n].double() - r2).abs() <= bound * S2).all()
                    assert torch.equal(out[..., n:], keep[..., n:])


def test_projections_are_twice_differentiable(cuda):
    """Second derivatives of in_proj and out_proj against float64 autograd."""
    gen = torch.Generator().manual_seed(1)
    B, n, K, D, E = 2, 9, 2, 16, 12
    h = torch.randn(B, n, E, generator=gen).cuda().requires_grad_()
    Wi = torch.randn(K * D, E, generator=gen).cuda().requires_grad_()
    Wo = torch.randn(K, E, D, generator=gen).cuda().requires_grad_()
    res = torch.randn(B, n, E, generator=gen).cuda()

    def second(out, ts):
        gs = torch.autograd.grad(out.tanh().sum(), ts, create_graph=True)
        return torch.autograd.grad(sum(g.square().sum() for g in gs), ts)

    got = second(gemm.out_proj(gemm.in_proj(h, Wi).view(B, n, K, D), Wo) + res, (h, Wi, Wo))
    hd, wi, wo = [t.detach().double().cpu().requires_grad_() for t in (h, Wi, Wo)]
    out = torch.einsum("bnkd,ked->bne", (hd @ wi.t()).view(B, n, K, D), wo) + res.double().cpu()
    for a, r in zip(got, second(out, (hd, wi, wo))):
        # tanh's argument is off by the products' roundings (a few 2^-24 of a sum of 100), its second
        # derivative by as much again
        assert (a.double().cpu() - r).norm() <= 1e-4 * r.norm()


@pytest.mark.parametrize("tb", [False, True])
def test_batched_takes_overlapping_and_single_rows(cuda, tb):
    """Operands with rows that share memory (an expanded row), or one row of
    any stride: torch's product, as for other layouts the kernels do not take."""
    gen = torch.Generator().manual_seed(1)
    rn = lambda *s: torch.randn(*s, generator=gen).cuda()  # noqa: E731
    a = rn(2, 37, 40)
    b = (rn(2, 1, 40).expand(2, 24, 40) if tb else rn(2, 1, 24).expand(2, 40, 24))
    one = rn(2 * 40).as_strided((2, 1, 40), (40, 1, 1))
    for A in (a, one):
        ref = A.double() @ (b.transpose(1, 2) if tb else b).contiguous().double()
        S = A.double().abs() @ (b.transpose(1, 2) if tb else b).contiguous().double().abs()
        # (any order of 40 float32 additions)
        assert ((gemm.batched(A, b, tb=tb).double() - ref).abs() <= 42 * 2.0 ** -24 * S).all()


def test_block_with_an_expanded_projection(cuda):
    """x_proj's weight as one row for all outputs: the block of the same values
    laid out in full."""
    import mlx_vision_mamba_amd as mvm
    torch.manual_seed(0)
    m = mvm.MambaBlock(32, d_state=4, scan_mode="hip").to(cuda)
    x = torch.randn(2, 20, 32, generator=torch.Generator().manual_seed(1)).to(cuda)
    w = m.x_proj.weight.detach()[:1].expand(m.x_proj.weight.shape)
    out = []
    for v in (w, w.clone()):
        m.x_proj.weight = torch.nn.Parameter(v)
        y = m(x)
        out.append([y, *torch.autograd.grad(y.sum(), m.parameters())])
    for p, q in zip(*out):
        assert (p - q).abs().max() <= 1e-5 * q.abs().max()


@pytest.mark.parametrize("akm,bkm", [(1, 1), (1, 0), (0, 1), (0, 0)])
@pytest.mark.parametrize("k,splits", [(20, 1), (64, 1), (333, 3)])
@pytest.mark.parametrize("kind", ["one row", "one column", "times large", "single terms", "subnormal row", "both small"])
def test_tiny_values_beside_normal_ones(cuda, akm, bkm, k, splits, kind):
    """Operands whose low parts are finer than bf16's smallest subnormal keep
    float32's precision: (k + 4) roundings of 2^-23 S, S = sum |a b|, each of
    at least half a float32 subnormal."""
    m, n = 140, 70
    gen = torch.Generator().manual_seed(k)
    a, A, lda, _ = _operand(m, k, akm, 1, 0, gen)
    b, B, ldb, _ = _operand(n, k, bkm, 1, 0, gen)
    a, b = a[0], b[0]
    if kind == "one row":
        a[71] *= 2.0 ** -118
    elif kind == "one column":
        b[3] *= 2.0 ** -121
    elif kind == "times large":
        a *= 2.0 ** -118
        b *= 2.0 ** 60
    elif kind == "single terms":  # tiny values reach the result alone, in rows of normal ones
        a[:, 5] *= 2.0 ** -120
        b[9] = 0.0
        b[9, 5] = 2.0 ** 90
    elif kind == "subnormal row":
        a[100] *= 2.0 ** -138
        b *= 2.0 ** 20
    else:
        a *= 2.0 ** -60
        b *= 2.0 ** -58
    C = torch.empty(m, n, device="cuda")
    d = _lib.GemmDesc(m, n, k, 1, lda, ldb, n, 0, 0, 0, 0, 0, akm, bkm, 0, splits)
    _run(d, A, B, C)
    ref = a.double() @ b.double().t().contiguous()
    S = a.abs().double() @ b.abs().double().t().contiguous()
    assert ((C.double() - ref).abs() <= (k + 4) * (2.0 ** -23 * S + 2.0 ** -149)).all()


@pytest.mark.parametrize("m", [4095, 4096])
def test_streamed_product_on_both_sides_of_its_rule(cuda, m):
    """delta_raw's gradient times W_dt, 4 x m rows of 768 channels: the
    kernels below 12 Mi streamed values, torch from there on."""
    gen = torch.Generator().manual_seed(m)
    a, b = [torch.randn(*s, generator=gen).cuda() for s in ((4, m, 768), (4, 768, 24))]
    out = torch.empty(4, m, 56, device="cuda")
    gemm.batched(a, b, out=out[..., :24], stream=True)
    ref, S = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    # (any order of 768 float32 additions; both are far below it)
    assert ((out[..., :24].double() - ref).abs() <= 770 * 2.0 ** -24 * S).all()


def test_training_and_inference_form_delta_alike(cuda):
    """A block of more than 16384 batch x rows: the same output bit for bit
    with and without gradients."""
    import mlx_vision_mamba_amd as mvm
    torch.manual_seed(0)
    m = mvm.MambaBlock(48, d_state=4, scan_mode="hip").to(cuda)
    x = torch.randn(9, 1900, 48, generator=torch.Generator().manual_seed(1)).to(cuda)
    y = m(x)
    with torch.no_grad():
        assert torch.equal(m(x), y)
