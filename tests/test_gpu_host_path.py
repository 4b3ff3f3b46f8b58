"""The C++ host path (csrc/torch_ext.cpp): what its autograd Functions have
to keep besides the numbers the other tests check -- saved-tensor hooks,
streams, in-place checks, error types, launch timing, and the carry passes at
the edges of their batches."""

import numpy as np
import pytest
import torch

import mlx_vision_mamba_amd as mvm
from mlx_vision_mamba_amd import _lib, scan, synthetic
from mlx_vision_mamba_amd.conv import causal_conv_silu
from mlx_vision_mamba_amd.norm import layer_norm
from oracle import ref_lib, torch_ref

pytestmark = pytest.mark.gpu


def _block(cuda):
    torch.manual_seed(0)
    m = mvm.MultiDirectionalMambaBlock(32, d_state=4, num_directions=4, grid_shape=(4, 5), scan_mode="hip").to(cuda)
    x = torch.randn(2, 20, 32, generator=torch.Generator().manual_seed(1)).to(cuda).requires_grad_()
    g = torch.randn(2, 20, 32, generator=torch.Generator().manual_seed(2)).to(cuda)
    return m, x, g


def _step(m, x, g):
    y = m(x)
    return [y.detach(), *torch.autograd.grad(y, [x, *m.parameters()], g)]


def test_saved_tensor_hooks_and_side_stream(cuda):
    """The same results with every saved tensor moved to the host and back
    between forward and backward, and on another stream."""
    m, x, g = _block(cuda)
    ref = _step(m, x, g)
    seen = []

    def pack(t):
        seen.append(tuple(t.shape))
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(cuda)):
        got = _step(m, x, g)
    assert len(seen) >= 14
    for a, b in zip(got, ref):
        assert torch.equal(a, b)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = _step(m, x, g)
    torch.cuda.current_stream().wait_stream(s)
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


def test_inplace_change_of_a_saved_input_raises(cuda):
    u, dl, A, Bm, Cm, Dv, g = [t.to(cuda) for t in synthetic.make(1, 20, 8, 4, seed=0)]
    u.requires_grad_()
    y = scan.selective_scan(u, dl, A, Bm, Cm, Dv)
    dl.add_(0.1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward(g)


def test_no_checkpoints_without_a_gradient(cuda):
    """Under no_grad, and for inputs that need no gradient, nothing is kept."""
    u, dl, A, Bm, Cm, Dv, _ = [t.to(cuda) for t in synthetic.make(1, 20, 8, 4, seed=0)]
    assert scan.selective_scan(u, dl, A, Bm, Cm, Dv).grad_fn is None
    with torch.no_grad():
        assert scan.selective_scan(u.requires_grad_(), dl, A, Bm, Cm, Dv).grad_fn is None
    assert not scan.selective_scan_metal(u, dl, A, Bm, Cm, Dv).requires_grad
    assert scan.selective_scan(u, dl, A, Bm, Cm, Dv).grad_fn is not None


def test_error_types(cuda):
    """Library refusals stay ScanError with their code, bad shapes ValueError,
    tensors elsewhere RuntimeError."""
    K = 65536
    u, A = torch.zeros(1, 1, K, 1, device=cuda), torch.zeros(K, 1, 1, device=cuda)
    with pytest.raises(_lib.ScanError) as e:
        scan.scan_forward(u, u, A, u, u, torch.zeros(K, 1, device=cuda))
    assert e.value.code == _lib.MVM_ERR_UNSUPPORTED and "65535" in str(e.value)
    x = torch.zeros(1, 4, 8, device=cuda)
    with pytest.raises(ValueError, match="d_state"):
        scan.selective_scan(x, x, torch.zeros(8, 17, device=cuda), torch.zeros(1, 4, 17, device=cuda),
                            torch.zeros(1, 4, 17, device=cuda), torch.zeros(8, device=cuda))
    with pytest.raises(ValueError, match="B and C"):
        scan.selective_scan(x, x, torch.zeros(8, 2, device=cuda), torch.zeros(1, 4, 3, device=cuda),
                            torch.zeros(1, 4, 2, device=cuda), torch.zeros(8, device=cuda))
    with pytest.raises(RuntimeError, match="must be on"):
        scan.selective_scan(x, x, torch.zeros(8, 2), torch.zeros(1, 4, 2, device=cuda),
                            torch.zeros(1, 4, 2, device=cuda), torch.zeros(8, device=cuda))


@pytest.mark.parametrize("name", ["conv1d", "x_proj", "dt_proj", "in_proj", "out_proj"])
def test_block_refuses_parameters_that_do_not_fit(cuda, name):
    """A submodule left on the CPU, or replaced by one of another width, is
    an error of the host before anything of it is read on the GPU."""
    blk = mvm.MambaBlock(32, d_state=4, scan_mode="hip").to(cuda)
    x = torch.zeros(1, 8, 32, device=cuda)
    getattr(blk, name).to("cpu")
    with pytest.raises(RuntimeError):
        blk(x)
    getattr(blk, name).to(cuda)
    blk(x)
    lay = getattr(blk, name)
    if name == "conv1d":
        lay.weight = torch.nn.Parameter(torch.zeros(72, *lay.weight.shape[1:], device=cuda))
    else:
        lay.weight = torch.nn.Parameter(torch.zeros(lay.weight.shape[0], lay.weight.shape[1] + 4, device=cuda))
    with pytest.raises((RuntimeError, ValueError)):
        blk(x)


def test_launch_timing_records(cuda):
    m, x, g = _block(cuda)
    rec = []
    scan.set_scan_timing(rec)
    try:
        _step(m, x, g)
    finally:
        scan.set_scan_timing(None)
    _step(m, x, g)
    torch.cuda.synchronize()
    assert [r[0] for r in rec] == ["fwd", "bwd"]
    f, b = scan.algorithmic_bytes_fused(2 * 4, 20, 64, 4, 4)
    assert [r[3] for r in rec] == [f, b] and all(r[1].elapsed_time(r[2]) > 0 for r in rec)


@pytest.mark.parametrize("nchunk", [9, 16, 17, 24, 25])
def test_carry_batches(cuda, nchunk):
    """The carry passes load 8 chunks at a time: chunk counts at the edges of
    the batches (the last chunk partial) against the float64 oracle."""
    L = 16 * nchunk - 5
    ins = synthetic.make(2, L, 40, 16, seed=nchunk)
    t = [v.to(cuda) for v in ins]
    u4, d4, A3, B4, C4, D2 = t[0][:, :, None], t[1][:, :, None], t[2][None], t[3][:, :, None], t[4][:, :, None], t[5][None]
    y, ck = scan.scan_forward(u4, d4, A3, B4, C4, D2, chunk_len=16, save_ckpt=True)
    got = [y, *scan.scan_backward(u4, d4, A3, B4, C4, D2, t[6][:, :, None], ck, chunk_len=16)]
    np_in = [v.numpy() for v in ins]
    refs = [ref_lib.scan_fwd(*np_in[:6])] + list(ref_lib.scan_vjp(*np_in))
    for name, a, r in zip(["y", "du", "ddelta", "dA", "dB", "dC", "dD"], got, refs):
        a = a.double().cpu().numpy().reshape(r.shape)
        assert (np.abs(a - r) <= 1e-5 + 1e-4 * np.abs(r)).all(), name


@pytest.mark.parametrize("bsz,L,D", [(10, 331, 400), (3, 1037, 1000), (1, 70, 192)])
def test_bf16_forward_alone_takes_longer_chunks(cuda, bsz, L, D):
    """bf16 results without checkpoints: chunks of 48 or 64 positions where
    training takes 32 (the same 32 for the smallest), in the workspace sized
    for the shorter ones; within bf16's rounding of the oracle (8 significant
    bits: half of the spacing is at most 2^-8 of the value)."""
    ins = [t.to(torch.bfloat16) if i in (0, 3, 4) else t for i, t in enumerate(synthetic.make(bsz, L, D, 16, seed=3)[:6])]
    t = [v.to(cuda) for v in ins]
    ref = ref_lib.scan_fwd(*[v.float().numpy() for v in ins])
    with torch.no_grad():
        alone = scan.selective_scan(*t)
    trained = scan.selective_scan(t[0].requires_grad_(), *t[1:])
    for y in (alone, trained.detach()):
        assert y.dtype == torch.bfloat16
        assert (np.abs(y.double().cpu().numpy() - ref) <= 1e-5 + (2.0 ** -8 + 1e-4) * np.abs(ref)).all()


class _Norm(torch.nn.Module):
    def __init__(self):
        super().__init__()
        self.n = torch.nn.LayerNorm(32)

    def forward(self, x):
        h, xr = layer_norm(x, self.n, residual=True)
        return h * 2 + xr


class _Conv(torch.nn.Module):
    def __init__(self):
        super().__init__()
        self.w = torch.nn.Parameter(torch.randn(1, 32, 4, generator=torch.Generator().manual_seed(3)))
        self.b = torch.nn.Parameter(torch.zeros(1, 32))

    def forward(self, x):
        return causal_conv_silu(x.unsqueeze(2), self.w, self.b)


class _Scan(torch.nn.Module):
    def __init__(self, seed=4):
        super().__init__()
        ins = synthetic.make(2, 20, 32, 4, seed=seed)
        self.p = torch.nn.ParameterList([torch.nn.Parameter(t) for t in ins[2:6]])

    def forward(self, x):
        A, B, C, D = self.p
        return scan.selective_scan(x, x.abs(), A, B, C, D)


@pytest.mark.parametrize("make", [
    lambda: mvm.MambaBlock(32, d_state=4, scan_mode="hip"),
    lambda: mvm.MambaBlock(32, d_state=4, scan_mode="sequential"),
    lambda: mvm.ResidualMambaBlock(32, d_state=4, scan_mode="hip"),
    lambda: mvm.BidirectionalMambaBlock(32, d_state=4, scan_mode="hip"),
    lambda: mvm.MultiDirectionalMambaBlock(32, d_state=4, num_directions=4, grid_shape=(4, 5), scan_mode="hip"),
    _Norm, _Conv, _Scan], ids=["mamba", "sequential", "residual", "bidirectional", "multi", "norm", "conv", "scan"])
def test_traced_modules_compute(cuda, make):
    """A torch.jit trace runs the calls again on new inputs, with and without
    gradients: the same outputs and gradients as the module's own."""
    torch.manual_seed(0)
    m = make().to(cuda)
    rn = lambda seed: torch.randn(2, 20, 32, generator=torch.Generator().manual_seed(seed)).to(cuda)  # noqa: E731
    m(rn(0))  # (builds the parameter buffers)
    t = torch.jit.trace(m, rn(0))
    x = rn(1).requires_grad_()
    y, r = t(x), m(x)
    assert torch.equal(y, r)
    g = torch.randn(r.shape, generator=torch.Generator().manual_seed(2)).to(cuda)
    ps = [x, *m.parameters()]
    for _ in range(2):
        for a, b in zip(torch.autograd.grad(y, ps, g, retain_graph=True), torch.autograd.grad(r, ps, g, retain_graph=True)):
            assert torch.equal(a, b)
    with torch.no_grad():
        assert torch.equal(t(x), m(x))
        assert t(x).grad_fn is None


@pytest.mark.parametrize("grid", [(4, 5), (37, 57)])  # 160 and 16,872 batch x rows
def test_second_derivative_of_a_block_raises(cuda, grid):
    """The core's backward is raw launches: asked for a graph of it, the block
    refuses (with frozen parameters, where the first derivative was always
    given, as soon as a derivative through it is taken)."""
    torch.manual_seed(0)
    m = mvm.MultiDirectionalMambaBlock(32, d_state=4, num_directions=4, grid_shape=grid, scan_mode="hip").to(cuda)
    x = torch.randn(2, grid[0] * grid[1], 32, generator=torch.Generator().manual_seed(1)).to(cuda).requires_grad_()
    ref = torch.autograd.grad(m(x).square().sum(), x)[0]
    with pytest.raises(RuntimeError, match="not twice differentiable"):
        torch.autograd.grad(m(x).square().sum(), x, create_graph=True)
    m.requires_grad_(False)
    (g,) = torch.autograd.grad(m(x).square().sum(), x, create_graph=True)
    assert torch.allclose(g, ref, rtol=1e-4, atol=1e-4 * ref.abs().max().item())
    with pytest.raises(RuntimeError, match="not twice differentiable"):
        torch.autograd.grad(g.square().sum(), x)
    with pytest.raises(RuntimeError, match="not twice differentiable"):
        (m(x).sum() + g.square().sum()).backward()


@pytest.mark.parametrize("make", [_Norm, _Conv, _Scan], ids=["norm", "conv", "scan"])
def test_second_derivative_of_the_kernels_raises(cuda, make):
    """create_graph gives the same first derivatives; a derivative through
    them raises instead of lacking the kernel's part."""
    m = make().to(cuda)
    x = torch.randn(2, 20, 32, generator=torch.Generator().manual_seed(1)).to(cuda).requires_grad_()
    ps = [x, *m.parameters()]
    ref = torch.autograd.grad(m(x).square().sum(), ps)
    got = torch.autograd.grad(m(x).square().sum(), ps, create_graph=True)
    for a, b in zip(got, ref):
        assert torch.equal(a, b)
    for p in (x, ps[-1]):
        with pytest.raises(RuntimeError, match="not twice differentiable"):
            torch.autograd.grad(sum(a.square().sum() for a in got), p, retain_graph=True)


def test_gradient_of_out_proj_is_differentiable(cuda):
    """A penalty on the gradient of out_proj's weight: its graph leads through
    the core's first derivative only.  Against the float64 restatement."""
    torch.manual_seed(0)
    m = mvm.MambaBlock(32, d_state=4, scan_mode="hip").to(cuda)
    x = torch.randn(2, 20, 32, generator=torch.Generator().manual_seed(1))

    def penalty(y, w, xx):
        (g,) = torch.autograd.grad(y.square().sum(), w, create_graph=True)
        return torch.autograd.grad(g.square().sum(), [xx, w])

    xg = x.to(cuda).requires_grad_()
    got = penalty(m(xg), m.out_proj.weight, xg)
    params = torch_ref.params_from_module(m)
    xd = x.double().requires_grad_()
    ref = penalty(torch_ref.mamba_block(params, "", xd, d_state=4, d_conv=4), params["out_proj.weight"], xd)
    for a, r in zip(got, ref):
        assert (a.double().cpu() - r).norm() <= 1e-5 * r.norm()


@pytest.mark.parametrize("make", [
    lambda: mvm.MambaBlock(32, d_state=4, scan_mode="hip"),
    lambda: mvm.ResidualMambaBlock(32, d_state=4, scan_mode="hip"),
    lambda: mvm.BidirectionalMambaBlock(32, d_state=4, scan_mode="hip"),
    lambda: mvm.MultiDirectionalMambaBlock(32, d_state=4, num_directions=4, grid_shape=(4, 5), scan_mode="hip"),
    _Conv, _Scan], ids=["mamba", "residual", "bidirectional", "multi", "conv", "scan"])
def test_outputs_can_be_changed_in_place(cuda, make):
    """No output is a view made inside a Function: in-place changes of it are
    recorded as those of any other tensor."""
    torch.manual_seed(0)
    m = make().to(cuda)
    x = torch.randn(2, 20, 32, generator=torch.Generator().manual_seed(1)).to(cuda).requires_grad_()
    w = torch.randn(32, generator=torch.Generator().manual_seed(2)).to(cuda).requires_grad_()
    ps = [x, w, *m.parameters()]
    y = m(x)
    ref = torch.autograd.grad(torch.relu((y + w) * 2).square().sum(), ps)
    y = m(x)
    y += w
    y.mul_(2)
    torch.relu_(y)
    for a, b in zip(torch.autograd.grad(y.square().sum(), ps), ref):
        assert torch.equal(a, b)


@pytest.mark.parametrize("which,change,error,match", [
    ("u", lambda t: t[:, :-1], ValueError, "equal shape"),
    ("ckpt", lambda t: torch.cat([t[:1], t])[1:], _lib.ScanError, "16-byte aligned"),
    ("u", lambda t: t.cpu(), RuntimeError, "only on the GPU")])
def test_error_types_of_a_backward(cuda, which, change, error, match):
    """What a backward's host checks refuse (here: saved tensors that a hook
    hands back changed) keeps its type through the autograd engine."""
    u, *ins = [t.to(cuda) for t in synthetic.make(1, 20, 8, 4, seed=0)[:6]]
    pick = {"u": lambda t: t.shape == u.shape and torch.equal(t, u), "ckpt": lambda t: t.dim() == 1 and t.numel() > 8}
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: change(t) if pick[which](t) else t):
        y = scan.selective_scan(u.clone().requires_grad_(), *ins)
    with pytest.raises(error, match=match) as e:
        y.sum().backward()
    assert type(e.value) is error
    if error is _lib.ScanError:
        assert e.value.code == _lib.MVM_ERR_INVALID_ARG


@pytest.mark.parametrize("shape", [(0, 9, 2, 8), (2, 0, 2, 8), (1, 1, 1, 8), (3, 1, 2, 8)])
def test_conv_backward_of_an_expanded_gradient(cuda, shape):
    """The gradient of a sum is expanded: strides of zero, which an empty
    tensor keeps through contiguous()."""
    gen = torch.Generator().manual_seed(1)
    x = torch.randn(*shape, generator=gen).to(cuda).requires_grad_()
    w = torch.randn(shape[2], 8, 4, generator=gen).to(cuda).requires_grad_()
    b = torch.randn(shape[2], 8, generator=gen).to(cuda).requires_grad_()
    got = torch.autograd.grad(causal_conv_silu(x, w, b).sum(), (x, w, b))
    xd, wd, bd = [t.detach().double().cpu().requires_grad_() for t in (x, w, b)]
    pad = torch.nn.functional.pad(xd, (0, 0, 0, 0, 3, 0))
    z = sum(pad[:, j:j + shape[1]] * wd[..., j] for j in range(4)) + bd
    ref = torch.autograd.grad(torch.nn.functional.silu(z).sum(), (xd, wd, bd))
    for a, r in zip(got, ref):
        assert a.shape == r.shape and torch.allclose(a.double().cpu(), r, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("cls", [mvm.MambaBlock, mvm.ResidualMambaBlock])
def test_batched_gradients_of_out_proj(cuda, cls):
    """A Jacobian's rows in one vmapped backward, as far as out_proj's weight."""
    torch.manual_seed(0)
    m = cls(32, d_state=4, scan_mode="hip").to(cuda)
    w = getattr(m, "mamba", m).out_proj.weight
    gen = torch.Generator().manual_seed(1)
    y = m(torch.randn(2, 20, 32, generator=gen).to(cuda))
    v = torch.randn(3, 2, 20, 32, generator=gen).to(cuda)
    (got,) = torch.autograd.grad(y, w, v, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        (ref,) = torch.autograd.grad(y, w, v[i], retain_graph=True)
        # (40 terms in any order)
        assert (got[i] - ref).abs().max() <= 1e-5 * ref.abs().max()
