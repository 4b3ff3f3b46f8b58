"""Host-side checks of include/mvm_gemm.h and of the products and parameter
buffers of csrc/torch_ext.cpp (no GPU, no launches)."""

import ctypes
import os
import re

import pytest
import torch

import mlx_vision_mamba_amd as mvm
from mlx_vision_mamba_amd import _lib, gemm, mamba_block

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_declared_functions_are_bound():
    text = open(os.path.join(ROOT, "include", "mvm_gemm.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    arity = {name: params.count(",") + 1
             for name, params in re.findall(r"\b(mvm_[a-z0-9_]+)\s*\(([^)]*)\)\s*;", text)}
    assert arity == {name: len(args) for name, (_, args) in _lib.GEMM_SIGNATURES.items()}
    for name in arity:
        assert hasattr(_lib.lib(), name)


def _desc(**kw):
    d = _lib.GemmDesc(8, 8, 64, 1, 64, 64, 8, 0, 0, 0, 0, 0, 1, 1, 0, 0)
    for k, v in kw.items():
        setattr(d, k, v)
    return d


@pytest.mark.parametrize("kw,code", [
    (dict(), 0), (dict(m=0), 0), (dict(k=0), 0), (dict(b_seg=32, b_seg_stride=512, ldb=32), 0),
    (dict(batch=2, c_stride_batch=64), 0),
    (dict(m=-1), _lib.MVM_ERR_INVALID_ARG), (dict(lda=60), _lib.MVM_ERR_INVALID_ARG),
    (dict(lda=66), _lib.MVM_ERR_UNSUPPORTED), (dict(a_kmajor=0, lda=9), 0),
    (dict(a_kmajor=2), _lib.MVM_ERR_INVALID_ARG), (dict(splits=65), _lib.MVM_ERR_INVALID_ARG),
    (dict(ldb=1 << 21), _lib.MVM_ERR_UNSUPPORTED), (dict(b_seg=16, ldb=16), 0), (dict(b_seg=8), _lib.MVM_ERR_INVALID_ARG),
    (dict(b_seg=96), _lib.MVM_ERR_INVALID_ARG), (dict(batch=2), _lib.MVM_ERR_INVALID_ARG),
    (dict(ldc=7), _lib.MVM_ERR_INVALID_ARG), (dict(m=1 << 31), _lib.MVM_ERR_UNSUPPORTED),
])
def test_validation(kw, code):
    assert _lib.lib().mvm_gemm_validate(ctypes.byref(_desc(**kw))) == code


def test_workspace_is_the_split():
    """The plan leaves large products whole and splits long sums of few tiles."""
    ws = lambda **kw: _lib.lib().mvm_gemm_workspace_bytes(ctypes.byref(_desc(**kw)))  # noqa: E731
    assert ws(m=6272, n=6144, k=384, lda=384, ldb=384, ldc=6144) == 0
    assert ws(splits=3) == 3 * 64 * 4
    n = ws(m=6272, n=384, k=6144, lda=6144, ldb=6144, ldc=384)
    assert n > 0 and n % (6272 * 384 * 4) == 0


@pytest.mark.parametrize("a,b,out,ta,tb,what", [
    ((2, 6, 8), (2, 4, 7), None, False, True, "do not fit"),       # summed lengths differ
    ((2, 6, 8), (3, 8, 4), None, False, False, "do not fit"),      # batches differ
    ((2, 8, 6), (2, 8, 4), (2, 6, 5), True, False, "do not fit"),  # output columns
    ((6, 8), (2, 8, 4), None, False, False, "3-D|out of range"),
    ((2, 6, 8), (2, 8, 4), None, False, False, "only on the GPU"),
])
def test_batched_products_refuse_operands_that_do_not_fit(a, b, out, ta, tb, what):
    """The kernels see pointers only, so the host refuses what torch's
    batched product would refuse (and CPU tensors: there is no fallback)."""
    with pytest.raises((RuntimeError, IndexError), match=what):
        gemm.batched(torch.zeros(a), torch.zeros(b), None if out is None else torch.zeros(out), ta=ta, tb=tb)


def test_stacks_of_an_older_pickle_are_rebuilt():
    """A direction module pickled whole by an older version holds a (buffers,
    pointers) tuple where the buffers are now: rebuilt, values kept."""
    m = mvm.BidirectionalMambaBlock(8, d_state=2, scan_mode="hip")
    blocks = [m.forward_mamba, m.backward_mamba]
    before = {k: v.clone() for k, v in m.state_dict().items()}
    bufs = mamba_block._direction_stacks(m, blocks)
    assert mamba_block._direction_stacks(m, blocks) is bufs
    m.__dict__["_param_stacks"] = (bufs, [(0, torch.float32, (1,))])
    again = mamba_block._direction_stacks(m, blocks)
    assert isinstance(again, list) and mamba_block._direction_stacks(m, blocks) is again
    for k, v in m.state_dict().items():
        assert torch.equal(v, before[k])
