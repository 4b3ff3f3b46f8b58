"""Host-side checks of include/mvm_gemm.h (no GPU, no launches)."""

import ctypes
import os
import re

import pytest

from mlx_vision_mamba_amd import _lib

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
