"""Operands that the eager entry points refuse before they launch anything (CPU
tensors here, so a call that got past its checks would fail differently)."""

from __future__ import annotations

import pytest
import torch

from kernels import gemm as G

BF = torch.bfloat16


def _t(*shape, dtype=BF):
    return torch.zeros(shape, dtype=dtype)


@pytest.mark.parametrize("x,w,y,msg", [
    (_t(2, 64, dtype=torch.float16), _t(8, 64), _t(2, 8), "x must be bfloat16"),
    (_t(2, 64), _t(8, 72), _t(2, 8), "w must have 64 columns"),
    (_t(2, 64), _t(8, 64, 1)[:, :, 0:1], _t(2, 8), "w must be 2-D"),
    (_t(2, 64), _t(8, 64), _t(3, 8), "y must have 2 rows"),
    (_t(2, 64), _t(8, 64), _t(2, 9), "y must have 8 columns"),
    (_t(64, 2).t(), _t(8, 64), _t(2, 8), "x rows must be contiguous"),
    (_t(2, 64), _t(8, 64), _t(2, 8), "x must be a GPU tensor"),
])
def test_gemm_into_refuses(x, w, y, msg):
    with pytest.raises(ValueError, match=msg):
        G.gemm_into(x, w, y)


def test_other_entry_points_refuse_cpu_tensors():
    x, w, g = _t(2, 64), _t(8, 64), _t(64)
    with pytest.raises(ValueError, match="GPU"):
        G.add_rms_norm(x, _t(2, 64), g, 1e-6)
    with pytest.raises(ValueError, match="one GPU"):
        G.gemm_noalloc(x, w, _t(2, 8))
    sel = G.SkinnySelect(2, 8, 64, "cpu", 1)
    with pytest.raises(ValueError, match="GPU"):
        sel.run(x, w, torch.zeros((2, 1), dtype=torch.int64))
    with pytest.raises(ValueError, match="do not match"):
        G.SkinnyMatmul(3, 8, 64, "cpu")(x, w)
    with pytest.raises(ValueError, match="w_norm"):
        G.add_rms_norm(x, _t(2, 64), _t(72), 1e-6)


def test_projection_objects_check_their_own_sizes():
    """The sizes of a call are the object's M, N and K, whatever else it was
    built with: an object that lacks later attributes (pickled by an earlier
    version), or whose M was changed, refuses what does not fit it."""
    op = G.SkinnyMatmul.__new__(G.SkinnyMatmul)
    op.__dict__.update(M=2, N=8, K=64, config=None, workspace=None, out_cols=8)
    with pytest.raises(ValueError, match="must be a GPU tensor"):
        op(_t(2, 64), _t(8, 64))
    op.M = 3
    with pytest.raises(ValueError, match="do not match"):
        op(_t(2, 64), _t(8, 64))
    for a in (_t(3, 72), _t(3, 64, 1)):
        with pytest.raises(ValueError):
            op(a, _t(8, 64))
