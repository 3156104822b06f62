"""The LayerNorm kernel (with the residual add) against float64, and the calls it leaves to torch."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from conftest import announce

pytestmark = pytest.mark.gpu

HALF_STEP = 2.0 ** -8  # bf16 keeps 8 significant bits: rounding to nearest is off by at most 2^-8 of the value


def _bf16(*shape, seed=0, std=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, generator=g, device="cuda") * std).bfloat16()


# 8-column pieces per lane: 1 (<= 512), 2 (<= 1024), 4 (<= 2048), 8 (<= 4096), each at both edges
@pytest.mark.parametrize("rows,cols", [(1, 8), (3, 504), (4, 512), (5, 520), (257, 768), (33, 1024), (9, 1032),
                                       (4, 2048), (6, 2056), (5, 4096)])
@pytest.mark.parametrize("residual", [False, True])
def test_layer_norm_matches_float64(pe, rows, cols, residual):
    announce(f"layer norm {rows} x {cols} residual={residual}")
    x = _bf16(rows, cols, seed=rows, std=3.0) + 5.0  # a mean well off zero
    r = _bf16(rows, cols, seed=cols)
    w = _bf16(cols, seed=7)
    assert pe.hip_dense.layer_norm(x, w, 1e-5) is not None  # the kernel's call
    with torch.no_grad():
        if residual:
            s, out = pe.ops.add_layer_norm(x, r, w, 1e-5)
            assert torch.equal(s, x + r)
        else:
            s, out = x, pe.ops.layer_norm(x, w, 1e-5)
    want = F.layer_norm(s.double(), (cols,), w.double(), None, 1e-5)
    # the output's own rounding, and fp32 arithmetic on deviations of values near 20 in size
    err = (out.double() - want).abs()
    assert (err <= HALF_STEP * want.abs() + 1e-5 * w.double().abs() + 1e-38).all(), err.max()


def test_layer_norm_of_extreme_rows(pe):
    announce("layer norm of extreme rows")
    cols = 768
    x = _bf16(4, cols)
    x[0] = 2.0  # no variance
    x[1, 5] = float("inf")
    x[2, 3] = float("nan")
    x[3] *= 1e30  # squares overflow: the deviations vanish against an infinite variance
    w = torch.ones(cols, device="cuda").bfloat16()
    with torch.no_grad():
        out = pe.ops.layer_norm(x, w, 1e-5)
    assert (out[0] == 0).all() and out[1].isnan().all() and out[2].isnan().all() and (out[3] == 0).all()


def test_other_calls_run_in_torch(pe):
    """Calls the kernels do not serve give torch's own results."""
    announce("dense calls left to torch")
    w = _bf16(768)
    for x in (_bf16(4, 768).float(), _bf16(4, 1536)[:, ::2], _bf16(4 * 768 + 1)[1:].view(4, 768), _bf16(4, 768).cpu()):
        ww = w.to(x.device, x.dtype)
        assert pe.hip_dense.layer_norm(x, ww, 1e-5) is None
        assert pe.hip_dense.add_layer_norm(x, x, ww, 1e-5) is None
        assert torch.equal(pe.ops.layer_norm(x, ww, 1e-5), F.layer_norm(x, (768,), ww, None, 1e-5))
    x = _bf16(4, 768)
    assert pe.hip_dense.layer_norm(x[:, :12], w[:12], 1e-5) is None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert pe.ops.layer_norm(x, w, 1e-5).dtype == F.layer_norm(x, (768,), w, None, 1e-5).dtype
    x.requires_grad_()
    pe.ops.add_layer_norm(x, x, w, 1e-5)[1].sum().backward()
    assert x.grad is not None
    y = _bf16(3, 4, 768)
    batched = torch.func.vmap(lambda t: pe.ops.layer_norm(t, w, 1e-5))(y)
    assert torch.equal(batched, F.layer_norm(y, (768,), w, None, 1e-5))
