"""The LayerNorm (with the residual add) and GeGLU kernels against float64, and the calls they leave
to torch."""

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


def test_geglu_of_every_bf16_value(pe):
    announce("geglu of every bf16 value")
    bits = torch.arange(1 << 16, dtype=torch.int32, device="cuda").to(torch.int16)
    x = bits.view(torch.bfloat16).view(-1, 64)
    with torch.no_grad():
        out = pe.ops.geglu(torch.cat((x, torch.ones_like(x)), -1))
        torch_out = F.gelu(x)
    want = F.gelu(x.double())
    lower = x.double() * torch.special.erfc(x.double().abs() * 0.5 ** 0.5) * 0.5  # the negative tail's own digits
    want = torch.where(x < 0, lower, want)
    fine = x.isfinite()
    err = (out.double() - want).abs()
    # the output's rounding; the power of two's argument, up to 150, carries three fp32 roundings (150 * 3 *
    # 2^-24 * ln 2 < 2^-15); Phi(x) under 2^-126 may be flushed to zero, |x| times that in the product
    flushed = 2.0 ** -126 * x.double().abs().clamp(min=1)
    assert (err[fine] <= ((HALF_STEP + 2.0 ** -15) * want.abs() + flushed)[fine]).all()
    assert torch.equal(out[~fine].isnan(), torch_out[~fine].isnan())
    assert torch.equal(out[x == float("inf")], x[x == float("inf")])


@pytest.mark.parametrize("rows,width", [(1, 8), (7, 16), (3, 1152), (100, 1152), (31, 2624), (1000, 24)])
def test_geglu_matches_float64(pe, rows, width):
    announce(f"geglu {rows} x {width}")
    proj = _bf16(2, rows, 2 * width, seed=width, std=2.0)
    with torch.no_grad():
        out = pe.ops.geglu(proj)
    a, b = proj.double().chunk(2, -1)
    want = F.gelu(a) * b
    assert out.shape == want.shape
    assert ((out.double() - want).abs() <= (HALF_STEP + 2.0 ** -15) * want.abs() + 1e-12).all()


def test_other_calls_run_in_torch(pe):
    """Calls the kernels do not serve give torch's own results."""
    announce("dense calls left to torch")
    w = _bf16(768)
    for x in (_bf16(4, 768).float(), _bf16(4, 1536)[:, ::2], _bf16(4 * 768 + 1)[1:].view(4, 768), _bf16(4, 768).cpu()):
        ww = w.to(x.device, x.dtype)
        assert pe.hip_dense.layer_norm(x, ww, 1e-5) is None
        assert pe.hip_dense.add_layer_norm(x, x, ww, 1e-5) is None and pe.hip_dense.geglu(x) is None
        assert torch.equal(pe.ops.layer_norm(x, ww, 1e-5), F.layer_norm(x, (768,), ww, None, 1e-5))
        assert torch.equal(pe.ops.geglu(x), F.gelu(x[..., :384]) * x[..., 384:])
    x = _bf16(4, 768)
    assert pe.hip_dense.layer_norm(x[:, :12], w[:12], 1e-5) is None and pe.hip_dense.geglu(_bf16(4, 24)) is None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert pe.ops.layer_norm(x, w, 1e-5).dtype == F.layer_norm(x, (768,), w, None, 1e-5).dtype
    x.requires_grad_()
    pe.ops.geglu(pe.ops.add_layer_norm(x, x, w, 1e-5)[1]).sum().backward()
    assert x.grad is not None
    y = _bf16(3, 4, 768)
    batched = torch.func.vmap(lambda t: pe.ops.geglu(pe.ops.layer_norm(t, w, 1e-5)))(y)
    each = torch.stack([F.gelu(n[:, :384]) * n[:, 384:] for n in F.layer_norm(y, (768,), w, None, 1e-5)])
    assert torch.equal(batched, each)


def test_batched_derivatives_reach_the_torch_operations(pe):
    """The batching that ``is_grads_batched`` and vectorised derivatives use hands backward functions
    tensors without storage: they go to torch, as those of ``torch.func.vmap`` do."""
    announce("batched derivatives")
    w = _bf16(768)

    class Gate(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x.clone()

        @staticmethod
        def backward(ctx, grad):
            return pe.ops.layer_norm(grad, w, 1e-5)

    x, grads = _bf16(4, 768).requires_grad_(), _bf16(3, 4, 768, seed=1)
    got = torch.autograd.grad(Gate.apply(x), x, grads, is_grads_batched=True)[0]
    assert torch.equal(got, F.layer_norm(grads, (768,), w, None, 1e-5))


@pytest.mark.parametrize("d,theta", [(64, 160000.0), (64, 10000.0), (128, 10000.0), (256, 500.0)])
def test_rope_rows_are_the_gathered_tables(pe, d, theta):
    announce(f"rope rows d={d} theta={theta}")
    positions = torch.cat([torch.arange(n) for n in (1, 7, 8192, 300)]).cuda()
    cos, sin = pe.ops.rope_rows(positions, 8192, d, theta, torch.bfloat16)
    tables = pe.ops.rope_tables(8192, d, theta, torch.device("cuda"), torch.bfloat16)
    for got, table in ((cos, tables[0]), (sin, tables[1])):
        assert torch.equal(got, table[0].index_select(0, positions)[None])
    half = pe.ops.rope_rows(positions, 8192, d, theta, torch.float32)[0]  # another type: the tables' path
    assert half.dtype == torch.float32 and torch.equal(half.bfloat16(), cos)


@pytest.mark.parametrize("d", [64, 128, 256])
def test_rope_rows_outside_the_table_are_nan(pe, d):
    """Positions past ``max_seqlen`` or negative have no table row to gather: no angles come out for them."""
    announce(f"rope rows outside the table d={d}")
    positions = torch.tensor([0, 99, 100, 5, -1, 1 << 40, -(1 << 62), 42], device="cuda")
    outside = torch.tensor([False, False, True, False, True, True, True, False], device="cuda")
    for got, table in zip(pe.ops.rope_rows(positions, 100, d, 10000.0, torch.bfloat16),
                          pe.ops.rope_tables(100, d, 10000.0, torch.device("cuda"), torch.bfloat16)):
        assert torch.equal(got[0, ~outside], table[0].index_select(0, positions[~outside]))
        assert got[0, outside].isnan().all()
    with pytest.raises(IndexError):
        pe.ops.rope_rows(positions.cpu(), 100, d, 10000.0, torch.bfloat16)
