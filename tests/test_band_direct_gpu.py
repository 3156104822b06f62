"""Narrow-window calls that run without a plan, every workgroup finding its tile from cu_seqlens: the
bits of the planned (staged) call over segment counts at the edges of the lanes' share, short, empty
and over-long segments, heads and gates; and which calls run so."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,window,causal,gate", [(12, 12, (64, 64), False, False), (4, 2, (3, 200), False, True),
                                                       (8, 2, (250, -1), True, False), (3, 3, (0, 0), False, False)])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 64, 65, 255, 256, 257])
def test_direct_call_equals_the_planned_call(pe, n, hq, hkv, window, causal, gate):
    announce(f"direct band n={n} heads={hq}/{hkv} window={window} causal={causal} gate={gate}")
    rng = np.random.default_rng(n)
    lengths = rng.choice([0, 1, 64, 65, 127, 128, 129, 256, 300, 511], size=n)
    lengths[rng.integers(n)] = 700
    if n > 4:
        lengths[-1] = 900  # past max_seqlen: its rows stay unwritten
    total = int(lengths.sum())
    cu = torch.tensor([0, *np.cumsum(lengths)], dtype=torch.int32, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(n)
    q, k, v, gt = (torch.randn(total, h, 64, generator=g, device="cuda").bfloat16() for h in (hq, hkv, hkv, hq))

    def call():
        return pe.varlen_attention(q, k, v, cu, 700, window=window, causal=causal, gate=gt if gate else None)

    rows = total - (900 if n > 4 else 0)
    with torch.inference_mode():
        direct = call()
        with pe.shared_plans():
            planned = call()
        assert torch.equal(direct[:rows], planned[:rows])
    a, at = int(np.argmax(lengths == 700)), 0  # one segment against the oracle
    at = int(lengths[:a].sum())
    part = slice(at, at + 700)
    want = pe.runtime_attention.oracle_attention(q[part], k[part], v[part], [700], [700], causal, window)
    if gate:
        want = want * torch.sigmoid(gt[part].double())
    assert (direct[part].double() - want).abs().max() <= 2e-2


def test_over_long_segments_stay_unwritten(pe):
    announce("direct band: a segment past max_seqlen")
    cu = torch.tensor([0, 300, 1200, 1400], dtype=torch.int32, device="cuda")
    q = torch.randn(1400, 4, 64, device="cuda").bfloat16()
    out = torch.full_like(q, 7.0)
    from packed_encoders_amd import _lib
    from packed_encoders_amd.hip_attention import _args

    lib = _lib.library()
    a = _args(q, q, q, out, cu, 300, 0.125, 64, 64, False, None, -1)
    size = ctypes.c_size_t()
    assert lib.pe_attn_workspace_size(ctypes.byref(a), ctypes.byref(size)) == 0
    ws = torch.empty(size.value, dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.pe_varlen_attn_fwd(ctypes.byref(a), ws.data_ptr(), size.value, stream) == 0
    torch.cuda.synchronize()
    assert (out[300:1200] == 7.0).all() and not (out[:300] == 7.0).all() and not (out[1200:] == 7.0).all()


# segments, tokens each, query heads, kv heads, head_dim, window, causal, strip, band_kernel: planless or planned
FORMS = {
    "one segment": ((1, 300, 4, 4, 64, (64, 64), False, 0, 0), True),
    "256 segments": ((256, 130, 4, 4, 64, (64, 64), False, 0, 0), True),
    "257 segments": ((257, 130, 4, 4, 64, (64, 64), False, 0, 0), False),
    "window of 256 in all": ((4, 300, 4, 4, 64, (200, 56), False, 0, 0), True),
    "window of 257 in all": ((4, 300, 4, 4, 64, (200, 57), False, 0, 0), False),
    "causal, 256 to the left": ((4, 300, 4, 4, 64, (256, -1), True, 0, 0), True),
    "one side unbounded": ((4, 300, 4, 4, 64, (64, -1), False, 0, 0), False),
    "12,288 query tiles": ((1, 128 * 96, 128, 64, 64, (8, 8), False, 0, 0), True),
    "12,416 query tiles": ((1, 128 * 97, 128, 64, 64, (8, 8), False, 0, 0), False),
    "a strip of two": ((4, 300, 4, 4, 64, (64, 64), False, 2, 0), False),
    "the band kernel": ((4, 300, 4, 4, 64, (64, 64), False, 0, 1), False),
    "head_dim 128": ((4, 300, 4, 4, 128, (64, 64), False, 0, 0), False),
}


@pytest.mark.parametrize("form", FORMS)
def test_which_calls_run_without_a_plan(pe, form):
    """A plan writes the workspace's header, a planless call leaves it alone."""
    from packed_encoders_amd import _lib
    from packed_encoders_amd.hip_attention import _args

    announce(f"direct band: {form}")
    (n, tokens, hq, hkv, d, window, causal, strip, band), direct = FORMS[form]
    cu = torch.arange(0, (n + 1) * tokens, tokens, dtype=torch.int32, device="cuda")
    q, k = (torch.randn(n * tokens, h, d, device="cuda").bfloat16() for h in (hq, hkv))
    out = torch.empty_like(q)
    a = _args(q, k, k, out, cu, tokens, 0.125, *window, causal, None, -1, strip, band_kernel=band)
    lib, size = _lib.library(), ctypes.c_size_t()
    assert lib.pe_attn_workspace_size(ctypes.byref(a), ctypes.byref(size)) == 0
    ws = torch.full((size.value,), 0xFF, dtype=torch.uint8, device="cuda")
    assert lib.pe_varlen_attn_fwd(ctypes.byref(a), ws.data_ptr(), size.value, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    written, needed = ws[:8].view(torch.int32).tolist()
    assert (written, needed) == (-1, -1) if direct else written == needed > 0
