"""The short kernel at its key capacities' edges (32, 64, 96 and 128 keys), with and without the fused
RoPE, whose workgroups take fewer heads from 64 keys on."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


def _inputs(h, d, longest, seed):
    lengths = [longest, 1, 33, 0, longest - 1, 64, 97, 2, 31] * 40  # two or four heads per workgroup, too
    lengths = [min(n, longest) for n in lengths]
    g = torch.Generator(device="cuda").manual_seed(seed)
    qkv = torch.randn(sum(lengths), 3, h, d, generator=g, device="cuda").bfloat16()
    gate = torch.randn(sum(lengths), h, d, generator=g, device="cuda").bfloat16()
    return lengths, torch.tensor([0, *np.cumsum(lengths)], dtype=torch.int32, device="cuda"), qkv, gate


@pytest.mark.parametrize("longest", [64, 65, 95, 96, 97, 128])
@pytest.mark.parametrize("d,h,window", [(64, 12, (-1, -1)), (64, 5, (20, 20)), (128, 8, (-1, -1)), (128, 3, (0, 70))])
def test_capacity_edges(pe, d, h, window, longest):
    announce(f"short capacity d={d} h={h} window={window} longest={longest}")
    lengths, cu, qkv, gate = _inputs(h, d, longest, seed=d + longest)
    q, k, v = qkv.unbind(1)
    with torch.inference_mode():
        got = pe.varlen_attention(q, k, v, cu, longest, window=window, gate=gate)
        # the tables in one row per token, and in fewer rows than the batch or a segment has tokens
        for rows in (sum(lengths), 130, 50):
            cos, sin = (t[0] for t in pe.ops.rope_tables(rows, d, 10000.0, torch.device("cuda"), torch.bfloat16))
            rq, rk = pe.hip_attention.rope_qkv(qkv.view(-1, 3 * h * d), h, d, cos, sin)
            want = pe.varlen_attention(rq, rk, v, cu, longest, window=window, gate=gate)
            assert torch.equal(pe.varlen_attention(q, k, v, cu, longest, window=window, gate=gate, rope=(cos, sin)), want)
    n = sum(lengths[:9])  # one cycle of the lengths against the oracle
    exact = pe.runtime_attention.oracle_attention(q[:n], k[:n], v[:n], lengths[:9], lengths[:9], False, window)
    exact = exact * torch.sigmoid(gate[:n].double())
    assert (got[:n].double() - exact).abs().max() <= 2e-2
    assert torch.nn.functional.cosine_similarity(got[:n].double().flatten(1), exact.flatten(1)).min() >= 0.9999
