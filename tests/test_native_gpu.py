"""Calls launched natively (csrc/pe_torch.cpp) against the registered torch operators they bypass: the
same bits on every form the native code takes, the operators' errors and copies on the others."""

from __future__ import annotations

import gc
import sys
import threading
import time

import numpy as np
import pytest
import torch

from conftest import announce
from test_random_gpu import _device_inputs, draw_case

pytestmark = pytest.mark.gpu


def _cu(lengths):
    return torch.tensor([0, *np.cumsum(lengths).tolist()], dtype=torch.int32, device="cuda")


def _operator(q, k, v, cu, max_q, gate, cuk, max_k, c, floor):
    options = (c["d"] ** -0.5, *c["window"], c["causal"], gate, -1 if c["short_max"] is None else c["short_max"],
               c["band_kernel"], floor)
    if cuk is None:
        return torch.ops.pe_hip.varlen_attention(q, k, v, cu, max_q, *options)
    return torch.ops.pe_hip.varlen_attention_kv(q, k, v, cu, cuk, max_q, max_k, *options)


@pytest.mark.parametrize("seed", range(40, 64))
def test_attention_equals_the_operator(pe, seed):
    """Seeded calls over the argument space (strided rows, gates, windows, key segments of their own),
    alone and inside a shared_plans scope."""
    c = draw_case(seed)
    announce(f"native attention {c}")
    g = torch.Generator().manual_seed(seed)
    keys = c["keys"] if c["keys"] is not None else c["lengths"]

    def draw(tokens, heads):
        return torch.randn(tokens, heads, c["d"], generator=g).bfloat16()

    T, Tk = sum(c["lengths"]), sum(keys)
    gt = draw(T, c["hq"]) if c["gate"] else None
    q, k, v, gate = _device_inputs(c, draw(T, c["hq"]), draw(Tk, c["hkv"]), draw(Tk, c["hkv"]), gt)
    cu, cuk = _cu(c["lengths"]), None if c["keys"] is None else _cu(keys)
    floor = min(c["lengths"]) if c["bound"] else 0
    with torch.inference_mode():
        want = _operator(q, k, v, cu, max(c["lengths"]), gate, cuk, max(keys), c, floor)

        def call():
            return pe.varlen_attention(q, k, v, cu, max(c["lengths"]), window=c["window"], causal=c["causal"],
                                       gate=gate, short_max=c["short_max"], cu_seqlens_k=cuk,
                                       max_seqlen_k=None if cuk is None else max(keys),
                                       band_kernel=c["band_kernel"], min_seqlen=floor)

        assert torch.equal(call(), want)
        with pe.shared_plans():
            assert torch.equal(call(), want) and torch.equal(call(), want)


@pytest.mark.parametrize("d,h,longest", [(64, 12, 17), (64, 3, 64), (128, 4, 128), (64, 12, 300), (256, 2, 40)])
def test_rope_attention_equals_the_operators(pe, d, h, longest):
    announce(f"native rope attention d={d} h={h} longest={longest}")
    lengths = [longest, 1, 5, longest // 2]
    T, cu = sum(lengths), _cu(lengths)
    g = torch.Generator(device="cuda").manual_seed(d + longest)
    qkv = torch.randn(1, T, 3 * h * d, generator=g, device="cuda").bfloat16()
    cos, sin = (t[0, :T] for t in pe.ops.rope_tables(max(T, 512), d, 10000.0, torch.device("cuda"), torch.bfloat16))
    with torch.inference_mode():
        q, k = torch.ops.pe_hip.rope_qkv(qkv, cos, sin, h, d)
        v = qkv.view(1, T, 3, h, d)[0, :, 2]
        want = torch.ops.pe_hip.varlen_attention(q[0], k[0], v, cu, longest, d ** -0.5, 8, 8, False, None, -1)
        got_q, got_k = pe.hip_attention.rope_qkv(qkv, h, d, cos, sin)
        assert torch.equal(got_q, q) and torch.equal(got_k, k)
        for tables in ((cos, sin), (cos[None], sin[None])):
            got = pe.ops.flash_attention_qkv_bshd(qkv, h, d, cos=tables[0], sin=tables[1], window=(8, 8),
                                                  scaling=d ** -0.5, cu_seqlens=cu, max_seqlen=longest)
            assert got.shape == (1, T, h * d) and torch.equal(got.view(T, h, d), want)


def test_other_calls_reach_the_operators(pe):
    """Layouts that need a copy give the copy's result; bad calls raise the operators' errors."""
    announce("native attention: other calls")
    lengths = [40, 200, 7]
    T, cu = sum(lengths), _cu(lengths)
    q = torch.randn(T, 4, 64, device="cuda").bfloat16()
    odd = torch.randn(T, 260, device="cuda").bfloat16()[:, :256].unflatten(1, (4, 64))  # rows off 16 bytes
    off = torch.randn(T * 256 + 1, device="cuda").bfloat16()[1:].view(T, 4, 64)  # contiguous, but off 16 bytes
    with torch.inference_mode():
        assert torch.equal(pe.varlen_attention(odd, q, q, cu, 200), pe.varlen_attention(odd.clone(), q, q, cu, 200))
        assert pe.varlen_attention(q[:0], q[:0], q[:0], cu, 200).shape == (0, 4, 64)
        for bad in ((q.float(), q, q, cu), (off, q, q, cu), (q, q[:-1], q[:-1], cu), (q, q[:, :3], q[:, :3], cu), (q, q, q, cu.long()),
                    (q[:, :, :48], q[:, :, :48], q[:, :, :48], cu), (q, q, q, cu[None])):
            with pytest.raises(ValueError):
                pe.varlen_attention(*bad, 200)
        with pytest.raises(ValueError):
            pe.varlen_attention(q, q, q, cu, 200, rope=(q[:, 0], q[:, 0]))  # a segment past the short kernel
    with pytest.raises(ValueError):
        pe.varlen_attention(q.clone().requires_grad_(), q, q, cu, 200)


def test_compiled_and_transformed_calls_see_the_operator(pe):
    """Under a dispatch mode the call is the registered operator, as before."""
    from torch.utils._python_dispatch import TorchDispatchMode

    announce("native attention under a dispatch mode")
    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    q, cu = torch.randn(50, 4, 64, device="cuda").bfloat16(), _cu([20, 30])
    with torch.inference_mode():
        want = pe.varlen_attention(q, q, q, cu, 30)
    with torch.no_grad(), Watch():
        got = pe.varlen_attention(q, q, q, cu, 30)
    assert torch.equal(got, want) and any("pe_hip" in name for name in seen)


def _launches(pe):
    """One call of every native launch, by name."""
    h, d, T = 4, 64, 40
    x, w = torch.randn(T, 512, device="cuda").bfloat16(), torch.ones(512, device="cuda").bfloat16()
    qkv = torch.randn(1, T, 3 * h * d, device="cuda").bfloat16()
    q, k, v = (qkv.view(T, 3, h, d)[:, i] for i in range(3))
    positions, cu = torch.arange(T, device="cuda"), _cu([T])
    cos, sin = (t[0] for t in pe.ops.rope_tables(T, d, 10000.0, torch.device("cuda"), torch.bfloat16))
    return {
        "layer_norm": lambda: pe.hip_dense.layer_norm(x, w, 1e-5),
        "geglu": lambda: pe.hip_dense.geglu(x),
        "rope_rows": lambda: pe.ops.rope_rows(positions, T, d, 10000.0, torch.bfloat16),
        "rope": lambda: pe.hip_attention.rope_qkv(qkv, h, d, cos, sin),
        "attention": lambda: pe.varlen_attention(q, k, v, cu, T),
        "attention_qkv": lambda: pe.hip_attention.attention_qkv(qkv, h, d, cos, sin, cu, T, window=(-1, -1),
                                                                softmax_scale=0.125),
    }


@pytest.mark.parametrize("name", ["layer_norm", "geglu", "rope_rows", "rope", "attention", "attention_qkv"])
def test_other_threads_run_during_a_launch(pe, name):
    """A launch or an allocation that has to wait must not stop the process's other Python threads: the
    native calls give the interpreter lock up around both. With a switch interval that never passes,
    another thread runs only where the calling one lets go by itself."""
    announce(f"interpreter lock during {name}")
    ran, stop = [0], threading.Event()

    def other():
        while not stop.is_set():
            ran[0] += 1
            time.sleep(0)  # lets go and asks again

    with torch.inference_mode():
        call = _launches(pe)[name]
        assert call() is not None
        torch.cuda.synchronize()
        thread = threading.Thread(target=other)
        interval = sys.getswitchinterval()
        sys.setswitchinterval(1000.0)
        gc.disable()  # freeing a tensor lets go too: none is collected, the outputs are kept
        try:
            thread.start()
            before, outs = ran[0], []
            while ran[0] == before and len(outs) < 20000:
                outs.append(call())
            during = ran[0] - before
        finally:
            gc.enable()
            sys.setswitchinterval(interval)
            stop.set()
            thread.join()
        torch.cuda.synchronize()
    assert during > 0


def test_calls_without_the_extension_take_the_general_path(pe, monkeypatch):
    """A built library without ``_pe_torch.so``: the layer's norm and gate run in torch, attention
    through the registered operators with the bits of the native launch."""
    announce("calls without the extension")
    native = sys.modules[pe.__name__ + "._native"]
    x, w = torch.randn(40, 512, device="cuda").bfloat16(), torch.ones(512, device="cuda").bfloat16()
    q, cu = torch.randn(40, 4, 64, device="cuda").bfloat16(), _cu([10, 30])
    with torch.inference_mode():
        want = pe.varlen_attention(q, q, q, cu, 30)
        monkeypatch.setitem(sys.modules, pe.__name__ + "._pe_torch", None)
        monkeypatch.delattr(pe, "_pe_torch", raising=False)
        native._module.cache_clear()
        try:
            with pytest.warns(RuntimeWarning, match="native launches are off"):
                got = pe.ops.layer_norm(x, w, 1e-5)
            assert torch.equal(got, torch.nn.functional.layer_norm(x, (512,), w, None, 1e-5))
            assert torch.equal(pe.ops.geglu(x), torch.nn.functional.gelu(x[:, :256]) * x[:, 256:])
            assert torch.equal(pe.varlen_attention(q, q, q, cu, 30), want)
        finally:
            native._module.cache_clear()
