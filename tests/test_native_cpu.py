"""What the layer's functions do where no native launch is possible: recorded calls, a library
without its extension, a stale library (CPU only)."""

from __future__ import annotations

import shutil
import subprocess
import sys
import warnings

import pytest
import torch
import torch.nn.functional as F


def test_layer_functions_can_be_traced_symbolically(pe):
    """``torch.fx`` records the norms and the gate: a proxy reaches the torch operations, and the
    recorded graph gives their results."""
    x, r, w = torch.randn(5, 32), torch.randn(5, 32), torch.randn(32)

    class Layer(torch.nn.Module):
        def forward(self, x, r, w):
            s, n = pe.ops.add_layer_norm(x, r, w, 1e-5)
            return s, pe.ops.geglu(n), pe.ops.layer_norm(x, w, 1e-5)

    traced = torch.fx.symbolic_trace(Layer())
    s, gated, n = traced(x, r, w)
    a, b = F.layer_norm(x + r, (32,), w, None, 1e-5).chunk(2, -1)
    assert torch.equal(s, x + r) and torch.equal(gated, F.gelu(a) * b)
    assert torch.equal(n, F.layer_norm(x, (32,), w, None, 1e-5))


def test_attention_calls_can_be_traced_symbolically(pe):
    """A recorded attention call is the registered operator."""

    class Layer(torch.nn.Module):
        def forward(self, q, k, v, cu):
            return pe.varlen_attention(q, k, v, cu, 64, window=(64, 64))

    with torch.no_grad():
        graph = torch.fx.symbolic_trace(Layer()).graph
    assert any(node.target == torch.ops.pe_hip.varlen_attention for node in graph.nodes)


def test_layer_functions_compile_as_torchscript(pe):
    x, r, w = torch.randn(5, 32), torch.randn(5, 32), torch.randn(32)
    norm, add, gate = (torch.jit.script(f) for f in (pe.ops.layer_norm, pe.ops.add_layer_norm, pe.ops.geglu))
    want = F.layer_norm(x + r, (32,), w, None, 1e-5)
    s, n = add(x, r, w, 1e-5)
    assert torch.equal(s, x + r) and torch.equal(n, want) and torch.equal(norm(x + r, w, 1e-5), want)
    assert torch.equal(gate(x), F.gelu(x[:, :16]) * x[:, 16:])


def test_a_library_without_its_extension_warns_once(pe, monkeypatch):
    """No ``_pe_torch.so`` beside a built library: no error, the general path, one warning."""
    native = sys.modules[pe.__name__ + "._native"]
    if not native.LIBRARY.exists():
        pytest.skip("the library is not built")
    monkeypatch.setitem(sys.modules, pe.__name__ + "._pe_torch", None)  # its import fails
    monkeypatch.delattr(pe, "_pe_torch", raising=False)
    native._module.cache_clear()
    try:
        with pytest.warns(RuntimeWarning, match="native launches are off"):
            assert native._module() is None
        with warnings.catch_warnings():
            warnings.simplefilter("error")
            assert native._module() is None
    finally:
        native._module.cache_clear()


@pytest.mark.parametrize("version", [None, 8, 9])
def test_a_stale_library_is_an_import_error(pe, tmp_path, version):
    """A library of another ABI, or of this one but built before an entry point was added, is refused
    as the loader promises, whatever it lacks."""
    gcc = shutil.which("gcc")
    if gcc is None:
        pytest.skip("gcc is not available")
    src, lib = tmp_path / "stale.c", tmp_path / "stale.so"
    src.write_text("int pe_other(void) { return 0; }\n" if version is None
                   else f"int pe_attn_abi_version(void) {{ return {version}; }}\n")
    subprocess.run([gcc, "-shared", "-fPIC", str(src), "-o", str(lib)], check=True)
    with pytest.raises(ImportError, match="rebuild it"):
        pe._lib.library.__wrapped__(str(lib))
