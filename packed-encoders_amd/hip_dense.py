"""The encoder layer's LayerNorm and GeGLU on the HIP kernels (``csrc/pe_dense.h``).

``layer_norm``, ``add_layer_norm`` and ``geglu`` take the tensors of ``ops``' functions of the same
names and return None for a call the kernels do not serve (``csrc/pe_torch.cpp`` says which), which
``ops`` then runs in torch; so does every call while torch compiles, or without a built library
and extension (the ``"sdpa"`` backend works without either).
"""

from __future__ import annotations

from torch import Tensor

from ._native import native_for


def layer_norm(x: Tensor, weight: Tensor, eps: float) -> Tensor | None:
    native = native_for(x)
    return None if native is None else native.layer_norm(x, None, weight, eps)


def add_layer_norm(x: Tensor, residual: Tensor, weight: Tensor, eps: float) -> tuple[Tensor, Tensor] | None:
    native = native_for(x)
    return None if native is None or residual is None else native.layer_norm(x, residual, weight, eps)


def geglu(proj: Tensor) -> Tensor | None:
    native = native_for(proj)
    return None if native is None else native.geglu(proj)
