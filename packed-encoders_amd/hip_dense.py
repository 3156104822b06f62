"""The encoder layer's LayerNorm and GeGLU on the HIP kernels (``csrc/pe_dense.h``).

``layer_norm``, ``add_layer_norm`` and ``geglu`` take the tensors of ``ops``' functions of the same
names and return None for a call the kernels do not serve (``csrc/pe_torch.cpp`` says which), which
``ops`` then runs in torch; so does every call while torch compiles, or without a built library
(the ``"sdpa"`` backend works without one).
"""

from __future__ import annotations

from functools import lru_cache

import torch
from torch import Tensor

from ._build import LIBRARY


@lru_cache(maxsize=1)
def _native():
    """The extension module, or None without a built library; ``ImportError`` for a library built
    without its extension."""
    if not LIBRARY.exists():
        return None
    from . import _pe_torch

    return _pe_torch


def _off(x: Tensor) -> bool:
    return not x.is_cuda or torch.compiler.is_compiling() or _native() is None


def layer_norm(x: Tensor, weight: Tensor, eps: float) -> Tensor | None:
    return None if _off(x) else _native().layer_norm(x, None, weight, eps)


def add_layer_norm(x: Tensor, residual: Tensor, weight: Tensor, eps: float) -> tuple[Tensor, Tensor] | None:
    return None if _off(x) or residual is None else _native().layer_norm(x, residual, weight, eps)


def geglu(proj: Tensor) -> Tensor | None:
    return None if _off(proj) else _native().geglu(proj)
