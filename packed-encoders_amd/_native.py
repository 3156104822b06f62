"""The native launches (``csrc/pe_torch.cpp``), loaded with the library they call."""

from __future__ import annotations

from functools import lru_cache

import torch
from torch import Tensor

from ._build import LIBRARY


@lru_cache(maxsize=1)
def _module():
    """The extension module, or None without a built library; ``ImportError`` for a library built
    without its extension."""
    if not LIBRARY.exists():
        return None
    from . import _pe_torch

    return _pe_torch


def native_for(x: Tensor):
    """The extension module for a call on ``x``, or None where it has nothing to launch: tensors on
    another device, calls that torch compiles, stand-ins that record a call (``torch.fx`` proxies), a
    package without its library."""
    if not isinstance(x, Tensor) or not x.is_cuda or torch.compiler.is_compiling():
        return None
    return _module()
