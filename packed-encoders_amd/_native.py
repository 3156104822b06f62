"""The native launches (``csrc/pe_torch.cpp``), loaded with the library they call."""

from __future__ import annotations

import warnings
from functools import lru_cache

import torch
from torch import Tensor

from ._build import LIBRARY


@lru_cache(maxsize=1)
def _module():
    """The extension module, or None without a built library or, with a warning, without an extension
    that loads beside it (not built, or built against another library or torch): the same calls then
    go through the torch operators, and the layer's norm and gate through torch."""
    if not LIBRARY.exists():
        return None
    try:
        from . import _pe_torch
    except ImportError as exc:
        warnings.warn(f"native launches are off, calls take the slower general path: {exc}; rebuild with "
                      "__graft_entry__.build()", RuntimeWarning, stacklevel=4)
        return None
    return _pe_torch


def native_for(x: Tensor):
    """The extension module for a call on ``x``, or None where it has nothing to launch: tensors on
    another device, calls that torch compiles, stand-ins that record a call (``torch.fx`` proxies), a
    package without its library or extension."""
    if not isinstance(x, Tensor) or not x.is_cuda or torch.compiler.is_compiling():
        return None
    return _module()
