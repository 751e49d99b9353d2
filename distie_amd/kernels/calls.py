"""Calls of the kernels' C functions with tensors as arguments (`csrc/calls.cpp`): what every launch costs the host."""

from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import threading

from ..csrc import build

_KINDS = {ctypes.c_void_p: "p", ctypes.c_int: "w", ctypes.c_int64: "w", ctypes.c_float: "f"}
_lock = threading.Lock()
_module = None


def native():
    """The extension module (one a process: Python holds its types)."""
    global _module
    with _lock:
        if _module is None:
            loader = importlib.machinery.ExtensionFileLoader("distie_calls", str(build.ensure("calls")))
            module = importlib.util.module_from_spec(importlib.util.spec_from_loader("distie_calls", loader))
            loader.exec_module(module)
            _module = module
        return _module


def quicken(library: ctypes.CDLL) -> None:
    """The functions of `library` that were declared (`argtypes`) are called without ctypes from now on: a pointer may be a tensor, a
    number or None. Functions with arguments of other types stay as they are."""
    function = native().Function
    for name in [name for name in vars(library) if name.startswith("distie_")]:
        slow = getattr(library, name)
        if not isinstance(slow, function) and slow.restype is ctypes.c_int and slow.argtypes and all(kind in _KINDS for kind in slow.argtypes):
            setattr(library, name, function(slow, ctypes.cast(slow, ctypes.c_void_p).value,
                                            "".join(_KINDS[kind] for kind in slow.argtypes)))
