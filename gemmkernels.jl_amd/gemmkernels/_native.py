"""The module between torch tensors and the library (csrc/gk_torch.cpp): what a call that was seen before does, in C++.  ``load()`` gives it bound to the library, or
None where it was not built for this interpreter and its torch; the package's own Python then does the same."""
from __future__ import annotations

import ctypes
import importlib.util
import os
import sys
from typing import Optional

from . import _lib
from ._built_for import built_for

_PATH = os.path.join(os.path.dirname(_lib.LIB_PATH), "gk_torch.so")


class Prepared:
    """A launch that has passed every check but those of its addresses (gk_prepare), or one without a handle where the library makes none.
    (The bias of an epilogue is the caller's to keep.)"""

    __slots__ = ("handle", "_free")

    def __init__(self, conf_c, trans, epi, code: int):
        handle = ctypes.c_void_p()
        lib = _lib.lib()
        rc = lib.gk_prepare(ctypes.byref(conf_c), ctypes.byref(trans) if trans is not None else None, ctypes.byref(epi) if epi is not None else None, code,
                            ctypes.byref(handle))
        self.handle = handle.value if rc == _lib.GK_OK else None
        self._free = lib.gk_prepared_free

    def __del__(self):
        if getattr(self, "handle", None):
            self._free(self.handle)
            self.handle = None


_module = None
_tried = False


def _built_for_of(path: str) -> Optional[str]:
    try:
        return ctypes.string_at(ctypes.addressof(ctypes.c_char.in_dll(ctypes.CDLL(path), "gk_torch_built_for"))).decode()
    except (OSError, ValueError):               # (not to be linked here; a module that does not say)
        return None


def load():
    global _module, _tried
    if not _tried and "torch" in sys.modules:                # (without it there are no tensors to read, and nothing to link against)
        lib = _lib.lib()
        _tried = True
        if os.path.exists(_PATH):
            try:
                # (looked at before any of it runs: it would read the tensors of another torch at wrong offsets)
                what = _built_for_of(_PATH)
                if what is None or what != built_for():
                    return None
                spec = importlib.util.spec_from_file_location("gk_torch", _PATH)
                module = importlib.util.module_from_spec(spec)
                spec.loader.exec_module(module)
            except ImportError:
                return None
            address = lambda fn: ctypes.cast(fn, ctypes.c_void_p).value
            module.bind(*(address(fn) for fn in (lib.gk_matmul, lib.gk_matmul_sliced, lib.gk_matmul_split_k, lib.gk_stream_capture, lib.gk_run)))
            _module = module
    return _module
