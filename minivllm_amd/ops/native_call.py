"""How the kernel libraries' launchers are called: through ``_launch.so`` (``csrc/pyext/launch.cpp``), which makes a call of
25 arguments in 0.4 us, or, where it cannot be built or loaded (no Python headers, no x86-64), through ctypes, which takes
3 to 5.  The library is built on first use like the kernel libraries."""
from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import os

_PATH = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "_launch.so")


def _load():
    try:
        if not os.path.exists(_PATH):
            from minivllm_amd import build
            build.build_launch(verbose=False)
        loader = importlib.machinery.ExtensionFileLoader("_launch", _PATH)
        module = importlib.util.module_from_spec(importlib.util.spec_from_loader("_launch", loader))
        loader.exec_module(module)
        return module
    except Exception:                      # noqa: BLE001  (ctypes takes the calls)
        return None


_native = _load()
_LETTERS = {ctypes.c_void_p: "p", ctypes.c_int: "i", ctypes.c_long: "i", ctypes.c_uint64: "i", ctypes.c_float: "f"}


def bind(lib: ctypes.CDLL, name: str, argtypes, restype=ctypes.c_int):
    """The function ``name`` of ``lib`` as a callable; ``restype`` ``c_int`` or ``c_long``.  Pointers are Python ints or None."""
    f = getattr(lib, name)
    f.argtypes = list(argtypes)
    f.restype = restype
    if _native is None or not all(t in _LETTERS for t in argtypes):
        return f
    letters = "".join(_LETTERS[t] for t in argtypes)
    return _native.bind(ctypes.cast(f, ctypes.c_void_p).value, letters + ("L" if restype is ctypes.c_long else "I"))
