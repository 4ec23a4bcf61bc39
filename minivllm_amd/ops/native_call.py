"""How the kernel libraries' launchers are called: through an extension module (``csrc/pyext/launch.cpp``), which makes a call of
25 arguments in 0.4 us, or, where it cannot be built or loaded (no Python headers, no compiler, no x86-64), through ctypes, which
takes 3 to 5, with a warning.  The module is built on first use like the kernel libraries; its name says which source and which
interpreter it is for (``build.launch_lib``)."""
from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import warnings

from minivllm_amd import build


def _load():
    why = "it cannot be built here"
    try:
        path = build.build_launch(verbose=False)
        if path:
            loader = importlib.machinery.ExtensionFileLoader("_launch", path)
            module = importlib.util.module_from_spec(importlib.util.spec_from_loader("_launch", loader))
            loader.exec_module(module)
            return module
    except Exception as e:                 # noqa: BLE001  (ctypes takes the calls)
        why = str(e)
    warnings.warn(f"kernels are launched through ctypes, 3 to 5 us a call slower than by the launchers' module: {why}")
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
