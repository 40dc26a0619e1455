"""The native host path (``csrc/host_binding.cpp``): layer calls with their checks, allocations and autograd nodes in C++.

Like the HIP library it is built by ``python -m torchtune_amd.build`` and required: there is nothing to fall back to."""
from __future__ import annotations

import importlib.util
import threading
from pathlib import Path

from . import _lib

MODULE_NAME = "torchtune_amd_host"
MODULE_PATH = Path(__file__).resolve().parent / "lib" / f"{MODULE_NAME}.so"

_lock = threading.Lock()
_module = None


def load():
    """The extension module, loaded once."""
    global _module
    if _module is None:
        with _lock:
            if _module is None:
                _lib.load()  # the C ABI the extension is linked against
                if not MODULE_PATH.exists():
                    raise _lib.LibraryNotBuiltError(f"{MODULE_PATH} is missing. Build it with `python -m torchtune_amd.build`.")
                spec = importlib.util.spec_from_file_location(MODULE_NAME, MODULE_PATH)
                module = importlib.util.module_from_spec(spec)
                spec.loader.exec_module(module)
                _module = module
    return _module
