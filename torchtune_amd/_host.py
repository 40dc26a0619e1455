"""The native host path (``csrc/host_binding.cpp``): layer calls with their checks, allocations and autograd nodes in C++.

Like the HIP library it is built by ``python -m torchtune_amd.build`` and required: there is nothing to fall back to."""
from __future__ import annotations

import importlib.util
import threading
from pathlib import Path

import torch

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


class _TracedCall(torch.autograd.Function):
    """A host call as one node of a ``torch.jit.trace``, which records Python nodes but not native ones.  Backward: the call
    again, differentiated."""

    @staticmethod
    def forward(ctx, name: str, *args):
        ctx.name, ctx.rest = name, [None if isinstance(a, torch.Tensor) else (a,) for a in args]
        ctx.save_for_backward(*(a for a in args if isinstance(a, torch.Tensor)))
        return getattr(load(), name)(*args)

    @staticmethod
    def backward(ctx, *grads):
        saved = iter(ctx.saved_tensors)
        with torch.enable_grad():
            args = [next(saved).detach().requires_grad_(need) if a is None else a[0]
                    for a, need in zip(ctx.rest, ctx.needs_input_grad[1:])]
            outs = getattr(load(), ctx.name)(*args)
            need = [a for a, n in zip(args, ctx.needs_input_grad[1:]) if n]
            got = iter(torch.autograd.grad(outs, need, grads if isinstance(outs, tuple) else grads[0], allow_unused=True))
        return (None, *(next(got) if n else None for n in ctx.needs_input_grad[1:]))


def tracing() -> bool:
    return torch._C._get_tracing_state() is not None


def call(name: str, *args):
    """The host function ``name``; under ``torch.jit.trace`` as a node the trace can hold."""
    return _TracedCall.apply(name, *args) if tracing() else getattr(load(), name)(*args)
