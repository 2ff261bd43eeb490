"""``_step_ops`` (csrc/host/step_ops.cpp): the operators of small steps called without Python's share of a call.  Where it is not
built, or was built against another interface, nothing is taken and the functions of ``_C`` / ``_C_mixers`` do everything."""
from __future__ import annotations

import ctypes

import torch  # noqa: F401  (the extension links against its libraries)

try:
    from . import _step_ops as step_ops
except ImportError:
    class _NotBuilt:
        def __getattr__(self, name):
            if name.startswith("__"):
                raise AttributeError(name)
            return lambda *args: None
    step_ops = _NotBuilt()


def bind_library(lib: ctypes.CDLL, names, version: int, constant: str) -> None:
    """Tells the extension where ``lib``'s entry points are."""
    if getattr(step_ops, constant, None) == version:
        step_ops.bind({name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in names})
