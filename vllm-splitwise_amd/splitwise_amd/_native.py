"""``_step_ops`` (csrc/host/step_ops.cpp): the operators of small steps called without Python's share of a call.  Where it is not
built, or was built against another torch, Python or interface, nothing is taken and the functions of ``_C`` / ``_C_mixers`` do
everything."""
from __future__ import annotations

import ctypes
import glob
import importlib
import os
import warnings

import torch

# the extension reads tensors through torch's inline code: only the build that it was compiled against has that layout
_TORCH = f"{torch.__version__} {torch.version.git_version}"


class _NotBuilt:
    def __getattr__(self, name):
        if name.startswith("__") or name.isupper():
            raise AttributeError(name)
        return lambda *args: None


def _load():
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_step_ops*.so")
    try:
        found = importlib.import_module("._step_ops", __package__)
    except ImportError as error:
        if glob.glob(path):
            warnings.warn(f"{path} does not load and is not used, rebuild it (`make step-ops`): {error}")
        return _NotBuilt()
    if getattr(found, "TORCH", None) != _TORCH:
        warnings.warn(f"{found.__file__} was built for torch {getattr(found, 'TORCH', 'unknown')}, this is {_TORCH}: it is not used, "
                      "rebuild it (`make step-ops`)")
        return _NotBuilt()
    return found


step_ops = _load()


def bind_library(lib: ctypes.CDLL, names, version: int, constant: str) -> None:
    """Tells the extension where ``lib``'s entry points are."""
    if getattr(step_ops, constant, version) != version:
        warnings.warn(f"{step_ops.__file__} was built for another interface of the libraries and is not used, rebuild it "
                      "(`make step-ops`)")
    elif not isinstance(step_ops, _NotBuilt):
        step_ops.bind({name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in names})
