"""The native launch sequences of the fused layers (`csrc/host/host.cpp`, built as
`_qlora_host.so` beside this file): whole forwards and backwards of a projection group or of the
MLP in one call. There is no Python stand-in: a missing module raises, as a missing kernel
library does.
"""

from __future__ import annotations

import importlib.machinery
import importlib.util
import ctypes
import threading
from pathlib import Path

from . import _lib

MODULE_PATH = Path(__file__).resolve().parent / "_qlora_host.so"

_module = None
_bound = None  # the kernel library whose entry points the module calls
_lock = threading.Lock()


def load():
    """The module, bound to the loaded kernel library's entry points."""
    global _module, _bound
    lib = _lib.load()
    if _bound is lib:
        return _module
    with _lock:
        if _module is None:
            if not MODULE_PATH.exists():
                raise _lib.KernelLibraryMissing(
                    f"{MODULE_PATH.name} is not built: run `python -m hackathon_amd.build` "
                    f"(expected at {MODULE_PATH})")
            name = "_qlora_host"
            loader = importlib.machinery.ExtensionFileLoader(name, str(MODULE_PATH))
            spec = importlib.util.spec_from_file_location(name, MODULE_PATH, loader=loader)
            module = importlib.util.module_from_spec(spec)
            loader.exec_module(module)
            version = getattr(module, "abi_version", None)
            if version != _lib.ABI_VERSION:
                raise _lib.KernelLibraryMissing(
                    f"{MODULE_PATH.name} was built for C-ABI version {version}, the kernel "
                    f"library has {_lib.ABI_VERSION}: rebuild both with "
                    f"`python -m hackathon_amd.build`")
            _module = module
        _module.bind([ctypes.cast(getattr(lib, n), ctypes.c_void_p).value
                      for n in _module.entry_names()])
        _bound = lib
    return _module
