"""The ops in their plain form, in C++ (csrc/host/native.cpp): loads the module, gives it the entry points of the library that _lib
loaded, and hands out its functions as attributes of `native`.

Each of them takes the arguments of the op of that name in ops.py and answers None for anything that is not plain there."""
from __future__ import annotations

import ctypes as C
import importlib.machinery
import importlib.util
from pathlib import Path

from . import _lib

MODULE = "_odysseus_native"
PATH = Path(__file__).resolve().parent / "lib" / f"{MODULE}.so"


def _raise(name: str, status: int) -> None:
    raise _lib.OdysseusHipError(name, status, _lib.load().ody_last_error().decode("utf-8", "replace"))


def _load():
    import torch  # noqa: F401  (the module's symbols are torch's)
    from . import ops
    from .utils.globals import _Arena
    lib = _lib.load()
    if not PATH.exists():
        raise ImportError(f"{PATH} not found: build it with `python -m odysseus_transformer_amd.build`")
    spec = importlib.util.spec_from_loader(MODULE, importlib.machinery.ExtensionFileLoader(MODULE, str(PATH)))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    addresses = {name: C.cast(getattr(lib, name), C.c_void_p).value for name in _lib.SIGNATURES}
    module.bind(addresses, _Arena, ops.scratch, _raise)
    return module


class _Native:
    def __getattr__(self, name):   # the first use of any of them
        if name.startswith("__"):
            raise AttributeError(name)
        module = _load()
        self.__dict__.update({n: getattr(module, n) for n in dir(module) if not n.startswith("_")})
        return self.__dict__[name]


native = _Native()
