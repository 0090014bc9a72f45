"""The ops in their plain form, in C++ (csrc/host/native.cpp): loads the module, gives it the entry points of the library that _lib
loaded, and hands out its functions as attributes of `native`.

Each of them takes the arguments of the op of that name in ops.py and answers None for anything that is not plain there.  The module
saves host time and nothing else.  Where it is missing, or was built for another torch (it is tied to one build of it, as the kernels'
library is not), each of them answers None to everything, after one warning: the Python in ops.py calls the same kernels.
ODYSSEUS_NATIVE_LIB names a module in another place, as ODYSSEUS_HIP_LIB does for the kernels' library."""
from __future__ import annotations

import ctypes as C
import importlib.machinery
import importlib.util
import os
import warnings
from pathlib import Path

from . import _lib

MODULE = "_odysseus_native"
PATH = Path(__file__).resolve().parent / "lib" / f"{MODULE}.so"


def _raise(name: str, status: int) -> None:
    raise _lib.OdysseusHipError(name, status, _lib.load().ody_last_error().decode("utf-8", "replace"))


def _load():
    """The module, or None with a warning."""
    import torch
    from . import ops
    from .utils.globals import _Arena
    lib = _lib.load()
    path = Path(os.environ.get("ODYSSEUS_NATIVE_LIB", PATH))
    try:
        spec = importlib.util.spec_from_loader(MODULE, importlib.machinery.ExtensionFileLoader(MODULE, str(path)))
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
        if module.TORCH_VERSION != str(torch.__version__):
            raise ImportError(f"built for torch {module.TORCH_VERSION}, this is {torch.__version__}")
    except ImportError as e:
        warnings.warn(f"{path} cannot be used ({e}): the ops take their path through Python, at 10 us more of host time each.  "
                      "`python -m odysseus_transformer_amd.build` builds it.", RuntimeWarning, stacklevel=4)
        return None
    addresses = {name: C.cast(getattr(lib, name), C.c_void_p).value for name in _lib.SIGNATURES}
    module.bind(addresses, _Arena, ops.scratch, _raise, torch.OutOfMemoryError, lambda: ops._never_keeps_ds(), lambda *args: ops.attn_bwd(*args))
    return module


class _Nothing:
    """Stands for a module that cannot be used."""

    def __getattr__(self, name):
        if name.startswith("__"):
            raise AttributeError(name)
        answer = self.__dict__[name] = lambda *args: None
        return answer


class _Native:
    _stands_in = None

    def __getattr__(self, name):   # the first use of any of them; of each of them, without the module
        if name.startswith("__"):
            raise AttributeError(name)
        if self._stands_in is None:
            module = _load()
            if module is not None:
                self.__dict__.update({n: getattr(module, n) for n in dir(module) if not n.startswith("_")})
                return self.__dict__[name]
            self._stands_in = _Nothing()
        answer = self.__dict__[name] = getattr(self._stands_in, name)
        return answer


native = _Native()
