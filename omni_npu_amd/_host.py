"""Loader of the native host side of the decode steps (csrc/host/mla_host.cpp).

Its functions do a whole stage of a layer - checks, scratch, library GEMM, launches - in one call and answer False, with
nothing launched, where an argument is not what they know; the caller then takes the general path through ``kernels``.
"""
from __future__ import annotations

import importlib.util
import os

from . import _lib

EXT_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_mla_host.so")

_ext = None


def load():
    global _ext
    if _ext is None:
        if not os.path.exists(EXT_PATH):
            raise ImportError(f"{EXT_PATH} is not built; run `python -c 'import __graft_entry__ as g; g.build()'` "
                              "(or `make -C omni_npu_amd/csrc`).")
        _lib.load()
        import torch  # noqa: F401  (the extension links against its libraries)
        spec = importlib.util.spec_from_file_location("_mla_host", EXT_PATH)
        ext = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(ext)
        from . import kernels
        ext.set_workspace(lambda dev, nbytes, tag: kernels._workspace(dev, nbytes, tag))
        _ext = ext
    return _ext
