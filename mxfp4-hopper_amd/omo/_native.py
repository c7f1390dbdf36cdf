"""Loader of _omo_native.so, the native form of the wrappers' ordinary calls
(csrc/binding/omo_native.cpp). Like the kernel library it has no stand-in: a
missing file raises at import."""
from __future__ import annotations

import importlib.machinery
import importlib.util
import os

import torch  # noqa: F401  (its libraries are loaded first)

from . import _abi  # noqa: F401  (and the kernel library the binding calls)

PATH = os.path.join(os.path.dirname(_abi.LIB_PATH), "_omo_native.so")


def _load():
    if not os.path.exists(PATH):
        raise ImportError(f"omo: {PATH} is missing; build it with `make -C mxfp4-hopper_amd` "
                          "(or __graft_entry__.build()).")
    loader = importlib.machinery.ExtensionFileLoader("_omo_native", PATH)
    spec = importlib.util.spec_from_file_location("_omo_native", PATH, loader=loader)
    module = importlib.util.module_from_spec(spec)
    loader.exec_module(module)
    return module


native = _load()
