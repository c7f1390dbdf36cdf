"""Loader of _omo_native, the native form of the wrappers' ordinary calls
(csrc/binding/omo_native.cpp). Like the kernel library it has no stand-in: a
missing file raises at import, and so does one built for another torch (the
file's suffix names the interpreter)."""
from __future__ import annotations

import importlib.machinery
import importlib.metadata
import importlib.util
import os
import sys
import sysconfig

import torch  # noqa: F401  (its libraries are loaded first)

from . import _abi  # noqa: F401  (and the kernel library the binding calls)

PATH = os.path.join(os.path.dirname(_abi.LIB_PATH), "_omo_native" + sysconfig.get_config_var("EXT_SUFFIX"))
_BUILD = f"`make -C mxfp4-hopper_amd PYTHON={sys.executable}` (or __graft_entry__.build())"


def _load():
    if not os.path.exists(PATH):
        raise ImportError(f"omo: {PATH} is missing; build it with {_BUILD}.")
    loader = importlib.machinery.ExtensionFileLoader("_omo_native", PATH)
    spec = importlib.util.spec_from_file_location("_omo_native", PATH, loader=loader)
    module = importlib.util.module_from_spec(spec)
    loader.exec_module(module)
    if module.torch_version != importlib.metadata.version("torch"):
        raise ImportError(f"omo: {PATH} was built for torch {module.torch_version}, this is "
                          f"{importlib.metadata.version('torch')}; build it again with {_BUILD}.")
    return module


native = _load()
