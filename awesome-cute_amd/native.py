"""Loads the HIP library (libmarlin_amd.so, a C ABI) and the tensor calls over it
(_marlin_torch.so), both built in-tree.  A missing one is an import-time error:
nothing here has another implementation."""
import ctypes
import importlib.machinery
import importlib.util
import os

import torch  # noqa: F401  (its libraries have to be loaded before the binding)

_HERE = os.path.dirname(os.path.abspath(__file__))


def _path(name):
    path = os.path.join(_HERE, name)
    if not os.path.exists(path):
        raise ImportError(
            f"{path} is missing: build it first (python __graft_entry__.py build, or "
            "python awesome-cute_amd/build.py); the GEMMs have no other implementation")
    return path


def _binding():
    loader = importlib.machinery.ExtensionFileLoader("_marlin_torch", _path("_marlin_torch.so"))
    module = importlib.util.module_from_spec(
        importlib.util.spec_from_file_location("_marlin_torch", loader.path, loader=loader))
    loader.exec_module(module)
    return module


lib = ctypes.CDLL(_path("libmarlin_amd.so"))
torch_binding = _binding()
