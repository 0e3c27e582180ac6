"""Loads csrc/_khan_ops.so, the tensor side of `khan_amd.ops` in native code (csrc/torch_ops.cpp): checks, allocation and
the call into libkhan_aev.so.  There is no Python version of it: a missing module raises."""
import importlib.machinery
import importlib.util
import os

from . import _lib

PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc", "_khan_ops.so")
_module = None


def load():
    global _module
    if _module is None:
        if not os.path.exists(PATH):
            raise _lib.KhanError("%s is missing: build it with `python -m khan_amd.build` (g++, the installed torch)" % PATH)
        import torch  # noqa: F401  (its libraries have to be in the process before the module is)
        _lib.load()   # says what is missing in a form that helps
        loader = importlib.machinery.ExtensionFileLoader("_khan_ops", PATH)
        module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("_khan_ops", PATH, loader=loader))
        loader.exec_module(module)
        module.init(_lib.LIB_PATH, _lib.KhanError)
        _module = module
    return _module
