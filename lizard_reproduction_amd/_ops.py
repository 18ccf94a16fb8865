"""Loader of lizard_torch.so (csrc/torch_ops.cpp): the autograd nodes and the
layer's decode step over the C ABI, built in-tree beside liblizard_hip.so.

As with the library, a missing module raises; nothing falls back to it being
absent.
"""
import importlib.machinery
import importlib.util
import os

import torch

from . import _lib

MODULE = "lizard_torch"
MODULE_PATH = os.path.join(os.path.dirname(_lib.LIB_PATH), MODULE + ".so")

_module = None


def load():
    """The extension module, loaded once (after the library it calls)."""
    global _module
    if _module is None:
        _lib.load()
        if not os.path.exists(MODULE_PATH):
            raise RuntimeError(
                f"{MODULE_PATH} is missing: build it with `python -m lizard_reproduction_amd.build`")
        loader = importlib.machinery.ExtensionFileLoader(MODULE, MODULE_PATH)
        spec = importlib.util.spec_from_file_location(MODULE, MODULE_PATH, loader=loader)
        module = importlib.util.module_from_spec(spec)
        loader.exec_module(module)
        _module = module
    return _module


def plain():
    """Whether a call is an ordinary eager one.  Under a function transform
    (torch.func) or while torch.jit traces, the Python autograd nodes are used:
    they are what those recognise, to trace or to refuse."""
    return (torch._C._functorch.peek_interpreter_stack() is None
            and torch._C._get_tracing_state() is None)
