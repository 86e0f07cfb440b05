"""Loader of the native host path (csrc/host.cpp, built into `_host.so`).

`matmul`, `routing`, `view`, `int_views`, `reduce`, `downcast` and `upcast` are the extension's functions once it is loaded,
which the first call does.  Each answers None for a call it does not cover; the caller then runs its general path."""
import ctypes
import os

import torch

from . import _lib

HOST_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_host.so")


def load():
    """Loads the extension and hands it the library's addresses; raises if it has not been built, or for another torch: it is
    compiled against torch's headers and reads tensors in place."""
    import importlib.machinery
    import importlib.util

    from .matmul_details import opt_flags
    from .tensor import FP4, Tensor
    from .tensor_details.layout import CDNA4MXScaleLayout, CDNA4MXValueLayout
    lib = _lib.lib()
    if not os.path.exists(HOST_PATH):
        raise RuntimeError(f"{HOST_PATH} is missing: build it with `python -m triton_amd.build`")
    loader = importlib.machinery.ExtensionFileLoader("triton_amd._host", HOST_PATH)
    host = importlib.util.module_from_spec(importlib.util.spec_from_file_location("triton_amd._host", HOST_PATH, loader=loader))
    try:
        loader.exec_module(host)
        built_for = host.built_for
    except (ImportError, AttributeError) as e:  # (a symbol of another torch is missing, or a file from before the check)
        built_for = f"another torch ({e})"
    if built_for != str(torch.__version__):
        raise RuntimeError(f"{HOST_PATH} was built for torch {built_for}, this is {torch.__version__}: build it again with "
                           "`python -m triton_amd.build`")
    addresses = {n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value
                 for n in ("tamd_matmul_sized", "tamd_routing_gates", "tamd_reduce", "tamd_downcast_mxfp", "tamd_upcast_mxfp")}
    host.init(addresses, Tensor, CDNA4MXValueLayout, CDNA4MXScaleLayout, FP4, opt_flags._opt_flags_constraints,
              opt_flags._opt_flags)
    for name in _FUNCTIONS:
        globals()[name] = getattr(host, name)
    return host


def _on_first_call(name):
    def call(*args):
        load()
        return globals()[name](*args)
    return call


_FUNCTIONS = ("matmul", "routing", "view", "int_views", "reduce", "downcast", "upcast", "choose_block_m", "blocks_of_16_stream",
              "dense_block_m", "ring_rows", "routing_block_rows")
for _n in _FUNCTIONS:
    globals()[_n] = _on_first_call(_n)
