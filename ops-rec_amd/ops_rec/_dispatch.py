"""Puts the native dispatcher kernels (``csrc/torch_binding.cpp``) in the place of the Python implementations of ``_ops`` and
``_activation``.

A call in canonical form then never enters Python; any other call is handed to the Python implementation, which holds the
checks and conversions.  Where the binding has not been built the Python implementations stay registered and do everything.
"""

from __future__ import annotations

import importlib.machinery
import importlib.util
import os

from . import _activation, _build, _ops

binding = None


def attach() -> None:
    """Idempotent; does nothing when the binding has not been built."""
    global binding
    if binding is not None or not os.path.exists(_build.BINDING_PATH):
        return
    # the Python kernels leave the dispatcher before the module's static registrations take their places
    _ops._lib_cuda._destroy()
    name = f"{__package__}._torch_binding"
    loader = importlib.machinery.ExtensionFileLoader(name, _build.BINDING_PATH)
    module = importlib.util.module_from_spec(importlib.util.spec_from_file_location(name, _build.BINDING_PATH, loader=loader))
    loader.exec_module(module)
    module.set_fallbacks(_ops._forward_impl, _ops._backward_impl, _ops.hstu_paged, _activation.ln_mul,
                         _activation.distance_in_linear_silu, _activation.in_linear_silu_backward)  # fmt: skip
    _ops._fp8_native = module.fp8_forward
    binding = module


attach()
