"""Registers what runs for device tensors: the native dispatcher kernels (``csrc/torch_binding.cpp``), or the Python
implementations of ``_ops`` and ``_activation``.

With the native kernels a call in canonical form never enters Python; any other call is handed to the Python implementation, which
holds the checks and conversions.  Where the binding has not been built, or does not load (built for another torch), the Python
implementations are registered and do everything.
"""

from __future__ import annotations

import importlib.machinery
import importlib.util
import logging
import os

import torch

from . import _activation, _build, _ops

logger = logging.getLogger(__name__)

binding = None
_lib = None


def _load():
    name = f"{__package__}._torch_binding"
    loader = importlib.machinery.ExtensionFileLoader(name, _build.BINDING_PATH)
    module = importlib.util.module_from_spec(importlib.util.spec_from_file_location(name, _build.BINDING_PATH, loader=loader))
    loader.exec_module(module)  # (its static registrations put the native kernels into the dispatcher)
    module.set_fallbacks(_ops._forward_impl, _ops._backward_impl, _ops.hstu_paged, _activation.ln_mul,
                         _activation.distance_in_linear_silu, _activation.in_linear_silu_backward)  # fmt: skip
    return module


def attach() -> None:
    """Called once, when the package is imported."""
    global binding, _lib
    if os.path.exists(_build.BINDING_PATH):
        try:
            binding = _load()
            _ops._fp8_native = binding.fp8_forward
            return
        except Exception as err:  # noqa: BLE001  (the operators work without it)
            logger.warning("%s does not load (%s): the operators run through their Python implementations", _build.BINDING_PATH, err)
    _lib = torch.library.Library("ops_rec", "IMPL", "CUDA")
    for name, fn in _ops._PYTHON_KERNELS.items():
        _lib.impl(name, fn)


attach()
