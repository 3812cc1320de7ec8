"""The native half of the binding (``csrc/binding.cpp``): entry points as functions, checks of their operands.

Loaded (and, if need be, compiled) when the kernels' functions are imported; it needs no GPU. The kernel library itself is opened at its
first use (:mod:`pyre_amd.hip.lib`)."""

from __future__ import annotations

import importlib.machinery
import importlib.util

import torch  # noqa: F401  (the module is linked against its libraries)

from pyre_amd.hip import build as _build


class KernelError(RuntimeError):
    """A kernel entry point refused its arguments or failed to launch."""


def _load():
    path = str(_build.ensure_binding())
    loader = importlib.machinery.ExtensionFileLoader("pyre_binding", path)
    module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("pyre_binding", path, loader=loader))
    loader.exec_module(module)
    module.setup(KernelError)
    return module


binding = _load()
