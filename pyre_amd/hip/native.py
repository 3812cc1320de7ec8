"""The native half of the binding (``csrc/binding.cpp``): entry points as functions, checks of their operands.

Loaded (and, if need be, compiled) when one of its functions is first called, so that what only plans can be imported where there is
no compiler; it needs no GPU. The kernel library itself is opened at its first use (:mod:`pyre_amd.hip.lib`)."""

from __future__ import annotations

import importlib.machinery
import importlib.util
import threading

import torch  # noqa: F401  (the module is linked against its libraries)

from pyre_amd.hip import build as _build


class KernelError(RuntimeError):
    """A kernel entry point refused its arguments or failed to launch."""


class _Binding:
    """The extension module's functions, which become attributes when the first of them is asked for."""

    def __init__(self):
        self._lock = threading.Lock()
        self._module = None

    def __getattr__(self, name):
        if name.startswith("__"):
            raise AttributeError(name)
        with self._lock:
            if self._module is None:
                path = str(_build.ensure_binding())
                loader = importlib.machinery.ExtensionFileLoader("pyre_binding", path)
                module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("pyre_binding", path, loader=loader))
                loader.exec_module(module)
                module.setup(KernelError)
                self.__dict__.update({k: v for k, v in vars(module).items() if not k.startswith("__")})
                self._module = module
        return getattr(self._module, name)


binding = _Binding()


def late(namespace: dict, alias: str, name: str):
    """A function of the binding for ``namespace[alias]``, which puts the native function into its place at its first call."""

    def first(*args):
        namespace[alias] = fn = getattr(binding, name)
        return fn(*args)

    return first
