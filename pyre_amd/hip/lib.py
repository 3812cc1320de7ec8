"""The kernel library: opened, checked against this tree's sources, its entry points as functions.

The library is loaded (and, if need be, compiled) at the first use of ``lib()``.
There is no fallback: if it cannot be built or loaded, the caller gets the error.
"""

from __future__ import annotations

import ctypes
from ctypes import c_float, c_int, c_long, c_void_p

from pyre_amd.hip import build as _build
from pyre_amd.hip.native import KernelError, binding

ABI_VERSION = 31


P, I, L, F = c_void_p, c_int, c_long, c_float

#: entry points that answer a question about sizes; those that put work on the stream are in the native binding
_SIGNATURES = {
    "pyre_attn_generic_spans": [I],
    "pyre_attn_mfma_supports": [I, I, I, I],
    "pyre_attn_decode_work_rope_supports": [I, I, I, I, L],
    "pyre_attn_prefill_waves": [I, I],
    "pyre_compute_units": [],
    "pyre_gemm_skinny_supports": [I, I, I, L, L],
    "pyre_gemm_mid_supports": [I, I, I, L, L],
    "pyre_gemm_mid_silu_blocks": [I, I],
    "pyre_gemm_f32_adds": [I, I, I, L, L, I],
    "pyre_gemm_f32_tile_choice": [I, I, I, I],
    "pyre_gemm_f32_tile_mixed": [I, I, I, I],
    "pyre_gemm_tile_supports": [I, I, I, L, L],
    "pyre_gemm_tile_parts": [I, I, I],
    "pyre_attn_biased_spans": [I, I, I, I],
    "pyre_gla_chunks_scratch": [I, I, I, I, I],
    "pyre_latent_attn_spans": [I, I],
    "pyre_latent_heads_supports": [I, I, I],
}

_lib = None


def _open(path) -> ctypes.CDLL:
    handle = ctypes.CDLL(str(path))
    handle.pyre_last_error.restype = ctypes.c_char_p
    handle.pyre_abi_version.restype = c_int
    return handle


def _fits(handle) -> bool:
    """The library speaks this binding's ABI and was compiled from the sources of this tree."""
    if handle.pyre_abi_version() != ABI_VERSION or not hasattr(handle, "pyre_sources_digest"):
        return False
    handle.pyre_sources_digest.restype = ctypes.c_char_p
    return handle.pyre_sources_digest().decode() == _build.sources_digest()


def lib() -> ctypes.CDLL:
    global _lib
    if _lib is None:
        handle = _open(_build.ensure_built())
        if not _fits(handle):
            # A library from other sources under a stamp that says otherwise (a copied build
            # folder, an older checkout): rebuild once. The loader keeps the mapping of a path
            # it has already opened, so the new build is opened under a name of its own.
            import os
            import shutil

            path = _build.build(force=True)
            fresh = path.with_name(f"{path.stem}.{os.getpid()}{path.suffix}")
            shutil.copyfile(path, fresh)
            try:
                handle = _open(fresh)
                binding.open(str(fresh))
            finally:
                os.unlink(fresh)
            if not _fits(handle):
                raise KernelError(f"kernel library has ABI {handle.pyre_abi_version()} and the binding expects "
                                  f"{ABI_VERSION}, or it does not carry the digest of the sources it was built "
                                  "from: sources and binding are out of step")
        for name, argtypes in _SIGNATURES.items():
            fn = getattr(handle, name)
            fn.argtypes = argtypes
            fn.restype = c_int
        binding.open(handle._name)
        _lib = handle
    return _lib


def loaded_path() -> str | None:
    return None if _lib is None else _lib._name


_entry_points: dict = {}


def call(name: str, *args) -> None:
    """Put an entry point's work on the stream; tensors stand for their memory. Raises :class:`KernelError` with the library's message."""
    fn = _entry_points.get(name)
    if fn is None:
        lib()
        fn = _entry_points[name] = getattr(binding, name)
    fn(*args)
