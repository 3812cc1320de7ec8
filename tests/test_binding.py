"""The native half of the binding: what it refuses it refuses as the checks in Python did, and an entry's own refusal comes with the
library's message. No kernel runs here."""

from __future__ import annotations

import re
import shutil
import subprocess
import sys
import textwrap
from pathlib import Path

import pytest
import torch

from pyre_amd.hip import lib
from pyre_amd.hip.native import KernelError, binding


def test_checks_of_operands():
    t = torch.zeros(4, 6)
    assert binding.dev() is None and binding.dev(None) is None
    with pytest.raises(KernelError, match="not on a GPU"):
        binding.dev(None, t)
    with pytest.raises(TypeError):
        binding.dev(3)
    binding.contig("rows", t)
    with pytest.raises(KernelError, match="rows must be contiguous"):
        binding.contig("rows", t.t())
    ids = torch.zeros(5, dtype=torch.int32)
    binding.i32("ids", ids), binding.i32("ids", ids, 5), binding.i32("ids", ids, None)
    with pytest.raises(KernelError, match="ids holds 5 entries, 6 needed"):
        binding.i32("ids", ids, 6)
    with pytest.raises(KernelError, match="ids must be int32"):
        binding.i32("ids", ids.long())
    with pytest.raises(KernelError, match="ids must be contiguous"):
        binding.i32("ids", torch.zeros(6, dtype=torch.int32)[::2])
    assert [binding.dtype_code(x) for x in (t, torch.float32, torch.bfloat16, t.bfloat16())] == [0, 0, 1, 1]
    with pytest.raises(KernelError, match="unsupported element type"):
        binding.dtype_code(torch.float16)
    assert binding.ptr(None) is None and binding.ptr(t[1:]) == t.data_ptr() + 24
    assert not binding.sums(t, 24)  # not on a GPU
    with pytest.raises(KernelError, match="not on a GPU"):
        binding.product(t, t, 4)


def test_partial_sums():
    d, bias = torch.zeros(3, 4, 6), torch.zeros(6, dtype=torch.bfloat16)
    assert binding.partials(d, None, 6) == (d.data_ptr(), 0, 3, 24, None, 0)
    assert binding.partials(d, bias, 6) == (d.data_ptr(), 0, 3, 24, bias.data_ptr(), 1)
    with pytest.raises(KernelError, match="6 wide, 8 expected"):
        binding.partials(d, None, 8)
    with pytest.raises(KernelError, match="5 entries, 6 expected"):
        binding.partials(d, bias[:5], 6)


def test_entries():
    lib.lib()
    with pytest.raises(KernelError, match="M=0"):  # the library's own refusal
        lib.call("pyre_gemm_mid_bf16", None, 64, None, 64, None, 0, 64, 64, 1, 0, 0)
    with pytest.raises(KernelError, match="not on a GPU"):
        lib.call("pyre_gemm_mid_bf16", torch.zeros(4, 4), 64, None, 64, None, 0, 64, 64, 1, 0, 0)
    with pytest.raises(TypeError, match="takes 11 arguments, 10 given"):
        lib.call("pyre_gemm_mid_bf16", None, 64, None, 64, None, 0, 64, 64, 1, 0)
    with pytest.raises(TypeError):
        lib.call("pyre_gemm_mid_bf16", None, 64.5, None, 64, None, 0, 64, 64, 1, 0, 0)
    with pytest.raises(OverflowError):
        lib.call("pyre_gemm_mid_bf16", None, 64, None, 64, None, 1 << 40, 64, 64, 1, 0, 0)
    with pytest.raises(AttributeError):
        lib.call("pyre_no_such_entry")


def test_an_exception_in_an_entry_is_an_error_of_the_call(tmp_path):
    """A library whose entries throw (out of memory, say): the interpreter's lock is free while they run and held again when the
    error is made. In a process of its own, since the library takes the kernels' place."""
    compiler = shutil.which("g++")
    if compiler is None:
        pytest.skip("no C++ compiler")
    from pyre_amd.hip import build

    names = re.findall(r"X\((\w+)\)", (build.CSRC / "binding.cpp").read_text())
    assert "gemm_mid_bf16" in names
    source = tmp_path / "throws.cpp"
    source.write_text("#include <new>\n" + 'extern "C" const char* pyre_last_error() { return ""; }\n' +
                      "".join(f'extern "C" int pyre_{n}() {{ throw std::bad_alloc(); }}\n' for n in names))
    lib_path = tmp_path / "libthrows.so"
    subprocess.run([compiler, "-shared", "-fPIC", str(source), "-o", str(lib_path)], check=True)
    code = textwrap.dedent(f"""
        import threading
        from pyre_amd.hip.native import binding
        binding.open({str(lib_path)!r})
        def once():
            for _ in range(50):
                try:
                    binding.pyre_scale(None, 0, 1.0, None)
                except RuntimeError as e:
                    assert "bad_alloc" in str(e), e
                else:
                    raise SystemExit("no error")
        others = [threading.Thread(target=once) for _ in range(3)]
        [t.start() for t in others]
        once()
        [t.join() for t in others]
        print("held")
    """)
    done = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300,
                          cwd=Path(build.CSRC).parent.parent)
    assert done.returncode == 0 and "held" in done.stdout, (done.returncode, done.stderr[-2000:])


def without_compilers(tmp_path):
    import os

    return {**os.environ, "PYRE_AMD_BUILD_DIR": str(tmp_path / "empty"), "CXX": "/nowhere/g++", "HIPCC": "/nowhere/hipcc", "PATH": str(tmp_path)}


def test_what_plans_is_imported_without_a_compiler(tmp_path):
    """Nothing built, no compiler: the package imports and plans; the first check of an operand says what is missing."""
    code = textwrap.dedent("""
        import torch
        import pyre_amd.api, pyre_amd.parts.fast
        from pyre_amd.hip import build, ops
        from pyre_amd.parts.attention_work import decode_capacity
        assert decode_capacity(8, 28, 4) > 8 and ops.attn_biased_tile_plan(4, 6, 1, 600)
        for f in (lambda: ops.dtype_code(torch.float32), lambda: ops._dev(torch.zeros(1))):
            try:
                f()
            except build.BuildError as e:
                assert "no C++ compiler" in str(e), e
            else:
                raise SystemExit("no error")
    """)
    done = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300, env=without_compilers(tmp_path),
                          cwd=Path(lib.__file__).parents[2])
    assert done.returncode == 0, done.stderr[-2000:]


def test_the_binding_is_stale_when_it_would_be_compiled_otherwise(monkeypatch):
    from pyre_amd.hip import build

    digests = {build._binding_digest()}
    with monkeypatch.context() as m:
        m.setattr(build, "BINDING_FLAGS", [*build.BINDING_FLAGS, "-g"])
        digests.add(build._binding_digest())
    monkeypatch.setenv("CXX", "another-compiler")
    digests.add(build._binding_digest())
    assert len(digests) == 3


def test_the_binding_is_compiled_without_hipcc(monkeypatch, tmp_path):
    from pyre_amd.hip import build

    def missing():
        raise build.BuildError("hipcc not found")

    monkeypatch.setattr(build, "_hipcc", missing)
    command = build._binding_command(tmp_path / "x.so")
    assert command[0] == build._cxx() and any(c.endswith("/include") and Path(c[2:]).joinpath("hip").exists() for c in command if c.startswith("-I"))


def test_functions_of_the_binding_take_their_names_at_the_first_call():
    from pyre_amd.hip import ops

    assert ops.dtype_code(torch.bfloat16) == 1 and ops.dtype_code is binding.dtype_code
