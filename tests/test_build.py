"""The HIP library's build fails when a source fails to compile.

A copy of the package's Makefile, csrc/ and include/ is built in a temporary
directory with every object already present (empty stand-ins, newer than
their sources), then one source gets a syntax error: make must return
non-zero, leave no object for that source and not relink the library.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import time
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
PKG = ROOT / "montlok.cpp_amd"


@pytest.mark.skipif(not Path("/opt/rocm/bin/hipcc").exists(), reason="hipcc not installed")
def test_make_fails_on_a_broken_source(tmp_path):
    pkg = tmp_path / "pkg"
    (pkg / "_build").mkdir(parents=True)
    shutil.copy(PKG / "Makefile", pkg / "Makefile")
    shutil.copytree(PKG / "csrc", pkg / "csrc")
    shutil.copytree(ROOT / "include", tmp_path / "include")
    lib = pkg / "montlok" / "rdt" / "lib" / "libmlk_hip.so"
    lib.parent.mkdir(parents=True)
    past = time.time() - 3600
    for src in list((pkg / "csrc").iterdir()) + list((tmp_path / "include").iterdir()):
        os.utime(src, (past, past))
    for src in (pkg / "csrc").glob("*.hip"):
        (pkg / "_build" / f"{src.stem}.o").write_bytes(b"stale object")
    lib.write_bytes(b"stale library")
    # Only status.o is older than its source now; its compile must fail the build.
    with open(pkg / "csrc" / "status.hip", "a") as f:
        f.write("\nthis is not C++ ;\n")
    out = subprocess.run(["make", "-C", str(pkg)], capture_output=True, text=True, timeout=300)
    assert out.returncode != 0, out.stdout + out.stderr
    assert "hipcc failed" in out.stderr
    assert not (pkg / "_build" / "status.o").exists()
    assert lib.read_bytes() == b"stale library"


def test_build_entry_raises_on_make_failure(monkeypatch):
    import __graft_entry__ as ge

    def fake_run(*a, **k):
        return subprocess.CompletedProcess(a, 2, "", "hipcc failed (1)")

    monkeypatch.setattr(ge.subprocess, "run", fake_run)
    with pytest.raises(RuntimeError, match="failed"):
        ge._make("-C", str(PKG))


def _dry_run(*args):
    return subprocess.run(["make", "-n", "-C", str(PKG), *args], capture_output=True, text=True, timeout=120)


def test_the_library_builds_without_torch():
    """Without torch (here: without a Python at all) make builds the C ABI and says what it left out; with torch, both."""
    bare = _dry_run("-B", "PYTHON=/nonexistent/python3")
    assert bare.returncode == 0, bare.stderr
    assert "libmlk_hip.so" in bare.stdout and "torch_ops.cpp" not in bare.stdout and "is not built" in bare.stdout
    assert "torch_ops.cpp" not in _dry_run("-B", "lib").stdout
    full = _dry_run("-B", f"PYTHON={sys.executable}")
    assert full.returncode == 0 and "torch_ops.cpp" in full.stdout and "compiled_with_cxx11_abi" in full.stdout


def test_the_extension_follows_torch(tmp_path):
    """Built already, it is built again when the torch or the Python it was built against changes, and only then."""
    pkg = tmp_path / "pkg"
    (pkg / "_build").mkdir(parents=True)
    shutil.copy(PKG / "Makefile", pkg / "Makefile")
    shutil.copytree(PKG / "csrc", pkg / "csrc")
    shutil.copytree(ROOT / "include", tmp_path / "include")
    ops = pkg / "montlok" / "rdt" / "lib" / "_torch_ops.so"
    ops.parent.mkdir(parents=True)
    env = pkg / "_build" / "torch_ops.env"
    cxx = tmp_path / "cxx"  # writes its output and compiles nothing
    cxx.write_text('#!/bin/sh\nwhile [ $# -gt 0 ]; do [ "$1" = -o ] && echo built > "$2"; shift; done\n')
    cxx.chmod(0o755)

    def make(*args):
        out = subprocess.run(["make", "-C", str(pkg), f"PYTHON={sys.executable}", f"CXX={cxx}", *args], capture_output=True,
                             text=True, timeout=300)
        assert out.returncode == 0, out.stderr
        return out.stdout

    assert "torch_ops.cpp" in make("ops") and ops.read_text() == "built\n"
    assert len(env.read_text().split()) == 4
    assert "torch_ops.cpp" not in make("ops")
    env.write_text("/another/torch /another/python 2.0 3.9\n")
    assert "torch_ops.cpp" in make("ops")
    assert "torch_ops.cpp" not in make("ops")
