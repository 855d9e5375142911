"""Compiles and runs a C++ program against the headers of ``akv_amd/csrc``
that host and device code share (no GPU)."""

import shutil
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "akv_amd" / "csrc"


def run(tmp_path, source, *flags):
    """The program's output; its failures (nonzero status) raise."""
    cxx = next(c for c in ("g++", "clang++", "/opt/rocm/bin/amdclang++") if shutil.which(c))
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(source)
    built = subprocess.run([cxx, "-std=c++17", "-O2", "-Wall", *flags, f"-I{CSRC}", str(src), "-o", str(exe)],
                           capture_output=True, text=True)
    assert built.returncode == 0, built.stderr
    ran = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert ran.returncode == 0, ran.stdout + ran.stderr
    return ran.stdout
