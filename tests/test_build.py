"""The build's independent parts (gdnr_build.build, compilers replaced): the C
library is written whether or not torch is importable or the host extension
module compiles; a failed compile of either is reported."""

from __future__ import annotations

import sys
from pathlib import Path

import pytest

import gdnr_build


@pytest.fixture
def fake_build(monkeypatch, tmp_path):
    """Compiler calls that write their output; `broken` names a source whose compile fails."""
    broken = []
    for name, at in (("BUILD_DIR", "build"), ("LIBRARY", "lib.so"), ("HOST_MODULE", "host.so")):
        monkeypatch.setattr(gdnr_build, name, tmp_path / at)

    def run(cmd, verbose):
        if any(str(arg).endswith(b) for b in broken for arg in cmd):
            raise RuntimeError(f"build step failed (1): {broken}")
        Path(cmd[cmd.index("-o") + 1]).write_text("built")

    monkeypatch.setattr(gdnr_build, "_run", run)
    return tmp_path, broken


def test_build_writes_both(fake_build):
    out, _ = fake_build
    assert gdnr_build.build() == out / "lib.so"
    assert (out / "lib.so").exists() and (out / "host.so").exists()


def test_library_without_torch(fake_build, monkeypatch):
    out, _ = fake_build
    monkeypatch.setitem(sys.modules, "torch", None)  # (import torch raises ImportError)
    gdnr_build.build()
    assert (out / "lib.so").exists() and not (out / "host.so").exists()


def test_library_when_the_host_module_fails(fake_build):
    out, broken = fake_build
    broken.append("gdnr_host.cpp")
    with pytest.raises(RuntimeError, match="gdnr_host.cpp"):
        gdnr_build.build()
    assert (out / "lib.so").exists() and not (out / "host.so").exists()


def test_a_failed_kernel_writes_nothing(fake_build):
    out, broken = fake_build
    broken.append("gdnr_ring.hip")
    with pytest.raises(RuntimeError, match="gdnr_ring.hip"):
        gdnr_build.build()
    assert not (out / "lib.so").exists()
