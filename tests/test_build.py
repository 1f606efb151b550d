"""The build without compilers: what it links when the optional native call
module cannot be built, and what it refuses."""

from __future__ import annotations

import importlib.util
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _remarks(*sizes):
    """As the compiler reports them, one kernel per size of scratch."""
    return "".join(f"a.hip:3:1: remark: Function Name: kernel{i} [-Rpass-analysis]\n"
                   f"a.hip:3:1: remark:     ScratchSize [bytes/lane]: {v} [-Rpass-analysis]\n"
                   f"a.hip:3:1: remark:     SGPRs Spill: 0 [-Rpass-analysis]\n"
                   for i, v in enumerate(sizes))


@pytest.fixture
def build(tmp_path, monkeypatch):
    """build.py with every output under tmp_path and commands that only write
    their -o file; ``build.fail``: substrings of commands that fail."""
    spec = importlib.util.spec_from_file_location(
        "mxfp4_build_under_test", os.path.join(ROOT, "mxfp4-gfx936_amd", "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    for name in ("LIB", "PROBE_LIB", "HOST_LIB"):
        monkeypatch.setattr(mod, name, str(tmp_path / os.path.basename(getattr(mod, name))))
    monkeypatch.setattr(mod, "OBJ_DIR", str(tmp_path))
    monkeypatch.setattr(mod, "GEN_DIR", str(tmp_path))
    mod.fail = ()
    mod.remarks = _remarks(0, 0)

    def run(cmd, **kw):
        if any(f in c for f in mod.fail for c in cmd):
            return subprocess.CompletedProcess(cmd, 1, "", "made to fail")
        open(cmd[cmd.index("-o") + 1], "w").close()
        return subprocess.CompletedProcess(cmd, 0, "", mod.remarks)

    monkeypatch.setattr(mod.subprocess, "run", run)
    return mod


def test_library_is_built_without_torch(build, monkeypatch, capsys):
    monkeypatch.setitem(sys.modules, "torch", None)
    assert build.build() == build.LIB and os.path.exists(build.LIB)
    assert not os.path.exists(build.HOST_LIB) and "_host.so is not built" in capsys.readouterr().out


def test_failing_host_compiler_is_reported_after_the_library(build):
    build.fail = ("mxfp4_host.cpp",)
    with pytest.raises(RuntimeError, match="mxfp4_host.cpp"):
        build.build()
    assert os.path.exists(build.LIB) and os.path.exists(build.PROBE_LIB)


@pytest.mark.parametrize("remarks,what", [(_remarks(0, 24, 0), r"kernel1 \(24 bytes/lane\)"),
                                          ("", "no resource usage")])
def test_scratch_in_a_kernel_that_counts_loads_fails_the_build(build, remarks, what):
    assert all(os.path.exists(os.path.join(build.CSRC, f)) for f in build.NO_SCRATCH)
    build.remarks = remarks
    with pytest.raises(RuntimeError, match=what):
        build.build()
    assert not os.path.exists(build.LIB)
