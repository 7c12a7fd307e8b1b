"""What relax_amd/build.py does beside compiling: the libraries of the C ABI come out where there is no torch, and the Python extension
is compiled again for another torch."""
import os
import sys

import pytest

from relax_amd import build as b


@pytest.fixture
def small(tmp_path, monkeypatch):
    """A build of two sources whose compiler calls are recorded instead of run."""
    linked, compiled = [], []
    monkeypatch.setattr(b, "OBJDIR", str(tmp_path))
    monkeypatch.setattr(b, "CALLS_LIB", str(tmp_path / "_calls.so"))
    monkeypatch.setattr(b, "CALLS_STAMP", str(tmp_path / "_calls.torch"), raising=False)
    monkeypatch.setattr(b, "sources", lambda: [os.path.join(b.CSRC, n) for n in ("common.cc", "calibrate.hip")])
    monkeypatch.setattr(b, "_compile", lambda src: (tmp_path / (os.path.basename(src) + ".o")).write_text("object"))
    monkeypatch.setattr(b.subprocess, "check_call", lambda cmd: linked.append(cmd[cmd.index("-o") + 1]))

    class Done:
        returncode, stdout, stderr = 0, "", ""

    def run(cmd, **kw):
        compiled.append(cmd)
        (tmp_path / "_calls.so").write_text("extension")
        return Done()

    monkeypatch.setattr(b.subprocess, "run", run)
    return linked, compiled


def test_without_torch_the_libraries_are_built(small, monkeypatch):
    linked, compiled = small
    for name in [n for n in sys.modules if n == "torch" or n.startswith("torch.")]:
        monkeypatch.delitem(sys.modules, name)
    monkeypatch.setitem(sys.modules, "torch", None)  # `import torch` raises ImportError
    assert b.build(verbose=False) == b.LIB
    assert linked == [b.LIB, b.CALIBRATE_LIB] and compiled == []


def test_an_extension_that_does_not_compile_leaves_the_libraries(small, monkeypatch):
    pytest.importorskip("torch")
    linked, _ = small

    class Failed:
        returncode, stdout, stderr = 1, "", "no"

    monkeypatch.setattr(b.subprocess, "run", lambda cmd, **kw: Failed())
    with pytest.raises(RuntimeError):
        b.build(verbose=False)
    assert linked == [b.LIB, b.CALIBRATE_LIB]


def test_another_torch_makes_the_extension_stale(small, monkeypatch):
    pytest.importorskip("torch")
    _, compiled = small
    b.build(verbose=False)
    assert len(compiled) == 1
    b.build(verbose=False, incremental=True)
    assert len(compiled) == 1  # nothing changed
    monkeypatch.setattr(b, "_torch_version", lambda: "0.0.0", raising=False)
    b.build(verbose=False, incremental=True)
    assert len(compiled) == 2
    b.build(verbose=False, incremental=True)
    assert len(compiled) == 2
