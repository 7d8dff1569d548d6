"""The C library is built without torch and whatever becomes of the torch operators."""
import importlib.util
import os
import subprocess

import pytest

from chronicals_amd import build as _build


@pytest.fixture
def compilers(tmp_path, monkeypatch):
    """Compilers that write an empty output, in a library folder of their own; those named in `failing` fail."""
    failing = set()
    monkeypatch.setattr(_build, "LIB_DIR", str(tmp_path))
    monkeypatch.setattr(_build, "LIB_PATH", str(tmp_path / _build.LIB_NAME))
    monkeypatch.setattr(_build, "RESOURCES_PATH", str(tmp_path / "resources.txt"))

    def run(cmd, **kwargs):
        if os.path.basename(cmd[0]) in failing:
            return subprocess.CompletedProcess(cmd, 1, "", "")
        open(cmd[cmd.index("-o") + 1], "w").close()
        return subprocess.CompletedProcess(cmd, 0, "", "")
    monkeypatch.setattr(subprocess, "run", run)
    return failing


def test_the_c_library_stays_when_the_operators_fail(compilers):
    compilers.add("g++")
    with pytest.raises(RuntimeError, match="g\\+\\+"):
        _build.build()
    assert os.path.exists(_build.LIB_PATH)


def test_the_c_library_builds_without_torch(compilers, monkeypatch, capsys):
    find = importlib.util.find_spec
    monkeypatch.setattr(importlib.util, "find_spec", lambda name, *a: None if name == "torch" else find(name, *a))
    assert _build.build() == _build.LIB_PATH and os.path.exists(_build.LIB_PATH)
    assert "operators are not built" in capsys.readouterr().err
    monkeypatch.undo()


def test_both_libraries_are_built(compilers):
    _build.build()
    assert sorted(n for n in os.listdir(_build.LIB_DIR) if n.endswith(".so")) == sorted(
        [_build.LIB_NAME, os.path.basename(_build.torch_lib_path())])
