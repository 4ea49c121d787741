"""The build (no compiler runs here): what is left when the torch extension cannot be built."""

from __future__ import annotations

import importlib.util
from pathlib import Path

import pytest

import __graft_entry__


@pytest.fixture
def build(monkeypatch, tmp_path):
    """build.py with its outputs in tmp_path and commands that only write their output file;
    those named in `fail` raise."""
    spec = importlib.util.spec_from_file_location("_build_under_test", __graft_entry__.PKG_DIR / "build.py")
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    for name in ("LIB_PATH", "CALIB_LIB_PATH", "TORCH_LIB_PATH"):
        monkeypatch.setattr(module, name, tmp_path / getattr(module, name).name)
    monkeypatch.setattr(module, "BUILD", tmp_path / "_build")
    monkeypatch.setattr(module, "hipcc", lambda: "hipcc")
    module.fail = set()

    def run(cmd):
        if cmd[0] in module.fail or ("-shared" in cmd and cmd[0] + " link" in module.fail):
            raise RuntimeError(f"{cmd[0]} failed")
        Path(cmd[cmd.index("-o") + 1]).write_text("new")

    monkeypatch.setattr(module, "_run", run)
    module.TORCH_LIB_PATH.write_text("old")
    return module


def test_everything_is_built(build):
    assert build.build(require_torch_ext=True) == build.LIB_PATH
    for path in (build.LIB_PATH, build.CALIB_LIB_PATH, build.TORCH_LIB_PATH):
        assert path.read_text() == "new"


@pytest.mark.parametrize("fails", ["no g++", "link", "no torch"])
def test_the_library_needs_no_torch_extension(build, monkeypatch, fails):
    """The library is built, no extension of an earlier library stays beside it, and the
    failure is reported, or raised where the extension is asked for."""
    if fails == "no torch":
        def commands():
            raise ImportError("No module named 'torch'")

        monkeypatch.setattr(build, "_torch_commands", commands)
    else:
        build.fail = {"g++" if fails == "no g++" else "g++ link"}
    with pytest.warns(RuntimeWarning, match="_anima_torch.so is left out"):
        assert build.build() == build.LIB_PATH
    assert build.LIB_PATH.read_text() == build.CALIB_LIB_PATH.read_text() == "new"
    assert not build.TORCH_LIB_PATH.exists()
    with pytest.raises((RuntimeError, ImportError)):
        build.build(require_torch_ext=True)


def test_a_failed_library_build_raises(build):
    build.fail = {"hipcc"}
    with pytest.raises(RuntimeError, match="hipcc"):
        build.build()
