"""Which library the operators run on, and what is said and left behind when a part is missing (no GPU)."""

import os
import shutil
import sys

import pytest
import torch

import atlas_rnn_amd
from atlas_rnn_amd import _lib, build


def test_the_operators_run_on_the_loaded_library(tmp_path, monkeypatch):
    assert _lib.native().library() == os.path.abspath(_lib.LIB_PATH)
    other = str(tmp_path / "libatlas_mem_other.so")
    shutil.copy(_lib.LIB_PATH, other)
    lib = _lib.load(other)
    assert _lib.native().library() == os.path.abspath(_lib.LIB_PATH)   # a library loaded by its path is the caller's
    with monkeypatch.context() as m:
        m.setattr(_lib, "_LIB", lib)
        assert _lib.native().library() == other
    assert _lib.native().library() == os.path.abspath(_lib.LIB_PATH)


def test_a_failed_link_leaves_both_files(tmp_path, monkeypatch):
    paths = {n: str(tmp_path / os.path.basename(getattr(build, n))) for n in ("LIB_PATH", "HOST_PATH")}
    for n, p in paths.items():
        monkeypatch.setattr(build, n, p)
        with open(p, "w") as f:
            f.write("before")

    def run(cmd, verbose):
        out = cmd[cmd.index("-o") + 1]
        if os.path.basename(out).startswith("_host.so"):
            raise RuntimeError("no link")
        if out.startswith(str(tmp_path)):
            with open(out, "w") as f:
                f.write("after")

    monkeypatch.setattr(build, "_run", run)
    with pytest.raises(RuntimeError, match="no link"):
        build.build()
    assert [open(p).read() for p in paths.values()] == ["before", "before"]


def test_a_missing_extension_module_is_reported(monkeypatch):
    assert atlas_rnn_amd.get_cuda_status()["available"]
    monkeypatch.setattr(_lib, "_BOUND", None)
    monkeypatch.delattr(atlas_rnn_amd, "_host", raising=False)
    monkeypatch.setitem(sys.modules, "atlas_rnn_amd._host", None)   # its import fails
    status = atlas_rnn_amd.get_cuda_status()
    assert not status["available"] and status["loaded_via"] == "none" and "_host" in status["error"]
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    ready, message = atlas_rnn_amd.check_cuda_availability()
    assert not ready and "_host" in message
