"""Which library the operators run on (no GPU)."""

import os
import shutil

from atlas_rnn_amd import _lib


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

