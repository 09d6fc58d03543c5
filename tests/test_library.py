"""Which library the operators run on, what is said and left behind when a part is missing, and that other threads
run during a call (no GPU)."""

import os
import shutil
import sys
import threading
import time

import pytest
import torch

import atlas_rnn_amd
from atlas_rnn_amd import _lib, build
from atlas_rnn_amd import functional as F


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


def test_other_threads_run_during_a_call():
    x, w = torch.randn(2048, 2048), torch.randn(2048, 2048)
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.is_set():
            ticks.append(time.perf_counter())
            time.sleep(1e-3)

    thread = threading.Thread(target=tick)
    threads = torch.get_num_threads()
    torch.set_num_threads(1)
    thread.start()
    try:
        t0 = time.perf_counter()
        for _ in range(2):
            F.linear(x, w)         # some tens of milliseconds in one native call
        t1 = time.perf_counter()
    finally:
        stop.set()
        thread.join()
        torch.set_num_threads(threads)
    inside = [t for t in ticks if t0 < t < t1]
    assert t1 - t0 > 0.02 and len(inside) > 5
