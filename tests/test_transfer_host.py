"""The host side of the copies in pinned chunks (transfer.hip), compiled for
the CPU against a host stand-in for the HIP calls it makes (tests/host): what
the copying threads do while the stream is busy."""

from __future__ import annotations

import ctypes
import os
import subprocess
import time
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent
VP, SZ = ctypes.c_void_p, ctypes.c_size_t


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("transfer") / "libtransfer_host.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-pthread", "-Wl,-Bsymbolic", "-I", str(ROOT / "tests/host"), "-x", "c++",
                    str(ROOT / "roundabout_amd/csrc/transfer.hip"), str(ROOT / "tests/host/transfer_host.cpp"), "-o",
                    str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    lib.tr_new.restype = lib.tr_stream.restype = VP
    lib.tr_delete.argtypes = lib.tr_sync.argtypes = [VP]
    lib.tr_busy.argtypes = [VP, ctypes.c_double]
    lib.tr_to_host.argtypes = lib.tr_to_device.argtypes = [VP, VP, VP, SZ, VP]
    lib.tr_copy.argtypes = [VP, VP, VP, SZ]
    return lib


@pytest.fixture
def engine(lib):
    t = lib.tr_new()
    yield t
    lib.tr_delete(t)


def _p(a):
    return a.ctypes.data


@pytest.mark.parametrize("n", [1, (1 << 20) - 8, 1 << 20, (1 << 20) + 8, (4 << 20) + 8, (24 << 20) - 3, 64 << 20, (90 << 20) + 5])
def test_copies_whole(lib, engine, n):
    rng = np.random.default_rng(n)
    a = rng.integers(0, 255, n, dtype=np.uint8)
    dev, out, host = (np.zeros(n, dtype=np.uint8) for _ in range(3))
    s = lib.tr_stream()
    for turn in range(3):
        a ^= 1 + turn
        assert lib.tr_to_device(engine, _p(dev), _p(a), n, s) == 0
        assert lib.tr_to_host(engine, _p(out), _p(dev), n, s) == 0
        lib.tr_copy(engine, _p(host), _p(a), n)
        assert np.array_equal(out, a) and np.array_equal(host, a)


@pytest.mark.parametrize("way", ["to_host", "to_device"])
def test_threads_sleep_while_the_stream_is_busy(lib, engine, way):
    """A copy behind a long queue of work costs the time of its memcpys, not
    every thread's time until the queue has drained."""
    n = 96 << 20
    a, dev = np.ones(n, dtype=np.uint8), np.zeros(n, dtype=np.uint8)
    s = lib.tr_stream()
    f = lib.tr_to_host if way == "to_host" else lib.tr_to_device
    for busy in (0.0, 0.6):  # once to make the chunks and the threads
        lib.tr_sync(s)
        lib.tr_busy(s, busy)
        wall, cpu = time.perf_counter(), time.process_time()
        assert f(engine, _p(a), _p(dev), n, s) == 0
        wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    lib.tr_sync(s)
    print(f"{way}: wall {wall:.3f} s, process CPU {cpu:.3f} s")
    assert wall > 0.5 and cpu < 0.35


def test_a_thread_that_is_held_up_holds_up_nothing(lib, engine):
    """One of the copying threads loses its processor (a signal handler that
    sleeps): the others do its share."""
    n = 32 << 20
    a, b = np.arange(n, dtype=np.uint8), np.zeros(n, dtype=np.uint8)
    before = set(os.listdir("/proc/self/task"))
    lib.tr_copy(engine, _p(b), _p(a), n)
    helpers = sorted(set(os.listdir("/proc/self/task")) - before)
    if not helpers:
        pytest.skip("fewer than four processors: no copying threads")
    time.sleep(0.02)
    b[...] = 0
    lib.tr_hold(int(helpers[0]), 800)
    time.sleep(0.02)
    wall = time.perf_counter()
    lib.tr_copy(engine, _p(b), _p(a), n)
    wall = time.perf_counter() - wall
    print(f"wall {wall:.3f} s with one of {len(helpers)} threads held for 0.8 s")
    assert np.array_equal(a, b) and wall < 0.4
    time.sleep(0.9)  # the handler returns before the engine goes


def test_without_pinned_memory_no_error_is_left(lib):
    """No pinned chunks to be had: the runtime's own copy is taken, and the
    failed allocation is not left for the next hipGetLastError to report."""
    n = 5 << 20
    a, dev, out = np.full(n, 7, dtype=np.uint8), np.zeros(n, dtype=np.uint8), np.zeros(n, dtype=np.uint8)
    t, s = lib.tr_new(), lib.tr_stream()
    lib.tr_refuse_pinned(1)
    try:
        assert lib.tr_to_device(t, _p(dev), _p(a), n, s) == 0 and lib.tr_last_error() == 0
        assert lib.tr_to_host(t, _p(out), _p(dev), n, s) == 0 and lib.tr_last_error() == 0
    finally:
        lib.tr_refuse_pinned(0)
    assert np.array_equal(out, a)
    out[...] = 0
    assert lib.tr_to_host(t, _p(out), _p(dev), n, s) == 0 and np.array_equal(out, a)  # there is some again
    lib.tr_delete(t)


def test_without_memory_for_threads_the_caller_copies(lib):
    n = 5 << 20
    a, out = np.full(n, 3, dtype=np.uint8), np.zeros(n, dtype=np.uint8)
    t = lib.tr_new()
    lib.tr_no_memory(1)
    lib.tr_copy(t, _p(out), _p(a), n)  # std::bad_alloc through the C entry would end the process
    lib.tr_no_memory(0)
    assert np.array_equal(out, a)
    lib.tr_delete(t)
