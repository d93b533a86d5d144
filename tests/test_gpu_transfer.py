"""Copies between host arrays and the device in pinned chunks: every size
class (the runtime's own copy, small chunks, large chunks), a chunk more and
a cell less, into and out of arrays that start on no page or line boundary,
and the checks that moved to the device with the upload of h_layer.  Exact."""

from __future__ import annotations

import ctypes
import time

import numpy as np
import pytest

from roundabout_amd import synth
from roundabout_amd.rdb import ColumnEnsemble, ColumnPhysics, RdbError, _ffi
from test_gpu_contrib import say

pytestmark = pytest.mark.gpu


def _shifted(shape, rng):
    """A Fortran-ordered array 8 bytes off its allocation's start."""
    n = int(np.prod(shape))
    a = rng.standard_normal(n + 1)[1:]
    return a.reshape(shape, order="F")


# 1 MiB, 4 MiB and 64 MiB are where the chunks change
@pytest.mark.parametrize("nx,ny,nz", [(3, 2, 1), (64, 64, 31), (64, 64, 32), (64, 64, 33), (128, 128, 32), (131, 128, 32),
                                      (127, 131, 97), (256, 256, 127), (256, 256, 128), (257, 256, 129)])
def test_round_trips(gpu_lib, nx, ny, nz):
    say(f"[case] transfer {nx}x{ny}x{nz}: {nx * ny * nz / 131072:.2f} MiB")
    rng = np.random.default_rng(nx + nz)
    wet = np.asfortranarray((rng.random((nx, ny)) > 0.3).astype(float))
    with ColumnPhysics(nx, ny, nz, wet) as cp:
        for turn in range(2):
            sent = {}
            for name in ("temperature", "kv", "u_face_x_layer", "v_face_y_layer", "salinity"):
                sent[name] = _shifted(cp.shape_of(name), rng)
                cp.set_field(name, sent[name])
            for name, a in sent.items():
                assert np.array_equal(cp.get_field(name), a), (turn, name)
        shape = cp.shape_of("salinity")
        into = _shifted(shape, rng)
        st = gpu_lib.rdb_colphys_get_field(cp._handle(), b"salinity", into.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), *shape)
        assert st == _ffi.OK and np.array_equal(into, sent["salinity"])


def test_the_buffer_is_the_callers_again(gpu_lib):
    """set_field returns when it has read the array."""
    say("[case] transfer: arrays overwritten after set_field")
    rng = np.random.default_rng(1)
    a = np.asfortranarray(rng.standard_normal((200, 180, 60)))
    with ColumnPhysics(200, 180, 60, np.ones((200, 180), order="F")) as cp:
        for _ in range(3):
            want = a.copy(order="F")
            cp.set_field("temperature", a)
            a[...] = rng.standard_normal(a.shape)
            assert np.array_equal(cp.get_field("temperature"), want)


def test_members_share_one_engine(gpu_lib):
    say("[case] transfer: ensemble members")
    rng = np.random.default_rng(2)
    grids = [(150, 120, 20, np.ones((150, 120), order="F")), (90, 200, 30, np.ones((90, 200), order="F"))]
    with ColumnEnsemble(grids) as ens:
        sent = [np.asfortranarray(rng.standard_normal(g[:3])) for g in grids]
        for m, a in enumerate(sent):
            ens.member_set_field(m, "salinity", a)
        for m, a in enumerate(sent):
            assert np.array_equal(ens.member_get_field(m, "salinity"), a)


@pytest.mark.parametrize("nz", [1, 7, 8, 9, 40])
def test_land_contract_is_checked(gpu_lib, nz):
    """The first offending cell (lowest level, then lowest column) is named
    and the thicknesses held before stay."""
    say(f"[case] transfer: land contract nz={nz}")
    rng = np.random.default_rng(nz)
    wet = np.asfortranarray((rng.random((30, 20)) > 0.4).astype(float))
    h = np.asfortranarray(np.where((wet > 0.5)[:, :, None], 10.0 + rng.random((30, 20, nz)), 1.5e-4))
    with ColumnPhysics(30, 20, nz, wet) as cp:
        cp.set_field("h_layer", h)
        live = cp.stats()["live_levels"]
        assert live == int((wet > 0.5).sum()) * nz
        bad = h.copy(order="F")
        land = np.argwhere(wet < 0.5)
        (i0, j0), (i1, j1) = land[3], land[7]
        bad[i1, j1, nz - 1] = 2.0
        bad[i0, j0, nz // 2:] = 2.0
        cells = [(k, j, i) for k in range(nz) for i, j in ((i0, j0), (i1, j1)) if bad[i, j, k] > 1.5e-4]
        k, j, i = min(cells, key=lambda c: (c[0], c[1] * 30 + c[2]))
        with pytest.raises(RdbError, match=rf"i={i + 1}, j={j + 1}\) has a live layer k={k + 1} "):
            cp.set_field("h_layer", bad)
        assert np.array_equal(cp.get_field("h_layer"), h) and cp.stats()["live_levels"] == live
        h[:, :, : nz // 2] = np.minimum(h[:, :, : nz // 2], 1e-4)  # fillers
        cp.set_field("h_layer", h)
        assert cp.stats()["live_levels"] == int((wet > 0.5).sum()) * (nz - nz // 2)


@pytest.mark.parametrize("way", ["get", "set"])
def test_one_thread_waits_for_the_steps_in_flight(gpu_lib, way):
    """A copy behind steps that are still running costs one thread's wait."""
    say(f"[case] transfer: {way}_field behind a long run")
    nx, ny, nz = 480, 360, 75
    o = synth.make_ocean(nx, ny, nz, 1, land_frac=0.3, topo="zlevel", dmin=50.0, dmax=5500.0)
    with ColumnPhysics.from_ocean(o) as cp:
        T = cp.get_field("temperature")
        for n_steps in (1, 2000):  # once to make the chunks, the threads and the graph
            cp.set_field("temperature", T)
            cp.step(3600.0, 1)
            cp.synchronize()
            cp.step(3600.0, n_steps)
            wall, cpu = time.perf_counter(), time.process_time()
            if way == "get":
                cp.get_field("temperature")
            else:
                cp.set_field("temperature", T)
            wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    say(f"wall {wall:.3f} s, process CPU {cpu:.3f} s")
    assert wall > 0.1 and cpu < 2.0 * wall
