"""The remap kernels at the layer counts where their loads' blocks and rings
end, on fields with filler runs at the bed, inside and at the top, dead
columns and targets far from their sources, against the oracle, bitwise."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from roundabout_amd.rdb import remap as R
from test_gpu_remap import _field

pytestmark = pytest.mark.gpu


def _top_fillers(ho, hn, rng):
    """Runs of fillers at the top and all but one layer vanished."""
    nx, ny, nz = ho.shape
    for i in range(0, nx, 4):
        n = min(nz - 1, 1 + i % 5)
        ho[i, 0, nz - n:] = 1.0e-4
        hn[i, 0, nz - n:] = 1.0e-4
        k = int(rng.integers(0, nz))
        ho[i, 1, :] = hn[i, 1, :] = 8.0e-5
        ho[i, 1, k] = hn[i, 1, k] = 12.0
        for j in (0, 1):
            hn[i, j, int(np.argmax(hn[i, j]))] += ho[i, j].sum() - hn[i, j].sum()


@pytest.mark.parametrize("nz", [5, 6, 7, 8, 9, 10, 13])
def test_pqm_layer_counts(orc, nz):
    nx, ny = 33, 9
    ho, hn, c = _field(nx, ny, nz, 50 + nz)
    _top_fillers(ho, hn, np.random.default_rng(nz))
    u = np.asfortranarray(np.random.default_rng(3).normal(0, 0.2, (nx + 1, ny, nz)))
    d_ho, d_hn = R.DeviceArray.from_host(ho), R.DeviceArray.from_host(hn)
    for be, nu in ((0, 0), (1, 1)):
        print(f"[case] PQM {nx}x{ny}x{nz} be={be} nu={nu}", flush=True)
        bud = np.zeros_like(ho, order="F")
        want, _ = orc.remap_tracer_field(5, ho, hn, c, be, nu, budget=bud)
        d_c, d_b = R.DeviceArray.from_host(c), R.DeviceArray.zeros(c.shape)
        R.ocean_remap_tracer_field(d_ho, d_hn, d_c, 5, bnd_extrap=be, nonunif=nu, budget=d_b)
        assert np.array_equal(d_c.to_host(), want) and np.array_equal(d_b.to_host(), bud)
        d_u = R.DeviceArray.from_host(u)
        R.ocean_apply_ale_remap_faces(d_ho, d_hn, d_u, None, 5, conserve_ke=be, zlevel_faces=nu, bnd_extrap=be, nonunif=nu)
        assert np.array_equal(d_u.to_host(), orc.remap_face_velocity(0, ho, hn, u, 5, be, nu, be, nu))


def _tiled(ho, hn, c, nx, ny):
    """The field repeated to (nx, ny): enough columns for one lane each."""
    reps = (-(-nx // ho.shape[0]), -(-ny // ho.shape[1]), 1)
    return [np.asfortranarray(np.tile(a, reps)[:nx, :ny]) for a in (ho, hn, c)]


def _far_targets(ho, hn, rng):
    """Targets that run ahead of their sources (thin ones over a thick bed
    cell) and behind, and targets over three and more stale fillers."""
    nx, ny, nz = ho.shape
    for i in range(0, nx, 3):
        for j in range(0, ny, 2):
            kind = (i // 3 + j) % 4
            if kind == 0:
                ho[i, j, 0] = 40.0 * nz
                hn[i, j, :-1] = 0.5 + rng.random(nz - 1)
            elif kind == 1:
                hn[i, j, 0] = 40.0 * nz
                ho[i, j, :-1] = 0.5 + rng.random(nz - 1)
            elif kind == 2 and nz > 6:
                ho[i, j, 1:6] = 1.0e-4
                hn[i, j, :3] = 0.2
            elif kind == 3 and nz > 6:
                ho[i, j, -6:-1] = 7.0e-5
                hn[i, j, -2:] = 3.0
            total = ho[i, j].sum()
            hn[i, j, -1] = 0.0
            if hn[i, j].sum() > total:
                hn[i, j] *= 0.9 * total / hn[i, j].sum()
            hn[i, j, -1] = total - hn[i, j, :-1].sum()


@pytest.mark.parametrize("nx,ny,nz", [(31, 20, 3), (31, 20, 8), (31, 20, 33), (270, 250, 3), (270, 250, 9), (262, 251, 17)])
@pytest.mark.parametrize("method", [1, 2, 3, 4, 5])
def test_in_place_and_split_walks(orc, nx, ny, nz, method):
    """Below 65 537 columns a column's targets are split over lanes, above one
    lane walks them, with scratch for what runs ahead: both, in place and out of
    place, on targets ahead of and behind their sources."""
    rng = np.random.default_rng(nz)
    ho, hn, c = _field(31, 20, nz, 90 + nz)
    _far_targets(ho, hn, rng)
    be, nu = method % 2, nz % 2
    print(f"[case] walk {nx}x{ny}x{nz} method={method} be={be} nu={nu}", flush=True)
    bud = np.zeros_like(ho, order="F")
    want, want_cl = orc.remap_tracer_field(method, ho, hn, c, be, nu, budget=bud)
    want, want_cl, bud = _tiled(want, want_cl, bud, nx, ny)
    ho, hn, c = _tiled(ho, hn, c, nx, ny)
    d_ho, d_hn = R.DeviceArray.from_host(ho), R.DeviceArray.from_host(hn)
    for in_place in (True, False):
        d_c, d_b, d_cl = R.DeviceArray.from_host(c), R.DeviceArray.zeros(c.shape), R.DeviceArray(c.shape)
        d_o = None if in_place else R.DeviceArray(c.shape)
        out = R.ocean_remap_tracer_field(d_ho, d_hn, d_c, method, bnd_extrap=be, nonunif=nu, budget=d_b, clamp_out=d_cl,
                                         c_out=d_o)
        for name, g, w in (("c", out, want), ("budget", d_b, bud), ("clamp", d_cl, want_cl)):
            assert np.array_equal(g.to_host(), w), (name, in_place)
    u = np.asfortranarray(rng.normal(0, 0.2, (nx + 1, ny, nz)))
    d_u = R.DeviceArray.from_host(u)
    R.ocean_apply_ale_remap_faces(d_ho, d_hn, d_u, None, method, bnd_extrap=be, nonunif=nu)
    assert np.array_equal(d_u.to_host(), orc.remap_face_velocity(0, ho, hn, u, method, 0, 0, be, nu))
    d_q = R.DeviceArray.from_host(c.reshape(-1, nz, order="F"))
    cols = [R.DeviceArray.from_host(a.reshape(-1, nz, order="F")) for a in (ho, hn)]
    got = R.remap_column(*cols, d_q, method, bnd_extrap=be, nonunif=nu).to_host()
    R.remap_column(*cols, d_q, method, bnd_extrap=be, nonunif=nu, q_new=d_q)
    assert np.array_equal(d_q.to_host(), got)


@pytest.mark.parametrize("nx,ny,nz", [(31, 20, 3), (31, 20, 33), (270, 250, 9)])
@pytest.mark.parametrize("method", [1, 2, 3, 4, 5])
def test_round_off_negative_targets(orc, nx, ny, nz, method):
    """Targets a round-off below zero, as a difference of interfaces leaves
    them: the next target begins a little below where the last one ended."""
    print(f"[case] negative targets {nx}x{ny}x{nz} method={method}", flush=True)
    rng = np.random.default_rng(7 * nz)
    ho = 1.0 + 25.0 * rng.random((31, 20, nz))
    hn = ho * (0.4 + 1.2 * rng.random((31, 20, nz)))
    c = 30.0 + 5.0 * rng.random((31, 20, nz))
    hn[rng.random((31, 20, nz)) < 0.15] = -1.0e-15
    want, _ = orc.remap_tracer_field(method, ho, hn, c, 0, 0)
    want, ho, hn, c = _tiled(want, ho, c, nx, ny)[:1] + _tiled(ho, hn, c, nx, ny)
    d = [R.DeviceArray.from_host(a) for a in (ho, hn, c)]
    R.ocean_remap_tracer_field(*d, method)
    assert np.array_equal(d[2].to_host(), want)


@pytest.mark.parametrize("kind", ["negative", "nan", "negative source"])
@pytest.mark.parametrize("nz", [8, 33, 75])
def test_split_lanes_start_where_one_lane_would(nz, kind):
    """Thicknesses outside the stated range give what one lane a column gives
    (the same columns in a batch of more than 65 536)."""
    rng = np.random.default_rng(nz)
    ho = 1.0 + 25.0 * rng.random((31, 20, nz))
    hn = ho * (0.4 + 1.2 * rng.random((31, 20, nz)))
    c = 30.0 + 5.0 * rng.random((31, 20, nz))
    some = rng.random((31, 20, nz)) < 0.1
    if kind == "nan":
        hn[some & (rng.random(some.shape) < 0.4)] = np.nan
    else:
        a = hn if kind == "negative" else ho
        a[some] *= -rng.random(int(some.sum()))
    for method in (1, 2, 3, 4, 5):
        print(f"[case] {kind} nz={nz} method={method}", flush=True)
        got = []
        for shape in ((31, 20), (270, 250)):
            d = [R.DeviceArray.from_host(a) for a in _tiled(ho, hn, c, *shape)]
            R.ocean_remap_tracer_field(*d, method)
            got.append(d[2].to_host()[:31, :20])
        assert np.array_equal(*got, equal_nan=True), method


@pytest.mark.parametrize("nz", [7, 12, 24])
@pytest.mark.parametrize("method", [1, 3, 5])
def test_deferred_targets_and_many_excesses(orc, nz, method):
    """Thin targets far ahead of their sources, then one over a long run of
    stale fillers, in place: its excesses lie in scratch where the deferred
    targets wait."""
    rng = np.random.default_rng(nz)
    ho = 2.0 + 20.0 * rng.random((31, 20, nz))
    c = 30.0 + 5.0 * rng.random((31, 20, nz))
    hn = np.empty_like(ho)
    for i in range(31):
        for j in range(20):
            bed, thin = int(rng.integers(1, 3)), int(rng.integers(0, nz - 2))
            fill = int(rng.integers(2, max(3, nz - 1 - bed)))
            ho[i, j, :bed] = 100.0
            ho[i, j, bed:bed + fill] = 2.0e-5 + 1.2e-4 * rng.random(fill)
            total = ho[i, j].sum()
            hn[i, j, :thin] = 90.0 * bed / nz * rng.random(thin)
            rest = rng.random(nz - thin)
            rest[0] += 3.0
            hn[i, j, thin:] = rest * (total - hn[i, j, :thin].sum()) / rest.sum()
    bud = np.zeros_like(ho, order="F")
    print(f"[case] deferred targets and excesses nz={nz} method={method}", flush=True)
    want, want_cl = orc.remap_tracer_field(method, ho, hn, c, 0, 0, budget=bud)
    want, want_cl, bud = _tiled(want, want_cl, bud, 270, 250)
    ho, hn, c = _tiled(ho, hn, c, 270, 250)
    d_ho, d_hn, d_c = (R.DeviceArray.from_host(a) for a in (ho, hn, c))
    d_b, d_cl = R.DeviceArray.zeros(c.shape), R.DeviceArray(c.shape)
    R.ocean_remap_tracer_field(d_ho, d_hn, d_c, method, budget=d_b, clamp_out=d_cl)
    for name, g, w in (("c", d_c, want), ("budget", d_b, bud), ("clamp", d_cl, want_cl)):
        assert np.array_equal(g.to_host(), w), name


def test_in_place_calls_hold_one_field_of_scratch():
    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert R._hip().hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    print("[case] scratch of in-place calls, 128 MiB fields", flush=True)
    h = R.DeviceArray.from_host(np.full((65536, 256), 10.0, order="F"))
    q = h.copy()
    R.remap_column(h, h, q, 1, q_new=q)  # lanes share a column: through a buffer of one field
    R.synchronize()
    before = free()
    for a in (h, q):
        a.shape = (131072, 128)
    R.remap_column(h, h, q, 1, q_new=q)  # one lane a column
    for a in (h, q):
        a.shape = (512, 256, 128)
    R.ocean_remap_tracer_field(h, h, q, 1)
    R.synchronize()
    assert before - free() < 64 << 20
