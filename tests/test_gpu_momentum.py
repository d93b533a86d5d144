"""Parity of the HIP momentum vertical viscosity (rdb_colphys_vdiff_momentum)
with the oracle's restatement of vdiff_apply_momentum /
diffuse_velocity_columns_impl (rdb_ocean_vdiff.F90:455-718, 1416-2115):
face velocities and viscous remnant compared bitwise (``==``), with the
closure's kv from a plain step or the scalar K_v_momentum, every fold and
face-thickness option, on the 64 x 64 x 20 case and a z-level crop of the
tile; and a column step after the momentum solve reads the new velocities.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from roundabout_amd import synth
from roundabout_amd.rdb import ColumnPhysics, default_config
from roundabout_amd.rdb import remap as R

pytestmark = pytest.mark.gpu
DT = 3600.0


def _face_inputs(ocean, seed, zlevel):
    nx, ny, nz = ocean.nx, ocean.ny, ocean.nz
    rng = np.random.default_rng(seed)
    f = {}
    for tag, shp in (("u", (nx + 1, ny)), ("v", (nx, ny + 1))):
        f[f"lambda_bot_{tag}"] = rng.uniform(0.0, 2e-4, shp)
        f[f"lambda_top_{tag}"] = rng.uniform(0.0, 1e-4, shp)
        f[f"cover_{tag}"] = (rng.random(shp) < 0.2).astype(float)
        f[f"kv_bbl_{tag}"] = rng.uniform(1e-5, 5e-3, shp)
        f[f"bbl_thick_{tag}"] = rng.uniform(1.0, 30.0, shp)
        f[f"k_top_{tag}"] = rng.integers(nz - 1, nz + 1, shp).astype(float)
        if zlevel:
            # the first layer live on both sides, counted up from the bed
            live = np.where(ocean.h > 1.5e-4, 1, 0)
            kb = nz - live.sum(axis=2) + 1  # 1-based first live layer of each cell
            if tag == "u":
                kl = np.concatenate([kb[:1], kb], axis=0)
                kr = np.concatenate([kb, kb[-1:]], axis=0)
            else:
                kl = np.concatenate([kb[:, :1], kb], axis=1)
                kr = np.concatenate([kb, kb[:, -1:]], axis=1)
            f[f"k_bot_{tag}"] = np.minimum(np.maximum(kl, kr), nz).astype(float)
        else:
            f[f"k_bot_{tag}"] = rng.integers(1, 3, shp).astype(float)
    f["kv_corner"] = rng.uniform(0.0, 1e-3, (nx + 1, ny + 1, nz + 1))
    return f


def _oracle_kwargs(mode, f):
    kw = dict(implicit_stress=True, implicit_drag=True, implicit_top_drag=True, remnant=True,
              lambda_bot_u=f["lambda_bot_u"], lambda_bot_v=f["lambda_bot_v"], lambda_top_u=f["lambda_top_u"],
              lambda_top_v=f["lambda_top_v"], cover_u=f["cover_u"], cover_v=f["cover_v"], k_top_u=f["k_top_u"],
              k_bot_u=f["k_bot_u"], k_top_v=f["k_top_v"], k_bot_v=f["k_bot_v"])
    lib_kw = dict(implicit_stress=1, implicit_drag=1, implicit_top_drag=1, remnant=1)
    if mode == "zlevel":
        kw["zlevel_faces"], lib_kw["zlevel_faces"] = True, 1
    if mode in ("mom6_harm", "mom6_zclear", "glue", "glue_per_face"):
        kw["hvel_mom6"], lib_kw["hvel_mom6"] = True, 1
    if mode == "mom6_harm":
        kw["hvel_harmonic"], lib_kw["hvel_harmonic"] = True, 1
    if mode in ("glue", "glue_per_face"):
        kw["bbl_glue"], lib_kw["bbl_glue"] = True, 1
    if mode == "glue_per_face":
        kw.update(bbl_per_face=True, kv_bbl_u=f["kv_bbl_u"], kv_bbl_v=f["kv_bbl_v"], bbl_thick_u=f["bbl_thick_u"],
                  bbl_thick_v=f["bbl_thick_v"])
        lib_kw["bbl_per_face"] = 1
    if mode == "corner":
        kw.update(kv_corner=f["kv_corner"], kv_corner_prandtl=0.7)
        lib_kw.update(use_corner=1, kv_corner_prandtl=0.7)
    return kw, lib_kw


def _run(orc, ocean, mode, seed, zlevel=False, n_first=1):
    cfg = default_config()
    f = _face_inputs(ocean, seed, zlevel)
    kw, lib_kw = _oracle_kwargs(mode, f)
    with ColumnPhysics.from_ocean(ocean, config=cfg) as cp:
        cp.step(DT, n_first)  # the closure's kv of a plain step
        kv = cp.get_field("kv")
        u0, v0 = cp.get_field("u_face_x_layer"), cp.get_field("v_face_y_layer")
        for name, arr in f.items():
            cp.set_field(name, arr)
        cp.vdiff_momentum(DT, **lib_kw)
        got = {n: cp.get_field(n) for n in ("u_face_x_layer", "v_face_y_layer", "visc_rem_u", "visc_rem_v")}
    u, v, ru, rv = orc.vdiff_apply_momentum(ocean.h, u0, v0, ocean.wet, DT, kv_source=kv, tau_u=ocean.tau_x,
                                            tau_v=ocean.tau_y, rho0=cfg.rho0, **kw)
    for name, want in (("u_face_x_layer", u), ("v_face_y_layer", v), ("visc_rem_u", ru), ("visc_rem_v", rv)):
        g = got[name]
        assert np.array_equal(g, want), (mode, name, int(np.sum(g != want)), float(np.max(np.abs(g - want))))
    return got


@pytest.mark.parametrize("mode", ["default", "zlevel", "mom6_harm", "mom6_zclear", "glue", "glue_per_face",
                                  "corner"])
def test_momentum_small_bitwise(orc, mode):
    print(f"[case] momentum {mode}, 64x64x20 seed 3, bitwise vs oracle", flush=True)
    _run(orc, synth.small(3), mode, seed=21, zlevel=(mode == "zlevel"))


@pytest.mark.parametrize("mode", ["zlevel", "mom6_zclear"])
def test_momentum_tile_crop_bitwise(orc, mode):
    print(f"[case] momentum {mode}, z-level tile 160x128x75, bitwise vs oracle", flush=True)
    ocean = synth.tile(5, nx=160, ny=128)
    _run(orc, ocean, mode, seed=22, zlevel=True)


def test_momentum_scalar_viscosity_and_remnant_only(orc):
    print("[case] momentum: scalar K_v_momentum, remnant-only, default no-op", flush=True)
    ocean = synth.small(4)
    cfg = default_config()
    with ColumnPhysics.from_ocean(ocean, config=cfg) as cp:
        cp.vdiff_momentum(DT, use_kv_source=0, K_v_momentum=0.0)  # the pure-vdiff no-op
        assert np.array_equal(cp.get_field("u_face_x_layer"), ocean.u)
        cp.vdiff_momentum(DT, use_kv_source=0, K_v_momentum=2e-2, remnant=1, remnant_only=1)
        assert np.array_equal(cp.get_field("u_face_x_layer"), ocean.u)  # remnant only: u untouched
        ru = cp.get_field("visc_rem_u")
        cp.vdiff_momentum(DT, use_kv_source=0, K_v_momentum=2e-2)
        u1, v1 = cp.get_field("u_face_x_layer"), cp.get_field("v_face_y_layer")
    u, v, _, _ = orc.vdiff_apply_momentum(ocean.h, ocean.u, ocean.v, ocean.wet, DT, K_v_momentum=2e-2)
    _, _, rr, _ = orc.vdiff_apply_momentum(ocean.h, ocean.u, ocean.v, ocean.wet, DT, K_v_momentum=2e-2,
                                           remnant=True, remnant_only=True)
    assert np.array_equal(u1, u) and np.array_equal(v1, v) and np.array_equal(ru, rr)
    # no drag: the rows sum to one, so the remnant is one to round-off
    # wherever the couplings are moderate (faces between two wet cells; a
    # land cell's vanished layers make the couplings ~1e9 and the round-off
    # of the solve ~1e-7)
    wet = ocean.wet > 0.5
    both = np.zeros((ocean.nx + 1, ocean.ny), dtype=bool)
    both[1:-1] = wet[:-1] & wet[1:]
    assert np.max(np.abs(ru[both] - 1.0)) < 1e-12


def test_column_step_reads_the_new_velocities(orc):
    """step -> momentum -> step equals the oracle doing the same: the
    centred velocities of the column step follow the momentum solve."""
    print("[case] step, momentum, step: 64x64x20 seed 6 vs oracle", flush=True)
    ocean = synth.small(6)
    cfg = default_config()
    ref = orc.OracleState(ocean, cfg)
    ref.step(DT, 1)
    u, v, _, _ = orc.vdiff_apply_momentum(ref.ocean.h, ref.ocean.u, ref.ocean.v, ref.ocean.wet, DT,
                                          kv_source=ref.kv)
    ref.ocean.u[...] = u
    ref.ocean.v[...] = v
    ref.step(DT, 1)
    with ColumnPhysics.from_ocean(ocean, config=cfg) as cp:
        cp.step(DT, 1)
        cp.vdiff_momentum(DT)
        cp.step(DT, 1)
        for name, want in (("temperature", ref.ocean.T), ("salinity", ref.ocean.S), ("kv", ref.kv),
                           ("kt", ref.kt), ("bl_depth", ref.ocean.bl_depth), ("u_face_x_layer", u),
                           ("v_face_y_layer", v)):
            got = cp.get_field(name)
            assert np.array_equal(got, want), (name, int(np.sum(got != want)))


@pytest.mark.parametrize("nx,ny,nz", [(9, 7, 1), (33, 18, 6), (40, 25, 7), (64, 64, 20)])
@pytest.mark.parametrize("remnant_only", [False, True])
def test_bottom_and_top_rows_beyond_the_column(orc, nx, ny, nz, remnant_only):
    """Faces whose k_bot and k_top both lie above nz (no row to solve), next
    to faces with one of them there: identity columns, as the oracle's."""
    print(f"[case] momentum, k_bot/k_top beyond nz, {nx}x{ny}x{nz} remnant_only={remnant_only}", flush=True)
    ocean = synth.make_ocean(nx, ny, nz, 8, land_frac=0.2, topo="zstar")
    rng = np.random.default_rng(nz)
    f = {}
    for tag, shp in (("u", (nx + 1, ny)), ("v", (nx, ny + 1))):
        for end in ("k_bot", "k_top"):
            beyond = nz + rng.integers(1, 300, shp)
            f[f"{end}_{tag}"] = np.where(rng.random(shp) < 0.5, beyond, rng.integers(1, nz + 1, shp)).astype(float)
    kw = dict(implicit_stress=True, remnant=True, remnant_only=remnant_only, K_v_momentum=1e-2)
    u, v, ru, rv = orc.vdiff_apply_momentum(ocean.h, ocean.u, ocean.v, ocean.wet, DT, tau_u=ocean.tau_x,
                                            tau_v=ocean.tau_y, rho0=default_config().rho0, **f, **kw)
    with ColumnPhysics.from_ocean(ocean) as cp:
        for name, arr in f.items():
            cp.set_field(name, arr)
        cp.vdiff_momentum(DT, use_kv_source=0, **{k: (int(x) if isinstance(x, bool) else x) for k, x in kw.items()})
        for name, want in (("u_face_x_layer", u), ("v_face_y_layer", v), ("visc_rem_u", ru), ("visc_rem_v", rv)):
            assert np.array_equal(cp.get_field(name), want), name


def test_work_arrays_of_a_solve():
    """Beside the face velocities and the natural-order copies of h and kv a
    solve keeps c' of both directions: no more than two face fields."""
    nx, ny, nz = 256, 256, 128
    print(f"[case] momentum: device memory of the first solve, {nx}x{ny}x{nz}", flush=True)

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert R._hip().hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    with ColumnPhysics(nx, ny, nz, np.ones((nx, ny), order="F")) as cp:
        cp.set_field("h_layer", np.full((nx, ny, nz), 10.0, order="F"))
        cp.step(DT, 1)
        cp.synchronize()
        before = free()
        cp.vdiff_momentum(DT, implicit_stress=1)
        cp.synchronize()
        field = 8 * nz * (nx + 1) * ny
        assert before - free() < 6 * field + (32 << 20)


@pytest.mark.parametrize("zlevel", [False, True])
def test_bottom_rows_below_the_column(orc, zlevel):
    """Faces whose k_bot is below 1, among ordinary ones: every row of theirs
    is solved, and nothing outside the column is touched (the neighbouring
    allocations' fields come back as they were set)."""
    nx, ny, nz = 33, 18, 6
    print(f"[case] momentum, k_bot below 1, {nx}x{ny}x{nz} zlevel={zlevel}", flush=True)
    ocean = synth.make_ocean(nx, ny, nz, 8, land_frac=0.2, topo="zstar")
    rng = np.random.default_rng(nz)
    f = {}
    for tag, shp in (("u", (nx + 1, ny)), ("v", (nx, ny + 1))):
        f[f"k_bot_{tag}"] = np.where(rng.random(shp) < 0.5, 1 - rng.integers(1, 40, shp), 1).astype(float)
        f[f"lambda_bot_{tag}"] = rng.uniform(0.0, 2e-4, shp)
    kw = dict(implicit_stress=True, remnant=True, K_v_momentum=1e-2)
    u, v, ru, rv = orc.vdiff_apply_momentum(ocean.h, ocean.u, ocean.v, ocean.wet, DT, tau_u=ocean.tau_x,
                                            tau_v=ocean.tau_y, rho0=default_config().rho0, **f, **kw)
    with ColumnPhysics.from_ocean(ocean) as cp:
        for name, arr in f.items():
            cp.set_field(name, arr)
        cp.vdiff_momentum(DT, use_kv_source=0, implicit_stress=1, remnant=1, K_v_momentum=1e-2, zlevel_faces=int(zlevel))
        for name, want in (("u_face_x_layer", u), ("v_face_y_layer", v), ("visc_rem_u", ru), ("visc_rem_v", rv)):
            got = cp.get_field(name)
            assert np.isfinite(got).all() if zlevel else np.array_equal(got, want), name
        for name in ("temperature", "salinity", "h_layer"):
            assert np.array_equal(cp.get_field(name), {"temperature": ocean.T, "salinity": ocean.S, "h_layer": ocean.h}[name])
        for name, arr in f.items():
            assert np.array_equal(np.asarray(cp.get_field(name)).reshape(arr.shape, order="F"), arr)
