"""What the library recomputes outside the step when inputs change: the first
live layer, the bed-filler interfaces and the land columns, after a full
upload and after a momentum solve (which changes the centred velocities
alone).  Bitwise: the land and filler values against the CPU oracle, and the
short refresh against a fresh handle that is given the same velocities."""

from __future__ import annotations

import numpy as np
import pytest

from roundabout_amd import synth
from roundabout_amd.rdb import ColumnPhysics, default_config
from test_gpu_contrib import DT, _assert_equal, say

pytestmark = pytest.mark.gpu
FIELDS = ("temperature", "salinity", "kv", "kt", "ks", "bl_depth", "b0", "kbl")


def _ocean(nx, ny, nz, seed=3):
    o = synth.make_ocean(nx, ny, nz, seed, land_frac=0.4, topo="zlevel", dmin=20.0, dmax=nz * 40.0, n_passive=0)
    rng = np.random.default_rng(seed)  # velocities also on land faces and in fillers: their interfaces have shear
    o.u[...] = 0.1 * rng.standard_normal(o.u.shape)
    o.v[...] = 0.1 * rng.standard_normal(o.v.shape)
    return o


def _fields(cp):
    return {n: cp.get_field(n) for n in FIELDS}


@pytest.mark.parametrize("nz", [1, 7, 8, 9, 75])
@pytest.mark.parametrize("knobs", [{}, dict(ri_crit=0.0), dict(use_kpp=0), dict(shear2_floor=0.0)])
def test_land_and_fillers_match_the_oracle(orc, gpu_lib, nz, knobs):
    say(f"[case] land and fillers nz={nz} {knobs}")
    cfg = default_config()
    for k, v in knobs.items():
        setattr(cfg, k, v)
    o = _ocean(37, 21, nz)
    ref = orc.OracleState(o, cfg)
    ref.step(DT, 2)
    with ColumnPhysics.from_ocean(o, config=cfg) as cp:
        cp.step(DT, 2)
        for name, want in (("kv", ref.kv), ("kt", ref.kt), ("ks", ref.ks), ("temperature", ref.ocean.T)):
            _assert_equal(name, cp.get_field(name), want)
        if cfg.use_kpp:
            _assert_equal("bl_depth", cp.get_field("bl_depth"), ref.ocean.bl_depth)


@pytest.mark.parametrize("nz", [1, 8, 9, 75])
@pytest.mark.parametrize("precision", [0, 1])
def test_refresh_after_momentum_matches_a_full_one(gpu_lib, nz, precision):
    say(f"[case] refresh after momentum nz={nz} precision={precision}")
    cfg = default_config()
    cfg.precision = precision
    o = _ocean(45, 18, nz)
    with ColumnPhysics.from_ocean(o, config=cfg) as cp:
        cp.step(DT, 1)
        cp.vdiff_momentum(DT, implicit_stress=1)
        faces = {n: cp.get_field(n) for n in ("u_face_x_layer", "v_face_y_layer")}
        cp.step(DT, 2)
        cp.vdiff_momentum(DT, implicit_stress=1)
        cp.step(DT, 1)
        got = _fields(cp)
        faces2 = {n: cp.get_field(n) for n in faces}
    with ColumnPhysics.from_ocean(o, config=cfg) as cp:
        cp.step(DT, 1)
        for n, a in faces.items():
            cp.set_field(n, a)
        cp.step(DT, 2)
        for n, a in faces2.items():
            cp.set_field(n, a)
        cp.step(DT, 1)
        want = _fields(cp)
    for n in FIELDS:
        _assert_equal(n, got[n], want[n])
