"""EPBL columns mixed to the bottom of the water over a stack of bed fillers:
the sweeps that one workgroup makes side by side (foreseen guesses), against
the CPU oracle, bitwise.

Grids from one column to a few workgroups, one to six live layers over up to
88 fillers, mixing depths below and above the column's; the small grids leave
the foreseen sweeps fewer scratch columns than they have guesses, so the
sequential sweeps run as well.  Each handle solves four times: the list of
such columns has to be empty again after every solve.  One grid lists more
columns than the launch's workgroups take in one turn.
"""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from roundabout_amd import synth
from roundabout_amd.rdb import ColumnPhysics, default_config
from test_gpu_contrib import DT, _assert_equal, _compare, say

pytestmark = pytest.mark.gpu


def _shallow(nx, ny, nz, seed, live_max):
    o = synth.make_ocean(nx, ny, nz, seed, land_frac=0.1 if nx * ny > 4 else 0.0, topo="zlevel", dmin=20.0,
                         dmax=nz * 25.0)
    rng = np.random.default_rng(seed)
    live = rng.integers(1, live_max + 1, (nx, ny))
    wet = o.wet > 0.5
    h = np.full((nx, ny, nz), synth.FILLER_H)
    m = np.arange(nz)[::-1][None, None, :]
    h = np.where(m < live[:, :, None], rng.uniform(2.0, 30.0, (nx, ny, nz)), h)
    h[~wet] = synth.H_VANISHED
    live[~wet] = 0
    return dataclasses.replace(synth._with_state(rng, np.asfortranarray(h), o.wet, live.astype(np.int32), 0))


@pytest.mark.parametrize("nx,ny,nz,live_max,knobs", [
    (1, 1, 75, 3, {}),
    (7, 5, 14, 3, {}),
    (33, 17, 75, 4, dict(epbl_tke_diags=1)),
    (48, 30, 90, 6, dict(epbl_mld_bisection=1, epbl_tke_diags=1)),
    (48, 30, 75, 4, dict(epbl_mld_max_its=3, epbl_mld_use_prev_guess=1)),
    (40, 25, 60, 4, dict(epbl_mstar_scheme=3, epbl_vstar_scheme=2, epbl_use_lt=1, epbl_mixlen_exponent=1.5)),
    (40, 25, 60, 4, dict(epbl_mld_iteration=0)),
])
def test_bed_limited_columns(orc, gpu_lib, nx, ny, nz, live_max, knobs):
    say(f"[case] EPBL over fillers {nx}x{ny}x{nz} live<={live_max} {knobs}")
    cfg = default_config()
    cfg.epbl_enable = 1
    for k, v in knobs.items():
        setattr(cfg, k, v)
    o = _shallow(nx, ny, nz, 5, live_max)
    ref = orc.OracleState(o, cfg)
    with ColumnPhysics.from_ocean(o, config=cfg) as cp:
        for _ in range(4):
            cp.step(DT, 1)
            ref.step(DT, 1)
            _compare(cp, ref, cfg)
    _assert_equal("wet columns keep their thickness", o.h, ref.ocean.h)


def test_more_columns_than_one_turn(orc, gpu_lib):
    """256 workgroups of 64 columns: a list of more than 16 384 columns makes
    them go round again, over the same shared arrays and further scratch.  A
    column of one layer over 13 fillers is listed before its first interface."""
    nx, ny, nz = 210, 150, 14
    say(f"[case] EPBL over fillers {nx}x{ny}x{nz}, more than 16384 columns")
    cfg = default_config()
    cfg.epbl_enable = 1
    o = _shallow(nx, ny, nz, 6, 1)
    assert (o.wet > 0.5).sum() > 16384 + 64
    ref = orc.OracleState(o, cfg)
    with ColumnPhysics.from_ocean(o, config=cfg) as cp:
        for _ in range(2):
            cp.step(DT, 1)
            ref.step(DT, 1)
            _compare(cp, ref, cfg)
