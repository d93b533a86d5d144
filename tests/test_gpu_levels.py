"""The layer counts at which the rings, blocks and LDS tiers of the step's
kernels end, in the launch shape that a fresh handle starts from: the fused
step (up to four passives), the staged solve (five) and the contributors'
pass, bitwise against the oracle."""

from __future__ import annotations

import pytest

from roundabout_amd import synth
from roundabout_amd.rdb import ColumnPhysics, default_config
from test_gpu_contrib import DT, _compare, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [1, 2, 5, 6, 7, 8, 13, 33, 40])
@pytest.mark.parametrize("passive,knobs", [(0, {}), (4, {}), (5, {}), (1, dict(kt_bg=2e-5)),
                                           (3, dict(epbl_enable=1, conv_enable=1, ddiff_enable=1, kv_ml_invz2=1e-2)),
                                           (0, dict(conv_enable=1))])
def test_layer_counts(orc, gpu_lib, nz, passive, knobs):
    say(f"[case] levels nz={nz} passive={passive} {knobs}")
    cfg = default_config()
    for k, v in knobs.items():
        setattr(cfg, k, v)
    o = synth.make_ocean(29, 23, nz, 4, land_frac=0.2, topo="zlevel", dmin=30.0, dmax=60.0 * nz, n_passive=passive)
    ref = orc.OracleState(o, cfg)
    ref.step(DT, 3)
    with ColumnPhysics.from_ocean(o, config=cfg) as cp:
        cp.step(DT, 3)
        _compare(cp, ref, cfg)
