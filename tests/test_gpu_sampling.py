"""GPU tests of the samplers' row loads (two neighbours for the trilinear, four
for the tricubic lookup) where the nodes repeat the grid's edge: back-traces
that stay inside, reach a few cells, and leave the grid on every side, on rows
of 4 and 5 elements up to more than a wave. Bit for bit the oracle's."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(__file__))
from test_gpu_parity import B, compare, pair, random_state, settings  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vel", [0.05, 2.0, 400.0])
@pytest.mark.parametrize("res", [(4, 4, 4), (6, 5, 4), (4, 9, 13), (66, 6, 5), (128, 4, 7)],
                         ids=lambda r: "x".join(map(str, r)))
def test_advection_at_edges(res, vel):
    print(f"[sampling] {res} velocity {vel}", flush=True)
    s = settings(B, res, smoke_density=1.0)
    g, o = pair(s, random_state(s, 21, vel_scale=vel, smoke=True))
    for x in (g, o):
        x.run_stage(B.STAGE_ADVECT, 0.0, 1.0 / 24.0)
        x.run_stage(B.STAGE_VORTICITY, 0.0, 1.0 / 24.0)
    for w, name in enumerate(["T", "U", "V", "W", "density"]):
        compare(f"{res} {vel}: {name}", g.field(w), o.field(w))
