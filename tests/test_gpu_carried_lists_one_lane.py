"""Lists carried over substeps by the passes with one lane per particle (small tiles on, or
more than 65,536 particles): every output equals that of lists rebuilt by every pass."""
import numpy as np
import pytest

from conftest import small_dam
from test_gpu_parity import developed_state, make_ctx

pytestmark = pytest.mark.gpu

OUTPUTS = ("cell_ids", "particle_ids", "neighbour_counters", "densities", "lambdas", "delta_positions", "omegas",
           "positions", "predicted", "velocities", "colors", "external_forces")


@pytest.mark.parametrize("scene", ["rest", "developed"])
@pytest.mark.parametrize("side,small", [(24, 0), (24, 32), (24, 64), (42, 0)])
def test_gpu_one_lane_passes_keep_lists(F, O, scene, side, small):
    p = small_dam(F, side)
    for a in range(3):  # the dam break's box, for a lattice larger than the configuration's
        p.bounds_max[a] = max(p.bounds_max[a], side * 0.05 * (2 if a == 0 else 1))
        p.grid_dims[a] = max(p.grid_dims[a], int(np.ceil(p.bounds_max[a] / 0.1)))
    if scene == "developed":
        st = developed_state(F, O, p, 4)
        state = (st.x4, st.v4, st.c4, st.f4, st.p4)
    else:
        state = (*F.generate_box(p), None, None)
    runs = {}
    for skin in (0, 10):
        print(f"one-lane carry: {scene} {side}^3, small {small}, skin {skin}", flush=True)
        ctx = make_ctx(F, p, *state)
        ctx.set_launch_shape(small_tile_max=small, list_skin_pct=skin)
        ctx.reset_counters()
        outs = []
        for _ in range(4):
            ctx.compute()
            outs.append({k: ctx.download(k) for k in OUTPUTS})
        runs[skin] = (outs, ctx.counters())
        ctx.close()
    assert runs[0][1]["list_carries"] == 0 and runs[10][1]["list_carries"] > 0
    for a, b in zip(runs[0][0], runs[10][0]):
        for k in OUTPUTS:
            assert np.array_equal(a[k], b[k]), k
