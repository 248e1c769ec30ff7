"""The tile classification with 4, 16 and 64 flags a wave (grids of up to 2^17, 2^22 and
more blocks): the same lists whichever it takes, and a box far larger than its fluid costs
little more than clearing its cell table."""
import numpy as np
import pytest

from test_gpu_wide_tiles import _scene

pytestmark = pytest.mark.gpu

OUTPUTS = ("cell_ids", "particle_ids", "neighbour_counters", "densities", "lambdas", "delta_positions", "omegas",
           "positions", "velocities", "external_forces")


# per cell: sparse small tiles, small and crowded ones, whole and split blocks, halos past a half's capacity
@pytest.mark.parametrize("counts", [(1, 0, 0, 0, 0), (0, 0, 3, 1, 4, 0), (5, 6), (0, 0, 14, 9, 13), (16, 3, 20)])
@pytest.mark.parametrize("bits", [5, 6])
def test_gpu_tile_classes_do_not_depend_on_the_grid(F, counts, bits):
    want = None
    for rows in (8, 260, 520):  # 16, 1.0M and 8.4M blocks of 2^5 cells
        p, x, v = _scene(F, (8, 8, 8), counts, 0.98)
        p.tile_bits = bits
        p.grid_dims[1] = rows
        p.solver_iterations = 2
        ctx = F.Context(p, len(x))
        ctx.add_particles(x, v)
        ctx.set_launch_shape(small_tile_max=64)
        print(f"tile classes: counts {counts}, bits {bits}, {rows} rows", flush=True)
        for _ in range(2):
            ctx.compute()
        got = {k: ctx.download(k) for k in OUTPUTS}
        got["counters"] = np.array(list(ctx.counters().values()))
        ctx.close()
        want = want or got
        for k in want:
            assert np.array_equal(want[k], got[k]), (rows, k)


def test_gpu_tile_classes_of_a_sparse_grid(F):
    """5,000 particles in a grid of 1024 x 1024 x 1024 cells: the tile lists take less than a
    fifth of the cell table's clearing (with 4 flags a wave, they took half of it)."""
    p, x, v = _scene(F, (10, 10, 10), (5,), 0.98)
    for a in range(3):
        p.grid_dims[a] = 1024
    ctx = F.Context(p, len(x))
    ctx.add_particles(x, v)
    ctx.compute()
    ctx.set_timing(True)
    ctx.reset_timings()
    for _ in range(4):
        ctx.compute()
    ctx.sync()
    t = ctx.timings()
    ctx.close()
    print(f"sparse grid: {t['tile_list']} tile lists, {t['cell_reset']} cell table", flush=True)
    assert t["tile_list"][0] <= 0.2 * t["cell_reset"][0]
