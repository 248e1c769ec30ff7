"""Neighbour lists of the tile passes at the edges of their loads and scans: cells of
0 to 40 particles (groups of 8 lanes load 16 of a cell at once, a scan takes 32 slots
of a column), blocks with more and fewer particles than a workgroup or a wave, and
positions that are not numbers."""
import numpy as np
import pytest

from conftest import small_dam

pytestmark = pytest.mark.gpu


def _crowded(F, counts, seed=7):
    """A 4 x 8 x 8-cell scene whose cell k holds counts[k mod len] particles."""
    p = small_dam(F, 8)
    p.box_spawn_in_the_beginning = 0
    p.gravity = 0.0
    dims = (4, 8, 8)
    for a in range(3):
        p.grid_dims[a] = dims[a]
        p.bounds_min[a] = 0.0
        p.bounds_max[a] = dims[a] * 0.1
    p.solver_iterations = 1
    p.stabilization_iterations = 0
    rng = np.random.default_rng(seed)
    pos = []
    for k in range(dims[0] * dims[1] * dims[2]):
        c = np.array([k // 64, (k // 8) % 8, k % 8])
        pos.append((c + rng.uniform(0.02, 0.98, (counts[k % len(counts)], 3))) * 0.1)
    x = np.ones((sum(len(q) for q in pos), 4), np.float32)
    x[:, :3] = np.concatenate(pos)
    return p, x[rng.permutation(x.shape[0])]


# cell counts: vacancies; a group's 8 and 16 lanes and one more or less; columns of
# 3 cells at 31 / 32 / 33 slots; lists up to their 96 entries and longer ones
@pytest.mark.parametrize("counts", [(0, 0, 0, 1), (7, 8, 9), (15, 16, 17, 0), (10, 11, 10, 11, 12), (5, 40, 0, 3)])
@pytest.mark.parametrize("tile_bits,small_max", [(5, 0), (5, 64), (6, 64)])
def test_gpu_tile_lists_match_oracle(F, O, counts, tile_bits, small_max):
    p, x = _crowded(F, counts)
    p.tile_bits = tile_bits
    n = x.shape[0]
    print(f"tile lists: counts {counts}, n {n}, tile bits {tile_bits}, small tiles up to {small_max}", flush=True)
    ctx = F.Context(p, n)
    ctx.add_particles(x)
    ctx.set_launch_shape(small_tile_max=small_max)
    ctx.compute()
    got = {k: ctx.download(k) for k in ("cell_ids", "particle_ids", "neighbour_counters", "densities", "lambdas",
                                        "delta_positions", "omegas")}
    ctx.close()
    out = O.step(p, O.State(x))
    assert np.array_equal(got["cell_ids"], out["keys"]) and np.array_equal(got["particle_ids"], out["ids"])
    assert np.array_equal(got["neighbour_counters"], out["nbr_count"])
    # a sum of up to 1e3 positive float32 terms, each within a few roundings: 1e-5 of the
    # largest; lambda a quotient of two such sums: 1e-4 (the tolerances of the parity tests)
    assert np.abs(got["densities"] - out["density"]).max() <= 1e-5 * out["density"].max()
    assert np.abs(got["lambdas"] - out["lambda"]).max() <= 1e-4 * np.abs(out["lambda"]).max()
    dp = np.abs(out["dp4"][:, :3]).max()
    assert np.abs(got["delta_positions"][:, :3] - out["dp4"][:, :3]).max() <= 1e-4 * dp


def test_gpu_tile_lists_leave_nan_neighbours_out(F):
    """A particle whose position is not a number (either sign of NaN) is in nobody's
    list: the others step as they do without it."""
    p, x = _crowded(F, (6, 8))
    n = x.shape[0]

    def step(extra):
        ctx = F.Context(p, n + len(extra))
        ctx.add_particles(np.concatenate([x, np.array(extra, np.float32).reshape(-1, 4)]))
        ctx.compute()
        keep = ctx.download("particle_ids") < n
        out = {k: ctx.download(k)[keep] for k in ("densities", "lambdas", "positions")}
        ctx.close()
        return out

    nan = np.float32(np.nan)
    print("NaN neighbours", flush=True)
    ref, got = step([]), step([[nan, 0.05, 0.05, 1.0], [0.05, -nan, 0.05, 1.0], [-nan, -nan, -nan, 1.0]])
    for k in ref:
        assert np.array_equal(ref[k], got[k]), k


def test_gpu_tile_lists_leave_nan_neighbours_out_of_later_passes(F):
    """The same for the passes that follow a delta p pass, with its moves not applied (an
    applied one puts the particle onto the enclosure)."""
    p, x = _crowded(F, (6, 8))
    p.solver_iterations = 3
    p.stabilization_iterations = 1
    p.active_apply_delta_positions = 0
    n = x.shape[0]

    def step(extra):
        ctx = F.Context(p, n + len(extra))
        ctx.add_particles(np.concatenate([x, np.array(extra, np.float32).reshape(-1, 4)]))
        ctx.compute()
        keep = ctx.download("particle_ids") < n
        out = {k: ctx.download(k)[keep] for k in ("densities", "lambdas", "positions", "omegas")}
        ctx.close()
        return out

    nan = np.float32(np.nan)
    print("NaN neighbours, later passes", flush=True)
    ref, got = step([]), step([[nan, 0.05, 0.05, 1.0], [0.05, -nan, 0.05, 1.0], [-nan, -nan, -nan, 1.0]])
    for k in ref:
        assert np.array_equal(ref[k], got[k]), k
