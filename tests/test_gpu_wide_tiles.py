"""The lambda and omega passes with four lanes per particle at their edges: columns of
0 to 90 slots (two 32-slot scans are kept, the rest scanned again), lists up to 96 pairs
and longer ones (no list), blocks of a few particles, of more than a round's 256 and past
the halo's LDS capacity, kept lists, and the particle count where a lane per particle
takes over."""
import numpy as np
import pytest

from conftest import small_dam

pytestmark = pytest.mark.gpu


def _scene(F, dims, counts, spread, seed=11):
    """Cell k of a grid of `dims` cells holds counts[k mod len] particles within its middle `spread`."""
    p = small_dam(F, 8)
    p.box_spawn_in_the_beginning = 0
    p.gravity = 0.0
    p.tile_bits = 5
    for a in range(3):
        p.grid_dims[a] = dims[a]
        p.bounds_min[a] = 0.0
        p.bounds_max[a] = dims[a] * 0.1
    p.stabilization_iterations = 0
    rng = np.random.default_rng(seed)
    pos = []
    for k in range(dims[0] * dims[1] * dims[2]):
        c = np.array([k // (dims[1] * dims[2]), (k // dims[2]) % dims[1], k % dims[2]])
        pos.append((c + 0.5 + spread * rng.uniform(-0.5, 0.5, (counts[k % len(counts)], 3))) * 0.1)
    x = np.ones((sum(len(q) for q in pos), 4), np.float32)
    x[:, :3] = np.concatenate(pos)
    v = np.zeros_like(x)
    v[:, :3] = rng.normal(0.0, 0.05, (len(x), 3))
    order = rng.permutation(len(x))
    return p, x[order], v[order]


def _check(F, O, p, x, v):
    n = len(x)
    ctx = F.Context(p, n)
    ctx.add_particles(x, v)
    ctx.compute()
    got = {k: ctx.download(k) for k in ("cell_ids", "particle_ids", "neighbour_counters", "densities", "lambdas", "omegas")}
    ctx.close()
    out = O.step(p, O.State(x, v))
    assert np.array_equal(got["cell_ids"], out["keys"]) and np.array_equal(got["particle_ids"], out["ids"])
    assert np.array_equal(got["neighbour_counters"], out["nbr_count"])
    # a sum of up to 1e3 positive float32 terms, each within a few roundings: 1e-5 of the
    # largest; lambda a quotient of two such sums and omega a sum of signed ones: 1e-4
    # (the tolerances of the parity tests)
    assert np.abs(got["densities"] - out["density"]).max() <= 1e-5 * out["density"].max()
    assert np.abs(got["lambdas"] - out["lambda"]).max() <= 1e-4 * np.abs(out["lambda"]).max()
    # omega only where no delta p was applied: pushed apart from almost the same place, a
    # pair's direction is rounding
    om = out["omega3"][:, :3]
    if not p.active_apply_delta_positions:
        assert np.abs(got["omegas"][:, :3] - om).max() <= 1e-4 * np.abs(om).max()


# per cell: lone particles; columns of 3 cells at 30 to 36 slots; lists around 96 pairs;
# columns of 60 to 90 slots with few pairs apart; halos past the capacity
@pytest.mark.parametrize("counts,spread", [((1, 0, 0, 0, 0), 0.9), ((10, 11, 12), 0.98), ((4, 5), 0.98),
                                           ((20, 30, 25), 0.98), ((0, 0, 90), 0.3), ((40,), 0.98)])
@pytest.mark.parametrize("iterations", [1, 2])
def test_gpu_wide_tiles_match_oracle(F, O, counts, spread, iterations):
    p, x, v = _scene(F, (8, 8, 8), counts, spread)
    p.solver_iterations = iterations
    if iterations == 2:
        p.active_apply_delta_positions = 0  # the second lambda pass and omega see the same positions
    print(f"wide tiles: counts {counts}, n {len(x)}, iterations {iterations}", flush=True)
    _check(F, O, p, x, v)


# 65536 particles are the last that take four lanes each
@pytest.mark.parametrize("n", [65535, 65536, 65537])
def test_gpu_wide_tiles_line(F, O, n):
    p, x, v = _scene(F, (24, 32, 16), (5, 6), 0.98)
    p.solver_iterations = 1
    x, v = x[:n], v[:n]
    assert len(x) == n
    print(f"wide tiles: n {n}", flush=True)
    _check(F, O, p, x, v)
