"""Which blocks are small tiles (one wave each): up to 64 particles, and above 8 only if
the halo fits the 272 slots (630 of 2^6-cell blocks) a small tile holds; and blocks whose
halo exceeds the 1352 slots of a tile, which are two items."""
import numpy as np
import pytest

from conftest import small_dam

pytestmark = pytest.mark.gpu


def _block_scene(F, bits, own, halo, seed=5):
    """A block of 2^bits cells with `own` particles, `halo` in all with the ring of cells around it."""
    p = small_dam(F, 8)
    p.box_spawn_in_the_beginning = 0
    p.gravity = 0.0
    p.tile_bits = bits
    p.solver_iterations = 1
    p.stabilization_iterations = 0
    lo, ext = np.array([4, 4, 4]), np.array([2 if bits == 5 else 4, 4, 4])
    for a in range(3):
        p.grid_dims[a] = 12
        p.bounds_min[a] = 0.0
        p.bounds_max[a] = 1.2
    g = np.indices(ext + 2).reshape(3, -1).T - 1
    inside = ((g >= 0) & (g < ext)).all(1)
    count = np.zeros(len(g), int)
    for cells, total in ((np.flatnonzero(inside), own), (np.flatnonzero(~inside), halo - own)):
        count[cells] = total // len(cells)
        count[cells[:total % len(cells)]] += 1
    rng = np.random.default_rng(seed)
    x = np.ones((halo, 4), np.float32)
    x[:, :3] = (np.repeat(lo + g, count, 0) + rng.uniform(0.02, 0.98, (halo, 3))) * 0.1
    return p, x[rng.permutation(halo)]


@pytest.mark.parametrize("bits,cap", [(5, 272), (6, 630)])
@pytest.mark.parametrize("own,more", [(33, 0), (33, 1), (64, -1), (64, 0), (64, 1), (64, 300), (65, 1), (8, 0)])
def test_gpu_small_tiles_match_oracle(F, O, bits, cap, own, more):
    p, x = _block_scene(F, bits, own, cap + more)
    n = len(x)
    print(f"small tiles: bits {bits}, own {own}, halo {n}", flush=True)
    ctx = F.Context(p, n)
    ctx.add_particles(x)
    ctx.set_launch_shape(small_tile_max=64)
    ctx.compute()
    got = {k: ctx.download(k) for k in ("cell_ids", "particle_ids", "neighbour_counters", "densities", "lambdas")}
    left = ctx.counters()["unlisted_block"]
    ctx.close()
    out = O.step(p, O.State(x))
    assert np.array_equal(got["cell_ids"], out["keys"]) and np.array_equal(got["particle_ids"], out["ids"])
    assert np.array_equal(got["neighbour_counters"], out["nbr_count"])
    # the tolerances of the parity tests: sums of positive float32 terms, a quotient of two
    assert np.abs(got["densities"] - out["density"]).max() <= 1e-5 * out["density"].max()
    assert np.abs(got["lambdas"] - out["lambda"]).max() <= 1e-4 * np.abs(out["lambda"]).max()
    # no block is left to the passes over global memory
    assert left == 0


# halves: at and past the capacity, all own particles in one half, halves too crowded as well
@pytest.mark.parametrize("own,halo", [(300, 1352), (300, 1353), (64, 1500), (65, 1500), (300, 1920), (520, 2300)])
@pytest.mark.parametrize("small", [0, 64])
@pytest.mark.parametrize("side", [None, 0, 1])
def test_gpu_split_blocks_match_oracle(F, O, own, halo, small, side):
    p, x = _block_scene(F, 5, own, halo)
    p.solver_iterations = 2
    p.active_apply_delta_positions = 0  # the second pass may keep its lists
    if side is not None:  # own particles of y 4 to 7 cells into y 4, 5 or 6, 7
        c = np.floor(x[:, :3] / np.float32(0.1))
        inside = ((c >= 4) & (c < [6, 8, 8])).all(1)
        y = x[inside, 1]
        x[inside, 1] = 0.4 + 0.2 * side + np.mod(y, 0.2) * 0.95 + 0.005
    n = len(x)
    print(f"split blocks: own {own}, halo {n}, small {small}, side {side}", flush=True)
    ctx = F.Context(p, n)
    ctx.add_particles(x)
    ctx.set_launch_shape(small_tile_max=small)
    ctx.compute()
    got = {k: ctx.download(k) for k in ("cell_ids", "particle_ids", "neighbour_counters", "densities", "lambdas",
                                        "delta_positions")}
    ctx.close()
    out = O.step(p, O.State(x))
    assert np.array_equal(got["cell_ids"], out["keys"]) and np.array_equal(got["particle_ids"], out["ids"])
    assert np.array_equal(got["neighbour_counters"], out["nbr_count"])
    assert np.abs(got["densities"] - out["density"]).max() <= 1e-5 * out["density"].max()
    assert np.abs(got["lambdas"] - out["lambda"]).max() <= 1e-4 * np.abs(out["lambda"]).max()
    dp = np.abs(out["dp4"][:, :3]).max()
    assert np.abs(got["delta_positions"][:, :3] - out["dp4"][:, :3]).max() <= 1e-4 * dp
