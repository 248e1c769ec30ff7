"""Split blocks (halos of more than 1528 particles) beyond the plain step: with solids and
friction against the oracle, and on the capped grid of boxes with more than 2^20 blocks
against the direct one; and the edges of whole, split and small tiles."""
import numpy as np
import pytest

from conftest import small_dam
from test_gpu_phases import _ctx
from test_gpu_small_tiles import _block_scene
from test_gpu_wide_tiles import _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("small", [0, 64])
def test_gpu_split_blocks_with_solids_match_oracle(F, O, small):
    """A 22^3 lattice pressed together to 11.7 particles a cell (halos of about 1700), a third of
    it solid: positions, velocities and phases of one step, by the bounds of the mixed step."""
    p = small_dam(F, 22)
    p.friction_static = 0.5
    p.friction_kinetic = 0.4
    p.box_solid_fraction = 0.3
    p.box_solid_radius = 0.1
    p.solver_iterations = 1
    pos, vel, col = F.generate_box(p)
    ph = F.capi.generate_phases(p)
    pos[:, :3] *= np.float32(0.88)
    rng = np.random.default_rng(6)
    vel[:, :3] = rng.normal(0.0, 0.2, (len(pos), 3)).astype(np.float32)
    print(f"split blocks with solids: n {len(pos)}, small {small}", flush=True)
    ctx = _ctx(F, p, pos, vel, col, ph)
    ctx.set_launch_shape(small_tile_max=small)
    ctx.compute()
    got = {k: ctx.download(k) for k in ("cell_ids", "particle_ids", "neighbour_counters", "densities", "positions",
                                        "velocities", "phases")}
    unlisted = ctx.counters()["unlisted_block"]
    ctx.close()
    st = O.State(pos, vel, col, phase=ph)
    out = O.step(p, st)
    assert np.array_equal(got["cell_ids"], out["keys"]) and np.array_equal(got["particle_ids"], out["ids"])
    assert np.array_equal(got["neighbour_counters"], out["nbr_count"]) and np.array_equal(got["phases"], st.phase)
    count = np.bincount(np.unique(out["keys"] >> 5, return_inverse=True)[1])
    assert (count > 340).sum() >= 8  # crowded blocks, 375 in the full ones
    assert unlisted == 0
    assert np.abs(got["densities"] - out["density"]).max() <= 1e-5 * out["density"].max()
    h, dt = float(p.kernel_width_poly), O.derive(p).dt
    err = np.abs(got["positions"][:, :3] - out["x4"][:, :3]).max(axis=1)
    verr = np.abs(got["velocities"][:, :3] - out["v4"][:, :3]).max(axis=1)
    print(f"  position error: max {err.max():.2e}, 99.9th pct {np.quantile(err, 0.999):.2e}", flush=True)
    assert np.quantile(err, 0.999) < 1e-5 * h and err.max() < 1e-3 * h
    assert np.quantile(verr, 0.999) < 1e-5 * h / dt


def test_gpu_split_blocks_on_the_capped_grid(F):
    """1.25M particles at 11 and 12 a cell in a grid of 48 x 48 x 48 cells and in one of 48 x 48 x
    520, whose 2^22 blocks take the capped grid: the same cells and counts, the same outputs but
    for the rounding of two sets of kernels."""
    runs = []
    for depth in (48, 520):
        p, x, v = _scene(F, (48, 48, 48), (11, 11, 12), 0.98)
        p.grid_dims[2] = depth
        p.solver_iterations = 2
        p.active_apply_delta_positions = 0  # the sums of one set of positions
        print(f"split blocks, grid depth {depth}: n {len(x)}", flush=True)
        ctx = F.Context(p, len(x))
        ctx.add_particles(x, v)
        ctx.compute()
        runs.append({k: ctx.download(k) for k in ("cell_ids", "particle_ids", "neighbour_counters", "densities",
                                                  "lambdas", "delta_positions", "omegas", "velocities", "positions")})
        runs[-1]["unlisted"] = ctx.counters()["unlisted_block"]
        ctx.close()
    a, b = runs
    for k in ("cell_ids", "particle_ids", "neighbour_counters", "unlisted"):
        assert np.array_equal(a[k], b[k]), k
    # sums of float32 terms in one order: within the parity tests' bounds of the oracle's
    for k, tol in (("densities", 1e-5), ("lambdas", 1e-4), ("delta_positions", 1e-4), ("omegas", 1e-4),
                   ("velocities", 1e-5), ("positions", 1e-6)):
        assert np.abs(a[k] - b[k]).max() <= tol * np.abs(a[k]).max(), k


# at and past a tile's 1528 slots; halves at their own capacity and past it
@pytest.mark.parametrize("own,halo", [(300, 1528), (300, 1529), (65, 1529), (520, 2300), (520, 2700)])
@pytest.mark.parametrize("small", [0, 64])
def test_gpu_blocks_at_the_tile_capacity_match_oracle(F, O, own, halo, small):
    p, x = _block_scene(F, 5, own, halo)
    p.solver_iterations = 2
    p.active_apply_delta_positions = 0
    _match(F, O, p, x, small, f"own {own}, halo {halo}")


@pytest.mark.parametrize("small", [0, 64])
def test_gpu_layered_blocks_stay_on_tiles(F, O, small):
    """Layers of 9, 20, 20 and 9 particles a cell along y: the middle ones are in the halos of
    both halves of a block (1392 particles each of the block's 1824), which hold them."""
    p, x, _ = _scene(F, (6, 12, 12), (1,), 0.98)
    c = np.indices((6, 12, 12)).reshape(3, -1).T
    c = np.repeat(c, np.where((c[:, 1] % 4 == 1) | (c[:, 1] % 4 == 2), 20, 9), 0)
    x = np.ones((len(c), 4), np.float32)
    x[:, :3] = (c + np.random.default_rng(3).uniform(0.02, 0.98, c.shape)) * 0.1
    p.solver_iterations = 2
    p.active_apply_delta_positions = 0
    assert _match(F, O, p, x, small, "layers") == 0



# a small tile's 312 slots
@pytest.mark.parametrize("own,halo", [(12, 312), (12, 313), (64, 312), (64, 313), (9, 1400)])
def test_gpu_small_blocks_at_their_capacity_stay_on_tiles(F, O, own, halo):
    p, x = _block_scene(F, 5, own, halo)
    p.solver_iterations = 2
    p.active_apply_delta_positions = 0
    assert _match(F, O, p, x, 64, f"own {own}, halo {halo}") == 0


def test_gpu_few_particles_beside_a_crowd_stay_on_tiles(F, O):
    """A column of 9 particles a cell with spray beside it, one or two particles in a block
    whose halo holds 300 and more: no particle is walked from global memory."""
    p, _, _ = _scene(F, (32, 32, 32), (1,), 0.98)
    c = np.indices((32, 32, 32)).reshape(3, -1).T
    rng = np.random.default_rng(12)
    spray = (c[:, 0] >= 16) & (rng.uniform(size=len(c)) < 0.04)
    c = np.repeat(c, np.where(c[:, 0] < 16, 9, spray.astype(int)), 0)
    x = np.ones((len(c), 4), np.float32)
    x[:, :3] = (c + rng.uniform(0.02, 0.98, c.shape)) * 0.1
    assert len(x) > 1 << 16  # where small tiles are on by default
    p.solver_iterations = 2
    p.active_apply_delta_positions = 0
    assert _match(F, O, p, x, None, "spray") == 0


def _match(F, O, p, x, small, label):
    """One step against the oracle by the parity tests' bounds; the particles without a list
    for their block's halo."""
    print(f"tile capacity: {label}, n {len(x)}, small {small}", flush=True)
    ctx = F.Context(p, len(x))
    ctx.add_particles(x)
    if small is not None:
        ctx.set_launch_shape(small_tile_max=small)
    ctx.compute()
    got = {k: ctx.download(k) for k in ("cell_ids", "particle_ids", "neighbour_counters", "densities", "lambdas",
                                        "delta_positions")}
    unlisted = ctx.counters()["unlisted_block"]
    ctx.close()
    out = O.step(p, O.State(x))
    assert np.array_equal(got["cell_ids"], out["keys"]) and np.array_equal(got["particle_ids"], out["ids"])
    assert np.array_equal(got["neighbour_counters"], out["nbr_count"])
    assert np.abs(got["densities"] - out["density"]).max() <= 1e-5 * out["density"].max()
    assert np.abs(got["lambdas"] - out["lambda"]).max() <= 1e-4 * np.abs(out["lambda"]).max()
    dp = np.abs(out["dp4"][:, :3]).max()
    assert np.abs(got["delta_positions"][:, :3] - out["dp4"][:, :3]).max() <= 1e-4 * dp
    return unlisted
