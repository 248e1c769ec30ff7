"""The reference variant's passes with a wave per particle: stencils of one and two cells,
lists shorter and longer than 64 pairs (a round of the lanes) and 256 (what a wave's list
holds), the neighbour cap inside and past them, gates off, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _scene(F, per_cell, n=600, seed=3):
    """n particles spread over a cube at per_cell particles a cell, away from the walls."""
    p = F.default_params()
    p.box_spawn_in_the_beginning = 0
    p.gravity = 0.0
    for a in range(3):
        p.grid_dims[a] = 32
    rng = np.random.default_rng(seed)
    side = (n / per_cell) ** (1.0 / 3.0)
    x = np.ones((n, 4), np.float32)
    x[:, :3] = 8.0 + rng.uniform(0.0, side, (n, 3))
    v = np.zeros((n, 4), np.float32)
    v[:, :3] = rng.normal(0.0, 0.5, (n, 3))
    return p, x, v


# per cell: lists of about 20, 70, 230 and 380 of two-cell stencils, 16 to 80 of one-cell ones
@pytest.mark.parametrize("per_cell", [0.15, 0.6, 2.0, 4.0])
@pytest.mark.parametrize("kw,cap", [(1, 512), (2, 512), (2, 64), (2, 300), (3, 512)])
def test_gpu_wave_passes_match_oracle(F, O, per_cell, kw, cap):
    p, x, v = _scene(F, per_cell)
    p.kernel_width_neighbours = kw
    p.max_neighbours_per_particle = cap
    n = x.shape[0]
    print(f"wave passes: {per_cell} a cell, stencil {kw}, cap {cap}", flush=True)
    ctx = F.Context(p, n)
    ctx.add_particles(x, v)
    ctx.compute()
    got = {k: ctx.download(k) for k in ("cell_ids", "particle_ids", "neighbour_counters", "contact_counters",
                                        "densities", "lambdas")}
    ctx.close()
    out = O.step(p, O.State(x, v))
    assert np.array_equal(got["cell_ids"], out["keys"]) and np.array_equal(got["particle_ids"], out["ids"])
    assert np.array_equal(got["neighbour_counters"], out["nbr_count"])
    assert np.array_equal(got["contact_counters"], out["contact_count"])
    # sums of up to 512 float32 terms: 1e-5 of the largest density, 1e-4 of the largest lambda
    assert np.abs(got["densities"] - out["density"]).max() <= 1e-5 * out["density"].max()
    assert np.abs(got["lambdas"] - out["lambda"]).max() <= 1e-4 * np.abs(out["lambda"]).max()


@pytest.mark.parametrize("gate", ["active_find_contacts", "active_find_neighbours", "active_compute_delta_positions",
                                  "active_compute_vorticity", "active_compute_viscosity"])
def test_gpu_wave_passes_gates(F, O, gate):
    p, x, v = _scene(F, 0.6)
    setattr(p, gate, 0)
    print(f"wave passes: {gate} off", flush=True)
    ctx = F.Context(p, x.shape[0])
    ctx.add_particles(x, v)
    ctx.compute()
    cnt, lam, gx = ctx.download("neighbour_counters"), ctx.download("lambdas"), ctx.download("positions")
    ctx.close()
    out = O.step(p, O.State(x, v))
    assert np.array_equal(cnt, out["nbr_count"])
    assert np.abs(lam - out["lambda"]).max() <= 1e-4 * np.abs(out["lambda"]).max()
    # world positions near 16: a float32 ulp is 1e-6; a handful of roundings of pushes below 0.5
    assert np.quantile(np.abs(gx[:, :3] - out["x4"][:, :3]).max(axis=1), 0.99) <= 1e-5
