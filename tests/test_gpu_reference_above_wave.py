"""The reference variant just above the 98,304 particles up to which its passes take a wave
per particle: the thread-per-particle kernels at a two-cell stencil against the oracle, all
outputs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_gpu_reference_above_the_wave_passes(F, O):
    p = F.load_params(F.config_path("reference"))
    rng = np.random.default_rng(8)
    at = np.indices((47, 46, 46)).reshape(3, -1).T
    n = len(at)
    assert 98304 < n < 100000
    pos, vel, col = np.ones((n, 4), np.float32), np.zeros((n, 4), np.float32), np.ones((n, 4), np.float32)
    pos[:, :3] = 4.0 + 1.2 * at + rng.uniform(-0.05, 0.05, (n, 3))  # inside the enclosure, up to 62.5
    vel[:, :3] = rng.normal(0.0, 0.5, (n, 3))
    p.box_spawn_in_the_beginning = 0
    # the summed outputs of one set of positions
    p.active_apply_delta_positions = 0
    p.stabilization_iterations = 0
    print(f"reference variant, n {n}", flush=True)
    ctx = F.Context(p, n)
    ctx.add_particles(pos, vel, col)
    ctx.compute()
    got = {k: ctx.download(k) for k in ("cell_ids", "particle_ids", "neighbour_counters", "contact_counters", "densities",
                                        "lambdas", "delta_positions", "omegas", "positions", "velocities",
                                        "external_forces")}
    ctx.close()
    out = O.step(p, O.State(pos, vel, col))
    for k, o in (("cell_ids", "keys"), ("particle_ids", "ids"), ("neighbour_counters", "nbr_count"),
                 ("contact_counters", "contact_count")):
        assert np.array_equal(got[k], out[o]), k
    assert np.abs(got["densities"] - out["density"]).max() <= 1e-5 * out["density"].max()
    assert np.abs(got["lambdas"] - out["lambda"]).max() <= 1e-4 * np.abs(out["lambda"]).max()
    d = O.derive(p)

    def err(k, o):
        return np.abs(got[k][:, :3] - out[o][:, :3]).max(axis=1)

    assert err("positions", "x4").max() <= 1e-5 * d.h_spiky
    assert err("velocities", "v4").max() <= 1e-5 * d.h_spiky / d.dt
    # signed sums of about 70 terms
    for k, o in (("delta_positions", "dp4"), ("omegas", "omega3")):
        assert err(k, o).max() <= 1e-4 * np.abs(out[o][:, :3]).max(), k
    # a vorticity force divides by differences of coordinates: 95 % of the particles
    f = np.abs(out["f4"][:, :3]).max()
    assert (err("external_forces", "f4") > 2e-3 * f + 1e-6 * abs(p.gravity)).mean() <= 0.05
