"""The reference variant's passes with a wave per particle past the 256 neighbours that a
wave's list holds at a time: every output against the passes with a thread per particle
(which a context with friction takes, also where no particle is solid) and the oracle, and
no step of a crowded scene costs what one lane's walk of each particle did."""
import time

import numpy as np
import pytest

from test_gpu_wave_passes import _scene

pytestmark = pytest.mark.gpu

OUTPUTS = ("cell_ids", "particle_ids", "neighbour_counters", "contact_counters", "densities", "lambdas",
           "delta_positions", "omegas", "positions", "predicted", "velocities", "colors", "external_forces")


def _step(F, p, x, v, steps=1):
    ctx = F.Context(p, len(x))
    ctx.add_particles(x, v)
    for _ in range(steps):
        ctx.compute()
    got = {k: ctx.download(k) for k in OUTPUTS}
    ctx.close()
    return got


# lists of about 70, 230, 380 and more than 512 entries (cut off at the cap), and of exactly
# one window, one entry less and one more
@pytest.mark.parametrize("per_cell,cap", [(0.6, 512), (2.0, 512), (4.0, 512), (9.0, 512), (4.0, 255), (4.0, 256),
                                          (4.0, 257), (9.0, 700)])
@pytest.mark.parametrize("kw", [1, 2])
@pytest.mark.parametrize("gate", [None, "active_find_contacts", "active_compute_delta_positions"])
def test_gpu_wave_passes_equal_thread_passes(F, per_cell, cap, kw, gate):
    p, x, v = _scene(F, per_cell, n=900)
    p.kernel_width_neighbours = kw
    p.max_neighbours_per_particle = cap
    if gate:
        setattr(p, gate, 0)
    q = p.copy()
    q.friction_static, q.friction_kinetic = 0.5, 0.4
    print(f"wave lists: {per_cell} a cell, cap {cap}, stencil {kw}, gate {gate}", flush=True)
    wave, thread = _step(F, p, x, v, 2), _step(F, q, x, v, 2)
    for k in OUTPUTS:
        assert np.array_equal(wave[k], thread[k]), (k, np.abs(wave[k].astype(float) - thread[k]).max())


@pytest.mark.parametrize("per_cell", [2.0, 4.0, 9.0])
def test_gpu_wave_lists_match_oracle(F, O, per_cell):
    p, x, v = _scene(F, per_cell)
    # the summed outputs of one set of positions: no delta p applied before omega
    p.active_apply_delta_positions = 0
    p.stabilization_iterations = 0
    print(f"wave lists against the oracle: {per_cell} a cell", flush=True)
    got = _step(F, p, x, v)
    out = O.step(p, O.State(x, v))
    for k, o in (("cell_ids", "keys"), ("particle_ids", "ids"), ("neighbour_counters", "nbr_count"),
                 ("contact_counters", "contact_count")):
        assert np.array_equal(got[k], out[o]), k
    # sums of up to 512 float32 terms: 1e-5 of the largest density, 1e-4 of the largest lambda;
    # signed sums of up to 512 terms whose rounding (512 ulp at worst) is that of the largest
    assert np.abs(got["densities"] - out["density"]).max() <= 1e-5 * out["density"].max()
    assert np.abs(got["lambdas"] - out["lambda"]).max() <= 1e-4 * np.abs(out["lambda"]).max()
    for k, o in (("delta_positions", "dp4"), ("omegas", "omega3")):
        ref = out[o][:, :3]
        assert np.abs(got[k][:, :3] - ref).max() <= 1e-4 * np.abs(ref).max(), k


def test_gpu_wave_lists_cost(F):
    """A step of 30,000 particles with lists of about 400 takes no longer than one of 100,000,
    which go a thread per particle (with one lane walking, it took 2.8 times as long)."""
    ms = {}
    for n in (30000, 100000):
        p, x, v = _scene(F, 4.0, n=n)
        for a in range(3):
            p.grid_dims[a] = 64
        ctx = F.Context(p, n)
        ctx.add_particles(x, v)
        ctx.step(2, graph=True)
        ctx.sync()
        best = float("inf")
        for _ in range(5):
            t = time.perf_counter()
            ctx.step(4, graph=True)
            ctx.sync()
            best = min(best, time.perf_counter() - t)
        ctx.close()
        ms[n] = best / 4 * 1e3
        print(f"wave lists: {n} particles {ms[n]:.3f} ms a step", flush=True)
    assert ms[30000] <= ms[100000]
