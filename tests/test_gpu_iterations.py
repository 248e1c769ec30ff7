"""Solver iterations around the 8 that lists are carried over: the textbook passes on
tiles run any number of them, with four lanes per particle and with one, and agree with
the oracle."""
import numpy as np
import pytest

from conftest import small_dam
from test_gpu_adjoint import _gpu_grad, _scene
from test_gpu_parity import compare_one_step, developed_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("iterations", [8, 9, 10, 12])
@pytest.mark.parametrize("small", [0, 64])
def test_gpu_iterations_past_the_carried_ones(F, O, iterations, small):
    p = small_dam(F, 12)
    st = developed_state(F, O, p, 2)
    p.solver_iterations = iterations
    compare_one_step(F, O, p, st, f"{iterations} iterations, small tiles up to {small}", conditioned=True,
                     shape={"small_tile_max": small})


def test_gpu_adjoint_past_the_carried_iterations(F, O):
    """The gradient of one substep of 10 iterations, by the bounds of two substeps of 4
    (the parity test of the reverse mode): about as many passes."""
    p, x0, v0, rng = _scene(F, 8)
    p.substeps = 1
    p.delta_t *= 0.5
    p.solver_iterations = 10
    n = x0.shape[0]
    x64, v64 = x0.astype(np.float64), v0.astype(np.float64)
    xf, _, _, orig = O.forward64(p, x64, v64, nsub=1)
    target = xf[np.argsort(orig)] + rng.normal(0.0, 0.01, x0.shape)
    print(f"adjoint of 10 iterations: n {n}", flush=True)
    g, ids, xT = _gpu_grad(F, p, x0, v0, 1, 1, target)
    assert np.abs(xf[np.argsort(orig)] - xT[np.argsort(ids)]).max() < 1e-4
    gx = 2.0 * (xf - target[orig]) / n
    go = O.gradient64(p, x64, v64, gx, np.zeros_like(gx), nsub=1)
    for k in ("v0", "x0"):
        assert np.linalg.norm(g[k] - go[k]) < 1e-3 * np.linalg.norm(go[k]), k
    for k in ("rho0", "eps"):
        assert abs(g[k] - go[k]) < 1e-3 * abs(go[k]), k
