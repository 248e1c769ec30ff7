"""Solver iterations around the 8 that lists are carried over: the textbook passes on
tiles run any number of them, with four lanes per particle and with one, and agree with
the oracle."""
import pytest

from conftest import small_dam
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
