"""Records of a step's arrays by one launch: particle counts whose 4-byte arrays end in 1 to
3 words past the last 16 bytes, one particle, and a record read back after the steps went
on. The reverse of a recorded forward equals that of a forward recorded in pieces."""
import numpy as np
import pytest

from conftest import small_dam

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 1021, 1022, 1023, 4097])
@pytest.mark.parametrize("friction", [0.0, 0.4])
def test_gpu_copy_set_records(F, n, friction):
    p = small_dam(F, 17)
    p.box_spawn_in_the_beginning = 0
    p.friction_static = p.friction_kinetic = friction
    rng = np.random.default_rng(n)
    x = np.ones((n, 4), np.float32)
    x[:, :3] = 0.2 + rng.uniform(0.0, 0.05 * n ** (1.0 / 3.0), (n, 3))
    v = np.zeros((n, 4), np.float32)
    v[:, :3] = rng.normal(0.0, 0.2, (n, 3))
    gx = np.zeros((n, 4), np.float32)
    gx[:, :3] = rng.normal(0.0, 1.0, (n, 3))
    print(f"records: n {n}, friction {friction}", flush=True)
    out = []
    for every in (1, 2):  # checkpoints after every frame and after every second one
        ctx = F.Context(p, n)
        ctx.add_particles(x, v)
        if friction:
            ctx.upload("phases", (np.arange(n) % 3 == 0).astype(np.uint32))
        ctx.adj_forward(4, every)
        state = {k: ctx.download(k) for k in ("positions", "velocities", "predicted", "external_forces", "colors")}
        lam = ctx.download("lambdas")
        g = ctx.adj_backward(gx, None)
        again = {k: ctx.download(k) for k in state}
        ctx.close()
        for k in state:  # the reverse leaves the context as the forward left it
            assert np.array_equal(state[k], again[k], equal_nan=True), k
        out.append((state, lam, g))
    (s1, l1, g1), (s2, l2, g2) = out
    for k in s1:
        assert np.array_equal(s1[k], s2[k], equal_nan=True), k
    assert np.array_equal(l1, l2, equal_nan=True)
    # the same records, read by the same kernels in the same order
    for k in ("v0", "x0"):
        assert np.array_equal(g1[k], g2[k], equal_nan=True), k
