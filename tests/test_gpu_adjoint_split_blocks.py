"""Reverse lists taken from the forward where the forward's blocks are two items (halos of
more than 1528 particles): the gradients of the lists that the reverse builds, bit for bit,
and no block of a halo within the builders' capacity left to the redo pass."""
import numpy as np
import pytest

from test_gpu_adjoint import _ctx, _phased

pytestmark = pytest.mark.gpu


# a thread per (particle, chunk) below 2^19 particles, a thread per particle from there
@pytest.mark.parametrize("side,solids", [(36, False), (36, True), (84, False)])
def test_gpu_adjoint_lists_of_split_blocks(F, side, solids):
    if solids:
        p, x0, v0, ph, rng = _phased(F, side)
    else:
        p = F.load_params(F.config_path("adjoint_64k"))
        p.box_width = p.box_height = p.box_depth = side
        for a in range(3):
            p.bounds_max[a] = side * 0.05 * (2 if a == 0 else 1)
            p.grid_dims[a] = int(np.ceil(p.bounds_max[a] / 0.1))
        pos, _, _ = F.generate_box(p)
        x0, ph = pos[:, :3].astype(np.float32), None
        rng = np.random.default_rng(29)
        v0 = rng.normal(0.0, 0.1, x0.shape).astype(np.float32)
    # 11.7 particles a cell inside the block: halos of about 1700; a slab of y emptied, where
    # the blocks' halves differ
    x0 = x0 * np.float32(0.88)
    keep = np.abs(x0[:, 1] - 0.62) > 0.1
    x0, v0 = x0[keep], v0[keep]
    ph = ph[keep] if ph is not None else None
    n = x0.shape[0]
    target = x0.astype(np.float64) + rng.normal(0.0, 0.05, x0.shape)
    print(f"reverse lists of split blocks: n {n}, solids {solids}", flush=True)
    runs = {}
    for fwd in (True, False):
        ctx = _ctx(F, p, x0, v0)
        if ph is not None:
            ctx.upload("phases", ph)
        ctx.adj_set_lists(fwd)
        ctx.adj_forward(1, 1)
        ids = ctx.adj_ids().astype(np.int64)
        xT = ctx.download("positions")[:, :3].astype(np.float64)
        ctx.reset_counters()
        g = ctx.adj_backward(2.0 * (xT - target[ids]) / n, None)
        cnt = ctx.counters()
        ctx.close()
        print(f"  lists from the forward {fwd}: {cnt}", flush=True)
        runs[fwd] = (g, cnt)
    (g1, c1), (g0, c0) = runs[True], runs[False]
    lists = c1["adj_listed_tile"] + c1["adj_scanned"]
    assert c1["adj_from_forward"] > 0.9 * lists
    kinds = ("adj_listed_tile", "adj_listed_global", "adj_scanned")
    assert sum(c1[k] for k in kinds) == sum(c0[k] for k in kinds)
    assert np.isfinite(g1["v0"]).all()
    for k in ("v0", "x0", "rho0", "eps"):
        assert np.array_equal(g1[k], g0[k]), k
