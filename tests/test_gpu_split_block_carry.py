"""Lists carried from substep to substep where blocks are two items (halos of more than 1528
particles): the halves of calm blocks keep theirs, and a block that becomes one item or two
between substeps, or holds more than the halves do, steps as with lists rebuilt in every
pass, bit for bit, in every output."""
import numpy as np
import pytest

from test_gpu_wide_tiles import _scene

pytestmark = pytest.mark.gpu

OUTPUTS = ("cell_ids", "particle_ids", "neighbour_counters", "densities", "lambdas", "delta_positions", "omegas",
           "positions", "predicted", "velocities", "colors", "external_forces")


def _run(F, p, x, v, small, skin, steps):
    ctx = F.Context(p, len(x))
    ctx.add_particles(x, v)
    ctx.set_launch_shape(small_tile_max=small, list_skin_pct=skin)
    ctx.reset_counters()
    out = []
    for _ in range(steps):
        ctx.compute()
        out.append({k: ctx.download(k) for k in OUTPUTS})
    counters = ctx.counters()
    ctx.close()
    return out, counters


def _same(a, b):
    for s, (u, w) in enumerate(zip(a, b)):
        for k in OUTPUTS:
            assert np.array_equal(u[k], w[k]), (s, k)


# blocks past a tile's capacity (halos of 1700 to 1800) everywhere but at the walls
@pytest.mark.parametrize("small", [0, 64])
@pytest.mark.parametrize("counts", [(12, 12, 13), (11, 12, 13)])
def test_gpu_split_blocks_carry_their_lists(F, small, counts):
    p, x, v = _scene(F, (8, 12, 12), counts, 0.98)
    p.active_apply_delta_positions = 0  # calm: nothing moves but by its velocity
    v *= 0.0
    print(f"split blocks at rest: counts {counts}, small {small}, n {len(x)}", flush=True)
    want, _ = _run(F, p, x, v, small, 0, 4)
    got, c = _run(F, p, x, v, small, 10, 4)
    _same(want, got)
    print(f"  {c}", flush=True)
    # from the second substep on, three of four lambda passes and the omega pass keep the
    # lists of every tile, halves among them: 4 passes of 3 substeps
    assert c["unlisted_block"] == 0
    assert c["list_carries"] + c["unlisted_cap"] >= 0.99 * 12 * len(x)


# halos around 1528 and particles that change cells: blocks become one item and two from
# substep to substep; with moves past the skin in every pass (the corrections of particles
# at random places, nothing carries) and, the corrections not applied, without
@pytest.mark.parametrize("small", [0, 64])
@pytest.mark.parametrize("speed", [0.05, 0.6])
@pytest.mark.parametrize("applied", [1, 0])
def test_gpu_blocks_split_and_join_between_substeps(F, small, speed, applied):
    p, x, v = _scene(F, (8, 12, 12), (10, 11, 11), 0.98, seed=17)
    rng = np.random.default_rng(5)
    v[:, :3] = rng.normal(0.0, speed, (len(x), 3))
    p.active_apply_delta_positions = applied
    print(f"blocks split and join: speed {speed}, small {small}, applied {applied}, n {len(x)}", flush=True)
    want, _ = _run(F, p, x, v, small, 0, 5)
    got, c = _run(F, p, x, v, small, 20, 5)
    _same(want, got)
    print(f"  {c}", flush=True)
    if not applied:
        assert c["list_carries"] > 0


@pytest.mark.parametrize("small", [0, 64])
def test_gpu_crowded_blocks_keep_nothing_they_should_not(F, small):
    """Cells of 8 to 34 particles: halves past the capacity as well."""
    p, x, v = _scene(F, (8, 8, 8), (8, 20, 8, 34, 12), 0.98, seed=23)
    print(f"crowded blocks: small {small}, n {len(x)}", flush=True)
    want, _ = _run(F, p, x, v, small, 0, 4)
    got, _ = _run(F, p, x, v, small, 30, 4)
    _same(want, got)
