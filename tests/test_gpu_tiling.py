"""The Jacobi tiles' edges: every tile lies inside the grid, the first and the
last meet the grid's edges without a halo, waves take one of five forms of the
sweep (interior, tile columns at the grid's sides, grids smaller than a tile,
solid cells, nothing but solid cells).  k sweeps in any tile shape are bitwise
the oracle's k sweeps."""
import numpy as np
import pytest

from natrix_amd import FluidSimulator
from natrix_amd.autotune import SHAPES, lookup, supported
from oracle import fluid as F

pytestmark = pytest.mark.gpu


def _sim(w, h, solid, rng):
    sim = FluidSimulator(w, h)
    if solid is not None:
        sim.set_obstacle_map(solid)
    b = rng.standard_normal((h, w)).astype(np.float32)
    p = rng.standard_normal((h, w)).astype(np.float32)
    sim.upload("divergence", b)
    sim.upload("pressure", p)
    return sim, p, b


def _obstacles(kind, w, h, rng):
    if kind == "none":
        return None
    m = np.zeros((h, w), bool)
    if kind == "block":  # large enough to fill whole waves
        m[h // 4:3 * h // 4, w // 8:7 * w // 8] = True
    elif kind == "edge":  # solid columns and rows on the grid's sides, one cell inside
        m[:, 0] = m[0] = m[-1, w // 2:] = True
        m[h // 2, w // 2] = True
    else:
        m = rng.random((h, w)) < 0.1
    return m


# one tile exactly, one cell more and less than a tile or two, narrower and
# lower than a tile, a single row and column, odd sides
SIZES = [(64, 64), (128, 64), (128, 128), (129, 65), (127, 63), (256, 129), (1, 70), (70, 1),
         (5, 3), (200, 40), (40, 200), (237, 191)]


@pytest.mark.parametrize("w,h", SIZES)
@pytest.mark.parametrize("kind", ["none", "block", "edge", "random"])
def test_every_shape_at_its_edges(gpu, w, h, kind):
    rng = np.random.default_rng(w * 1000 + h)
    sim, p, b = _sim(w, h, _obstacles(kind, w, h, rng), rng)
    obs = F.obstacles_from_mask(sim.download("mask"))
    ref = {k: F.jacobi(p, b, obs, k) for k in (1, 7, 12, 20)}
    for r, wv, c in SHAPES:
        for k in ref:
            if not supported(k, r, wv, c):
                continue
            sim.upload("pressure", p)
            sim.jacobi_blocked(k, k, r, wv, c)
            assert np.array_equal(sim.download("pressure").view(np.uint32),
                                  ref[k].view(np.uint32)), (r, wv, c, k)
    sim.destroy()


def test_tuned_sweeps_of_reduced_storage_are_fixed():
    """Their launches round the pressure, so a retuned table may change the
    shape but not the sweeps per launch."""
    for st in ("bf16", "f16"):
        for side, k in ((96, 12), (256, 12), (512, 16), (700, 16), (900, 10), (1400, 10),
                        (2048, 10), (4096, 10)):
            assert lookup(side, side, st)[0] == k


def test_even_launches_reach_the_sweep_count(gpu):
    """Sweep counts just above and below whole launches: the launches are evened
    out, the sweeps are not."""
    rng = np.random.default_rng(3)
    sim, p, b = _sim(150, 90, None, rng)
    obs = F.obstacles_from_mask(sim.download("mask"))
    for n in (1, 23, 24, 25, 47, 49, 73):
        sim.upload("pressure", p)
        sim.jacobi_blocked(n, 24, 8, 8, 1)
        assert np.array_equal(sim.download("pressure"), F.jacobi(p, b, obs, n)), n
    sim.destroy()


@pytest.mark.parametrize("tile", [(8, 8, 8, 1), (12, 4, 16, 1), (8, 4, 8, 2), (20, 8, 8, 2)])
def test_residual_records_of_several_tiles(gpu, tile):
    """A tolerance solve on several uneven tiles with solids stops at the check,
    every ceil(60 / k) k sweeps, at which the oracle's residual meets the
    tolerance: each cell is in one tile's record."""
    w, h, tol = 150, 90, 1.5e-3
    rng = np.random.default_rng(8)
    y, x = np.mgrid[0:h, 0:w]
    solid = (x - 60) ** 2 + (y - 40) ** 2 <= 100
    solid[:, 100] = rng.random(h) < 0.5
    sim = FluidSimulator(w, h, bc_mode="free_slip")
    sim.vorticity, sim.viscosity = 0.3, 0.0
    sim.jacobi_tile, sim.tol, sim.check_every = tile, tol, 60
    sim.set_obstacle_map(solid)
    sim.upload("velocity", rng.uniform(-0.5, 0.5, (h, w, 2)).astype(np.float32))
    obs = F.obstacles_from_mask(sim.download("mask"))
    sim.update(1 / 60)
    st, got, b = sim.stats(), sim.download("pressure"), sim.download("divergence")
    sim.destroy()
    chunk = -(-60 // tile[0]) * tile[0]
    p, sweeps, checks = (np.float32(0) - b) * np.float32(0.25), 1, 0
    while checks < 400:
        before = F.jacobi(p, b, obs, chunk - 1)
        p = F.jacobi(before, b, obs, 1)
        sweeps, checks = sweeps + chunk, checks + 1
        if F.relative_residual(before, b, obs) <= tol and F.relative_residual(p, b, obs) <= tol:
            break
    assert st["converged"] and st["sweeps"] == sweeps and checks > 3
    assert np.array_equal(got, p)
    assert abs(st["residual"] - F.relative_residual(p, b, obs)) <= 1e-9
