"""Where a tolerance solve checks its residual decides the sweep it stops at, so
the interval belongs to the grid: a tuned tile's sweeps per launch may be any
number without moving it."""
import numpy as np
import pytest

from natrix_amd import autotune

# sweeps of one launch between which the intervals of these grids are counted
UNIT = {(64, 48): 12, (96, 64): 12, (256, 256): 12, (512, 320): 12, (400, 500): 16,
        (512, 512): 16, (1024, 640): 10, (1000, 700): 10, (1024, 1024): 10, (2048, 2048): 10,
        (3000, 2000): 10, (4096, 4096): 10}


@pytest.mark.parametrize("size,unit", sorted(UNIT.items()))
def test_interval_whatever_the_tile(size, unit):
    for every in (1, 7, 16, 64, 100, 256, 1000, 1024, 1999):
        want = -(-every // unit) * unit
        for k in (autotune.lookup(*size)[0], unit, 13, 20, 24, 28):
            d = autotune.solve_sweeps(*size, k, every)
            assert 1 <= d <= k
            if k >= unit:
                assert -(-every // d) * d == want, (every, k, d)


@pytest.mark.parametrize("size,unit", sorted(UNIT.items()))
def test_reduced_storage_keeps_its_sweeps(size, unit):
    for dtype in ("bf16", "f16"):
        tile = autotune.lookup(*size, dtype)
        assert tile[0] == unit and autotune.supported(*tile)


def test_default_interval_keeps_the_tuned_launches():
    for side in (96, 128, 256, 512, 1024, 2048, 4096):
        k = autotune.lookup(side, side)[0]
        assert autotune.solve_sweeps(side, side, k, 256) == k


@pytest.mark.gpu
@pytest.mark.parametrize("every", [100, 60, 256])
def test_tuned_tile_stops_where_the_unit_does(gpu, every):
    """96 x 64 (unit 12): the tuned tile stops at the same sweep, with the same
    pressure and velocity, as a tile of 12 sweeps a launch."""
    from natrix_amd import FluidSimulator
    w, h = 96, 64
    u = np.random.default_rng(4).uniform(-0.5, 0.5, (h, w, 2)).astype(np.float32)
    got = []
    for tile in (None, (12, 4, 8, 1)):
        sim = FluidSimulator(w, h, bc_mode="inflow")
        sim.vorticity, sim.viscosity = 0.3, 0.0
        if tile:
            sim.jacobi_tile = tile
        sim.tol, sim.check_every = 1e-3, every
        sim.upload("velocity", u)
        sim.update(1 / 60)
        st = sim.stats()
        assert st["converged"]
        got.append((st["sweeps"], sim.download("velocity"), sim.download("pressure")))
        assert (st["sweeps"] - 1) % (-(-every // 12) * 12) == 0
        sim.destroy()
    assert got[0][0] == got[1][0]
    assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][2], got[1][2])
