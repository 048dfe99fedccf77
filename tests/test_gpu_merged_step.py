"""The step's merged form (advection inside the following stages' kernel, the
projection inside the last Jacobi launch) against the oracle and, bitwise,
against the separate launches that a timed simulator runs."""
import numpy as np
import pytest

from natrix_amd import FluidSimulator
from oracle import fluid as F
from oracle import mixed as M

pytestmark = pytest.mark.gpu

BC = {"reference": F.BC_REFERENCE, "free_slip": F.BC_FREE_SLIP, "inflow": F.BC_INFLOW}


def _pair(w, h, storage, bc, visc, iters, seed):
    rng = np.random.default_rng(seed)
    # large velocities: back-traces reach the walls and leave the grid
    u = (1.5 * rng.standard_normal((h, w, 2))).astype(np.float32)
    solid = rng.random((h, w)) < 0.08
    out = []
    for timed in (False, True):
        sim = FluidSimulator(w, h, storage=storage, bc_mode=bc)
        sim.vorticity, sim.viscosity, sim.iterations = 0.3, visc, iters
        sim.set_obstacle_map(solid)
        sim.upload("velocity", u)
        if timed:
            sim.set_timing(True)
        out.append(sim)
    return out, u, solid


# tiles of the stages are 64 x 16 (halo 3 or 4): below, at and above one and two
# tiles, narrower than the halo, and enough tiles for the 256-thread form
@pytest.mark.parametrize("w,h", [(3, 3), (64, 16), (65, 17), (63, 40), (130, 33), (200, 7),
                                 (1300, 700)])
@pytest.mark.parametrize("bc,visc", [("reference", 0.0), ("free_slip", 0.1), ("inflow", 0.0)])
@pytest.mark.parametrize("storage", ["f32", "bf16", "f16"])
def test_merged_equals_separate(gpu, w, h, bc, visc, storage):
    sims, u, solid = _pair(w, h, storage, bc, visc, 14, w + h)
    for step in range(2):
        for sim in sims:
            sim.add_circle_obstacle((0.3, 0.6), 0.2 * min(w, h))
            sim.update(1 / 60)
        for f in ("velocity", "pressure", "divergence", "mask"):
            a, b = (sim.download(f) for sim in sims)
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), (step, f)
    for sim in sims:
        sim.destroy()


@pytest.mark.parametrize("iters", [1, 2, 25, 26])
def test_merged_step_is_the_oracle(gpu, iters):
    """One sweep (no launch to carry the projection) and whole or uneven launches."""
    w, h = 150, 90
    (sim, _), u, solid = _pair(w, h, "f32", "inflow", 0.0, iters, 7)
    sim.update(1 / 60)
    prm = F.Params(vorticity=0.3, viscosity=0.0, iterations=iters, bc_mode=F.BC_INFLOW)
    ref, p, _, _ = F.step(u, np.zeros((h, w), np.float32), np.zeros((h, w, 2), np.float32),
                          np.float32(1 / 60), prm, persistent=solid)
    assert np.array_equal(sim.download("velocity"), ref)
    assert np.array_equal(sim.download("pressure"), p)
    sim.destroy()


@pytest.mark.parametrize("storage", ["f32", "f16"])
def test_graph_of_many_launches_replays(gpu, storage):
    """Steps of ten launches and more are captured; replays, with other work and
    waits between them, give the eager steps."""
    w, h = 140, 70
    sims, u, _ = _pair(w, h, storage, "free_slip", 0.0, 40, 11)
    sims[1].set_timing(False)
    for sim in sims:
        sim.jacobi_tile = (3, 4, 8, 2)
    sims[0].use_graph = True
    for step in range(7):
        for sim in sims:
            if step % 3 == 2:
                sim.add_splats([(0.4, 0.5, 0.7, -0.3, 4.0, 0.0)])
            sim.update(1 / 60)
        for f in ("velocity", "pressure", "mask"):
            a, b = (sim.download(f) for sim in sims)
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), (step, f)
    for sim in sims:
        sim.destroy()


def test_splats_far_and_near_a_zero_weight(gpu):
    """Weights around the last one that does not round to zero (10.2 radii)."""
    w, h = 400, 24
    rng = np.random.default_rng(5)
    u = rng.standard_normal((h, w, 2)).astype(np.float32)
    u[::3] = -0.0
    sim = FluidSimulator(w, h)
    splats = [(0.02, 0.5, 1e30, -1e30, 7.0, 0.0), (0.9, 0.3, -2.0, 1e38, 11.5, 0.0),
              (-4.0, 0.5, 1.0, 1.0, 3.0, 0.0)]
    sim.upload("velocity", u)
    sim.add_splats(splats)
    ref, _ = F.gaussian_splat(u, None, [tuple(np.float32(v) for v in s) for s in splats])
    assert np.array_equal(sim.download("velocity").view(np.uint32), ref.view(np.uint32))
    sim.destroy()


@pytest.mark.parametrize("storage", ["bf16", "f16"])
@pytest.mark.parametrize("iters,corr", [(1, 8), (1, 0), (2, 0), (2, 16), (13, 3)])
def test_merged_reduced_storage_is_the_replay(gpu, storage, iters, corr):
    """One iteration leaves the correction launch alone, which also projects;
    no correction sweeps, and the most."""
    w, h = 150, 90
    sims, u, solid = _pair(w, h, storage, "inflow", 0.0, iters, 21)
    u = M.rounder(storage)(u)
    prm = F.Params(vorticity=0.3, viscosity=0.0, iterations=iters, bc_mode=F.BC_INFLOW)
    v, p, p32, b, _ = M.step_mixed(u, np.zeros((h, w, 2), np.float32), np.float32(1 / 60), prm,
                                   storage, 6, corr, persistent=solid)
    for sim in sims:
        sim.jacobi_tile = (6, 8, 8, 2)
        sim.correction_sweeps = corr
        sim.upload("velocity", u)
        sim.update(1 / 60)
        assert np.array_equal(sim.download("velocity"), v)
        assert np.array_equal(sim.download("pressure32"), p32)
        assert np.array_equal(sim.download("divergence"), b)
        sim.destroy()


@pytest.mark.parametrize("radius", [3.0, 6.0, 9.0, 40.0])
def test_splats_whose_reach_covers_little_or_all(gpu, radius):
    """Both forms of the weight, in a grid and in a batch: a reach of 10.25 radii is
    a fifth of 160 x 120 cells, about half, most, and all of them."""
    from natrix_amd.batch import BatchedScenes
    w, h = 160, 120
    rng = np.random.default_rng(6)
    u = rng.standard_normal((h, w, 2)).astype(np.float32)
    splats = [(0.3, 0.4, 0.5, -0.25, radius, 1.0), (0.6, 0.7, -1.5, 2.0, 1.3 * radius, 0.5)]
    s32 = [tuple(np.float32(v) for v in s) for s in splats]
    ref, q = F.gaussian_splat(u, np.zeros((h, w), np.float32), s32)
    sim = FluidSimulator(w, h, dye=True)
    sim.upload("velocity", u)
    sim.add_splats(splats)
    assert np.array_equal(sim.download("velocity").view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(sim.download("dye").view(np.uint32), q.view(np.uint32))
    sim.destroy()
    half = M.rounder("bf16")
    sim = FluidSimulator(w, h, storage="bf16")
    sim.upload("velocity", half(u))
    sim.add_splats(splats)
    assert np.array_equal(sim.download("velocity"), half(F.gaussian_splat(half(u), None, s32)[0]))
    sim.destroy()
    b, one = BatchedScenes([w, 50], [h, 40]), FluidSimulator(w, h)
    b.upload(0, "velocity", u)
    one.upload("velocity", u)
    b.set_step_splats([(0,) + s for s in splats])
    one.add_splats(splats)
    b.update(1 / 60)
    one.update(1 / 60)
    assert np.array_equal(b.download(0, "velocity"), one.download("velocity"))
    b.destroy()
    one.destroy()
