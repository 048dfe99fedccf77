"""Steps replayed from HIP graphs, single grids and batches, against the same
steps enqueued: bitwise, every replay, with other work and waits between them.
Tiles of a few sweeps give every step the ten launches from which it is
replayed, and graph_replays says that it was."""
import numpy as np
import pytest
from test_gpu_batch import SIZES, _batch, _setup

from natrix_amd import FluidSimulator

pytestmark = pytest.mark.gpu


def _same(a, b, *what):
    assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), what


@pytest.mark.parametrize("storage,fields", [
    ("f32", ("velocity", "pressure", "dye", "mask")),
    ("bf16", ("velocity", "pressure", "pressure32", "dye", "mask"))])
@pytest.mark.parametrize("iters", [40, 41])
def test_dye_and_forcing(gpu, storage, fields, iters):
    """The dye's parity is part of the graph's key; 41 iterations leave an even,
    40 an odd number of launches and so the other pressure buffer."""
    w, h = 150, 90
    rng = np.random.default_rng(9)
    u = rng.uniform(-0.5, 0.5, (h, w, 2)).astype(np.float32)
    solid = rng.random((h, w)) < 0.05
    sims = []
    for graph in (False, True):
        sim = FluidSimulator(w, h, dye=True, bc_mode="free_slip", storage=storage)
        sim.vorticity, sim.viscosity, sim.iterations = 0.3, 0.0, iters
        sim.jacobi_tile = (3, 4, 8, 2)
        sim.set_obstacle_map(solid)
        sim.upload("velocity", u)
        sim.use_graph = graph
        sims.append(sim)
    for step in range(10):
        for sim in sims:
            sim.add_splats([(0.3, 0.5, 1.0, 0.5, 3.0, 1.0)])
            if step % 4 == 1:
                sim.add_circle_obstacle((0.6, 0.4), 7.0)
            sim.update(1 / 60)
        for f in fields:
            _same(*(sim.download(f) for sim in sims), step, f)
    assert [sim.graph_replays for sim in sims] == [0, 10]
    # another dt is another graph; a timed step is not replayed
    for sim in sims:
        sim.update(1 / 50)
        sim.set_timing(True)
        sim.update(1 / 50)
    _same(*(sim.download("velocity") for sim in sims), "dt")
    assert [sim.graph_replays for sim in sims] == [0, 11]
    for sim in sims:
        sim.destroy()


def test_short_steps_are_enqueued(gpu):
    sim = FluidSimulator(64, 64)
    sim.use_graph = True
    sim.iterations = 20
    sim.update(1 / 60)
    assert sim.graph_replays == 0
    sim.destroy()


def test_single_grid_2048(gpu):
    n, steps = 2048, 20
    y, x = np.mgrid[0:n, 0:n]
    solid = (x - 0.4 * n) ** 2 + (y - 0.5 * n) ** 2 <= (0.1 * n) ** 2
    out = []
    for graph in (False, True):
        sim = FluidSimulator(n, n, bc_mode="inflow")
        sim.vorticity, sim.viscosity, sim.iterations = 0.3, 0.0, 80
        sim.set_obstacle_map(solid)
        if graph:
            sim.jacobi_tile = (8, 8, 8, 2)
            sim.use_graph = True
        for _ in range(steps):
            sim.update(1 / 60)
        assert sim.graph_replays == (steps if graph else 0)
        out.append((sim.download("velocity"), sim.download("pressure")))
        sim.destroy()
    for a, b in zip(*out):
        _same(a, b)


@pytest.mark.parametrize("iters", [34, 35, 36])
def test_batch(gpu, iters):
    """Uneven scenes with dye, obstacles and per-step splats, which change on the
    way (the graphs are made anew); whole and uneven last launches."""
    scenes = _setup(3)
    a = _batch(scenes, iters, tile=(3, 8, 8, 1))
    g = _batch(scenes, iters, tile=(3, 8, 8, 1), graph=True)
    for step in range(8):
        for b in (a, g):
            if step == 5:
                b.set_step_splats([(0, 0.5, 0.5, 0.4, -0.2, 4.0, 1.0)])
            if step % 3 == 2:
                b.add_circle_obstacle(1, (0.4, 0.6), 5.0)
            b.update(1 / 60)
        for i in range(len(SIZES)):
            for f in ("velocity", "pressure", "dye", "mask"):
                _same(g.download(i, f), a.download(i, f), step, i, f)
    assert (a.graph_replays, g.graph_replays) == (0, 8)
    a.destroy()
    g.destroy()


@pytest.mark.parametrize("sides,tiles", [((512, 512, 512), 768), ((512, 512, 512, 40), 771)])
@pytest.mark.parametrize("graph", [False, True])
def test_batch_on_either_side_of_the_advecting_form(gpu, sides, tiles, graph):
    """The last batch whose stages advect and the first whose do not, which leaves
    the velocity in the other buffer: against the timed batch's separate launches."""
    assert sum(-(-s // 64) * -(-s // 16) for s in sides) == tiles
    rng = np.random.default_rng(5)
    from natrix_amd.batch import BatchedScenes
    bs = [BatchedScenes(sides, dye=True) for _ in range(2)]
    for i, s in enumerate(sides):
        u = rng.uniform(-0.5, 0.5, (s, s, 2)).astype(np.float32)
        solid = rng.random((s, s)) < 0.03
        for b in bs:
            b.upload(i, "velocity", u)
            b.set_obstacle_map(i, solid)
    for b in bs:
        b.set_params(iterations=40, vorticity=0.3, viscosity=0.0, jacobi_tile=(4, 8, 8, 1))
    bs[0].use_graph = graph
    bs[1].set_timing(True)
    for step in range(5):
        for b in bs:
            b.update(1 / 60)
        for i in range(len(sides)):
            for f in ("velocity", "pressure", "dye"):
                _same(*(b.download(i, f) for b in bs), step, i, f)
    assert bs[0].graph_replays == (5 if graph else 0)
    for b in bs:
        b.destroy()


def test_benchmark_batch(gpu):
    import bench
    got = []
    for graph in (False, True):
        b, sides, _, _ = bench.make_batch()
        b.set_params(jacobi_tile=(6, 8, 8, 2))
        b.use_graph = graph
        for _ in range(4):
            b.update(1 / 60)
        assert b.graph_replays == (4 if graph else 0)
        got.append([b.download(i, f) for i in (0, 17, 40, 63) for f in ("velocity", "dye")])
        b.destroy()
    for x, y in zip(*got):
        _same(x, y)
