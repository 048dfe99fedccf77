"""The Chebyshev tiles where they can go wrong: grids of exactly one tile, one
cell more and less, lower or narrower than a tile, launches of one pass to the
most, with and without solid cells; bitwise against the float32 statement."""
import ctypes as C

import numpy as np
import pytest
import torch
from smoothers import cheb32, lap
from test_gpu_learned import dev, in_step_sim

from natrix_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solids", [True, False])
@pytest.mark.parametrize("W,H,tile,iters", [
    (128, 128, (20, 8, 8, 2), 18), (129, 127, (20, 8, 8, 2), 19), (127, 129, (9, 8, 8, 2), 20),
    (300, 40, (20, 8, 8, 2), 40), (17, 300, (12, 8, 8, 2), 25), (261, 263, (16, 4, 16, 2), 34),
    (128, 64, (2, 4, 16, 2), 3), (140, 70, (8, 8, 8, 1), 16), (131, 133, (7, 4, 8, 2), 6),
])
def test_tiles(gpu, rng, W, H, tile, iters, solids):
    sim = in_step_sim(rng, H, W)
    solid = sim.download("mask") != 0
    if not solids:
        dev(sim, "mask").zero_()
        solid[:] = False
    b = rng.normal(size=(H, W)).astype(np.float32)
    p = rng.normal(size=(H, W)).astype(np.float32)
    dev(sim, "divergence").copy_(torch.from_numpy(b))
    dev(sim, "pressure").copy_(torch.from_numpy(p))
    torch.cuda.synchronize()
    out = (C.c_double * 2)()
    _lib.call("nx_smooth_chebyshev", sim._alive(), iters, 0.01, (C.c_int * 4)(*tile), out)
    got = sim.download("pressure")
    assert np.array_equal(got, cheb32(p, b, solid, iters, 0.01))
    assert np.isfinite(out[0])
    _lib.call("nx_step_finish", sim._alive())
    sim.destroy()


@pytest.mark.parametrize("W,H,iters", [(140, 70, 5), (64, 33, 1), (17, 300, 4)])
@pytest.mark.parametrize("tile", [(1, 8, 8, 2, 0), (1, 4, 16, 1, 0), (1, 4, 8, 2, 24)])
def test_one_pass_a_launch(gpu, rng, W, H, iters, tile):
    """k = 1, tile and streaming: the first launch only sets up, each of the next
    runs one iteration, the last only takes the residual."""
    sim = in_step_sim(rng, H, W)
    solid = sim.download("mask") != 0
    b = rng.normal(size=(H, W)).astype(np.float32)
    p = rng.normal(size=(H, W)).astype(np.float32)
    dev(sim, "divergence").copy_(torch.from_numpy(b))
    dev(sim, "pressure").copy_(torch.from_numpy(p))
    torch.cuda.synchronize()
    sim.smoother_tile = tile if tile[4] else tile[:4]
    sim.set_timing(True)
    sim.collect_timing()
    out = (C.c_double * 2)()
    _lib.call("nx_smooth_chebyshev", sim._alive(), iters, 0.01, None, out)
    assert sim.collect_timing()["chebyshev"][1] == iters + 2
    got = sim.download("pressure")
    assert np.array_equal(got, cheb32(p, b, solid, iters, 0.01))
    _check_residual(out[0], got, b, solid)
    _lib.call("nx_step_finish", sim._alive())
    sim.destroy()


@pytest.mark.parametrize("W,H,tile,iters", [
    (129, 127, (20, 8, 8, 2), 19), (300, 40, (20, 8, 8, 2), 40), (261, 263, (16, 4, 16, 2), 34),
    (128, 64, (2, 4, 16, 2), 3), (140, 70, (8, 8, 8, 1), 16), (131, 133, (7, 4, 8, 2), 6),
    (200, 150, (3, 8, 16, 1), 1)])
def test_residual_of_several_tiles(gpu, rng, W, H, tile, iters):
    """The last launch's residual, whose tiles shrink by one stencil less than
    their passes: every fluid cell in one record."""
    sim = in_step_sim(rng, H, W)
    solid = sim.download("mask") != 0
    b = rng.normal(size=(H, W)).astype(np.float32)
    dev(sim, "divergence").copy_(torch.from_numpy(b))
    torch.cuda.synchronize()
    out = (C.c_double * 2)()
    _lib.call("nx_smooth_chebyshev", sim._alive(), iters, 0.01, (C.c_int * 4)(*tile), out)
    _check_residual(out[0], sim.download("pressure"), b, solid)
    _lib.call("nx_step_finish", sim._alive())
    sim.destroy()


def _check_residual(rel, p, b, solid):
    r = (b.astype(np.float64) - lap(p.astype(np.float64), solid))[~solid]
    bf = b.astype(np.float64)[~solid]
    n = r.size
    want = np.sqrt((np.sum(r * r) - np.sum(r) ** 2 / n) / (np.sum(bf * bf) - np.sum(bf) ** 2 / n))
    assert abs(rel - want) <= 1e-9 * want


@pytest.mark.parametrize("partial", [True, False])
@pytest.mark.parametrize("Wc,Hc,iters", [(128, 128, 5), (100, 72, 40), (7, 60, 12)])
def test_face_weights_outside_the_unit_interval_are_open(gpu, rng, Wc, Hc, iters, partial):
    """Whether or not the wave holds partial faces, whose form of the sweep
    multiplies by the weight."""
    sim = in_step_sim(rng, 64, 64)
    kinds = [0.0, 0.25, 0.75, 1.0] if partial else [0.0, 1.0, 1.0]
    plain = rng.choice(kinds, size=(2, Hc, Wc)).astype(np.float32)
    odd = plain.copy()
    at = rng.random(plain.shape) < 0.2
    odd[at] = rng.choice([1.5, -0.5, np.nan, np.inf], size=int(at.sum()))
    plain[at] = 1.0
    e0, rc = (rng.normal(size=(Hc, Wc)).astype(np.float32) for _ in range(2))
    mc = torch.zeros((Hc, Wc), dtype=torch.uint8, device="cuda")
    got = []
    for faces in (plain, odd):
        e, r, f = (torch.from_numpy(a).cuda() for a in (e0, rc, faces))
        torch.cuda.synchronize()
        _lib.call("nx_coarse_smooth_faces", sim._alive(), Wc, Hc,
                  *(C.c_void_p(t.data_ptr()) for t in (e, r, mc, f)), iters, 0.05)
        sim.synchronize()
        got.append(e.cpu().numpy())
    assert np.isfinite(got[0]).all()
    assert np.array_equal(got[0], got[1])
    _lib.call("nx_step_finish", sim._alive())
    sim.destroy()
