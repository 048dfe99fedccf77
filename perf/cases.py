"""Performance cases of the framework, through its public entry points.

Each case is one call, or the few calls of one frame, that a program using
the framework makes: fluid steps at a fixed number of pressure sweeps (every
storage format, eager and as a replayed graph), the demo's frame with its
display passes, a tolerance-driven step, learned steps, rollouts of batched
scenes and the layers and the training step of the pressure network.

``listed()`` names the fixed cases, ``draw(rng)`` gives further ones of the
same ranges, ``prepare`` makes the inputs and objects a program holds before
the call, ``run`` makes the call and returns its results, ``work`` states the
bytes and operations it cannot do without, and ``exact`` evaluates the same
mathematics in float64 with plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

DT = 1.0 / 60.0
SPEED = 500.0
STORAGE = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
BYTES = {"f32": 4, "bf16": 2, "f16": 2}


# ------------------------------------------------------------------ the cases
def _step(name=None, **kw):
    c = {"kind": "step", "width": 512, "height": 512, "iterations": 50, "storage": "f32",
         "walls": "reference", "vorticity": 0.0, "viscosity": 0.1, "dye": False, "splats": 0,
         "drag": False, "solid": "none", "graph": False}
    c.update(kw)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the reference's own defaults on a small grid with one mouse drag per
        # frame: the smallest call, where launches and latency count
        _step("drag_128", width=128, height=128, drag=True),
        # the CPU configuration of the benchmark: box, three splats a step,
        # dye, replayed as a graph
        _step("splats_256_graph", width=256, height=256, iterations=40, walls="free_slip",
              vorticity=0.3, viscosity=0.0, dye=True, splats=3, graph=True),
        # odd sides, half precision storage, walls with inflow, rectangles
        _step("f16_1001x699", width=1001, height=699, iterations=60, storage="f16",
              walls="inflow", vorticity=0.3, dye=True, splats=2, solid="rectangles"),
        # the benchmark's plain step: cylinder in an inflow, 80 sweeps
        _step("cylinder_2048", width=2048, height=2048, iterations=80, walls="inflow",
              vorticity=0.3, viscosity=0.0, solid="cylinder"),
        # the benchmark's largest grid, bfloat16 storage
        _step("bf16_4096", width=4096, height=4096, iterations=120, storage="bf16",
              walls="free_slip", vorticity=0.3, viscosity=0.0, dye=True, splats=8),
        # one frame of the demo: velocity on half the window, dye on the
        # window, drag, both advections and the two display passes
        {"name": "demo_frame_1280x720", "kind": "frame", "width": 1280, "height": 720,
         "iterations": 50, "arrows": 32.0},
        # plain Jacobi to a tolerance on a small grid: thousands of sweeps
        {"name": "tolerance_128x96", "kind": "tolerance", "width": 128, "height": 96,
         "tol": 1e-3, "solid": "none"},
        # the benchmark's learned step: three levels, cylinder in an inflow
        {"name": "learned_2048", "kind": "learned", "width": 2048, "height": 2048, "mid": 4,
         "smooth": 18, "solid": "cylinder"},
        # the learned step as set_guess() runs it, on a grid whose coarse
        # grid is padded
        {"name": "learned_1000x700", "kind": "learned", "width": 1000, "height": 700, "mid": 0,
         "smooth": 72, "solid": "none"},
        # a data set's rollout: twenty scenes of uneven sizes advanced by four
        # steps, then read back
        {"name": "rollout_20", "kind": "batch", "scenes": 20, "smallest": 64, "largest": 512,
         "steps": 4, "iterations": 60, "graph": False},
        # one convolution layer of the network, forward and backward, at the
        # trainer's batch
        {"name": "conv_32x64x64_64", "kind": "conv", "batch": 32, "height": 64, "width": 64,
         "cin": 64, "cout": 64},
        # the trainer's step: the whole network at batch 32, gradients of
        # every parameter
        {"name": "unet_32x128x128", "kind": "unet", "batch": 32, "height": 128, "width": 128},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("step", "step", "step", "frame", "tolerance", "learned", "batch", "conv",
                       "unet"))
    if kind == "step":
        storage = rng.choice(("f32", "f32", "bf16", "f16"))
        w, h = _log_int(rng, 96, 4096), _log_int(rng, 96, 4096)
        if storage == "f32" and w * h > (1 << 23):
            h = max(96, (1 << 23) // w)
        drag = storage == "f32" and rng.random() < 0.5
        return _step(width=w, height=h, storage=storage, iterations=rng.randint(20, 120),
                     walls=rng.choice(("reference", "free_slip", "inflow")),
                     vorticity=rng.choice((0.0, 0.3)), viscosity=rng.choice((0.0, 0.1)),
                     dye=rng.random() < 0.5, splats=0 if drag else rng.randint(0, 5), drag=drag,
                     solid=rng.choice(("none", "cylinder", "rectangles")),
                     graph=rng.random() < 0.3)
    if kind == "frame":
        w, h = _log_int(rng, 320, 2560), _log_int(rng, 240, 1440)
        return {"kind": kind, "width": w, "height": h, "iterations": rng.randint(20, 80),
                "arrows": rng.choice((16.0, 32.0, 25.0))}
    if kind == "tolerance":
        return {"kind": kind, "width": rng.randint(48, 128), "height": rng.randint(48, 96),
                "tol": 1e-3, "solid": rng.choice(("none", "cylinder"))}
    if kind == "learned":
        if rng.random() < 0.5:
            f = rng.choice((8, 12, 16))
            w, h = 128 * f - rng.randint(0, 64), 128 * f - rng.randint(0, 64)
            return {"kind": kind, "width": w, "height": h, "mid": 4, "smooth": 18,
                    "solid": "cylinder"}
        return {"kind": kind, "width": _log_int(rng, 256, 2048),
                "height": _log_int(rng, 256, 2048), "mid": 0, "smooth": 72,
                "solid": rng.choice(("none", "cylinder"))}
    if kind == "batch":
        lo = _log_int(rng, 32, 128)
        return {"kind": kind, "scenes": rng.randint(4, 20), "smallest": lo,
                "largest": _log_int(rng, lo, 512), "steps": rng.randint(1, 4),
                "iterations": rng.randint(20, 60), "graph": rng.random() < 0.5}
    if kind == "conv":
        level = rng.randint(0, 3)  # the network's levels: side and channels go together
        n = _log_int(rng, 1, 32)
        side = 128 >> level
        cin, cout = rng.choice((((32, 32), (96, 32)), ((32, 64), (64, 64), (192, 64)),
                                ((64, 128), (128, 128), (384, 128)),
                                ((128, 256), (256, 256)))[level])
        return {"kind": kind, "batch": n, "height": side - rng.randint(0, side // 4),
                "width": side - rng.randint(0, side // 4), "cin": cin, "cout": cout}
    return {"kind": kind, "batch": _log_int(rng, 1, 32), "height": 8 * rng.randint(4, 16),
            "width": 8 * rng.randint(4, 16)}


# ------------------------------------------------------------------ the inputs
def _flow(gen, w, h):
    """A smooth random velocity (h, w, 2) in float32: a few dozen Fourier modes, mostly
    solenoidal as a developed flow is, |v| mostly below 0.6."""
    x = (torch.arange(w, device="cuda", dtype=torch.float32) / w)[None, :]
    y = (torch.arange(h, device="cuda", dtype=torch.float32) / h)[:, None]
    v = torch.zeros((h, w, 2), device="cuda")
    modes = 12
    k = torch.randint(1, 9, (modes, 2), generator=gen).tolist()
    ph = (2 * math.pi * torch.rand((modes, 3), generator=gen)).tolist()
    amp = torch.rand((modes, 2), generator=gen).tolist()
    for i in range(modes):
        kx, ky = math.pi * k[i][0], math.pi * k[i][1]
        n = math.hypot(kx, ky)
        a, d = 0.12 + 0.12 * amp[i][0], 0.05 * amp[i][1]
        ax, ay = kx * x + ph[i][0], ky * y + ph[i][1]
        sx, cx, sy, cy = ax.sin(), ax.cos(), ay.sin(), ay.cos()
        v[..., 0] += (a * ky * sx * cy + d * kx * cx * sy) / n
        v[..., 1] += (d * ky * sx * cy - a * kx * cx * sy) / n
    return v


def _solid(kind, gen, w, h):
    """Obstacle map (h, w) as uint8, or None."""
    if kind == "none":
        return None
    r = torch.rand(64, generator=gen).tolist()
    y, x = np.arange(h)[:, None], np.arange(w)[None, :]
    if kind == "cylinder":
        cx, cy = (0.3 + 0.4 * r[0]) * w, (0.3 + 0.4 * r[1]) * h
        return ((x - cx) ** 2 + (y - cy) ** 2 <= (0.1 * min(w, h)) ** 2).astype(np.uint8)
    m = np.zeros((h, w), np.uint8)
    for i in range(5):
        rw, rh = int((0.05 + 0.1 * r[4 * i]) * w), int((0.05 + 0.1 * r[4 * i + 1]) * h)
        x0 = int((0.1 + 0.7 * r[4 * i + 2]) * w)
        y0 = int((0.1 + 0.7 * r[4 * i + 3]) * h)
        m[y0:y0 + rh, x0:x0 + rw] = 1
    return m


def _splats(gen, n, radius):
    """Gaussian splats (px, py, ax, ay, radius, dye) as the benchmark's scenes draw them."""
    out = []
    for _ in range(n):
        r = torch.rand(4, generator=gen).tolist()
        f, a = (50 + 150 * r[0]) * DT, 2 * math.pi * r[1]
        out.append((0.1 + 0.8 * r[2], 0.1 + 0.8 * r[3], f * math.cos(a), f * math.sin(a),
                    radius, 1.0))
    return out


def _dye_field(w, h):
    y = torch.arange(h, device="cuda")[:, None] * (9.0 / h)
    x = torch.arange(w, device="cuda")[None, :] * (7.0 / w)
    return 0.5 + 0.5 * torch.sin(x + 1.0) * torch.cos(y)


def _drag(gen):
    r = torch.rand(4, generator=gen).tolist()
    return ((0.2 + 0.6 * r[0], 0.2 + 0.6 * r[1]), (1.6 * r[2] - 0.8, 1.6 * r[3] - 0.8))


def _fluid_inputs(case, seed):
    """Everything a fluid case starts from, from the seed alone."""
    gen = torch.Generator().manual_seed(seed)
    w, h = case["width"], case["height"]
    vw, vh = (w // 2, h // 2) if case["kind"] == "frame" else (w, h)
    dtype = STORAGE[case.get("storage", "f32")]
    flow = _flow(gen, vw, vh).to(dtype)
    dye = None
    if case.get("dye") or case["kind"] == "frame":
        dye = _dye_field(w, h).to(dtype)
    return {"flow": flow, "dye": dye, "solid": _solid(case.get("solid", "none"), gen, vw, vh),
            "splats": _splats(gen, case.get("splats", 0), max(2.0, 0.02 * min(vw, vh))),
            "drag": _drag(gen)}


def _network_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n, h, w = case["batch"], case["height"], case["width"]

    def rand(*shape):
        return torch.randn(shape, generator=gen, device="cuda")
    if case["kind"] == "conv":
        # activations come out of a ReLU, gradients are small
        return {"x": rand(n, h, w, case["cin"]).relu_().to(torch.bfloat16),
                "w": rand(case["cout"], 9, case["cin"]) * math.sqrt(2.0 / (9 * case["cin"])),
                "b": 0.1 * rand(case["cout"]),
                "dy": (0.01 * rand(n, h, w, case["cout"])).to(torch.bfloat16)}
    solid = torch.zeros((n, h, w), dtype=torch.bool, device="cuda")
    solid[:, h // 3:h // 2, w // 3:w // 2] = True
    return {"rhs": rand(n, h, w), "solid": solid, "target": rand(n, h, w)}


def _batch_sizes(case):
    n, lo, hi = case["scenes"], case["smallest"], case["largest"]
    side = [int(round(lo * (hi / lo) ** (i / (n - 1)))) for i in range(n)]
    return [(s, side[(7 * i + 3) % n] // 2 + s // 2) for i, s in enumerate(side)]


def _batch_inputs(case, seed):
    gen = torch.Generator().manual_seed(seed)
    scenes = []
    for w, h in _batch_sizes(case):
        scenes.append({"flow": _flow(gen, w, h), "solid": _solid("rectangles", gen, w, h),
                       "dye": _dye_field(w, h), "splats": _splats(gen, 2, 0.06 * min(w, h))})
    return scenes


# ------------------------------------------------------------------ prepare, run
_TORCH_VIEW = {"f32": None, "bf16": torch.bfloat16, "f16": None}


class _Fields:
    """Zero-copy tensors over a simulator's fields; a field's two buffers are wrapped once."""

    def __init__(self, sim):
        self.sim, self.views = sim, {}

    def __getitem__(self, name):
        buf = self.sim.field_buffer(name)
        v = self.views.get(buf.ptr)
        if v is None:
            v = torch.as_tensor(buf, device="cuda")
            as_type = _TORCH_VIEW[self.sim.storage] if v.dtype == torch.uint16 else None
            v = self.views[buf.ptr] = v if as_type is None else v.view(as_type)
        return v


def _prepare_fluid(case, seed):
    from natrix_amd import FluidSimulator
    inp = _fluid_inputs(case, seed)
    kind = case["kind"]
    vw, vh = inp["flow"].shape[1], inp["flow"].shape[0]
    sim = FluidSimulator(vw, vh, storage=case.get("storage", "f32"),
                         dye=bool(case.get("dye", False)))
    s = {"case": case, "sim": sim, "fields": _Fields(sim), "inputs": inp}
    if kind == "step":
        sim.iterations, sim.vorticity = case["iterations"], case["vorticity"]
        sim.viscosity, sim.bc_mode = case["viscosity"], case["walls"]
        if case["graph"]:
            sim.use_graph = True
    elif kind == "frame":
        from natrix_amd.core.particles_area import SmoothParticlesArea
        sim.iterations = case["iterations"]
        s["area"] = SmoothParticlesArea(case["width"], case["height"], sim)
    else:
        sim.vorticity, sim.viscosity, sim.bc_mode = 0.3, 0.0, "inflow"
        if kind == "tolerance":
            sim.tol = case["tol"]
        else:
            from natrix_amd.learned.solver import LearnedGuess
            from natrix_amd.learned.train import load
            net, meta = load()
            s["guess"] = LearnedGuess(net, coarse=meta.get("size", 128), mid=case["mid"])
            if not case["mid"]:
                sim.set_guess(s["guess"])
        s["stream"] = torch.cuda.ExternalStream(sim.stream_handle())
    if inp["solid"] is not None:
        sim.set_obstacle_map(inp["solid"])
    sim.synchronize()
    s["fields"]["velocity"].copy_(inp["flow"])
    if inp["dye"] is not None:
        s["fields"]["dye"].copy_(inp["dye"])
    torch.cuda.synchronize()
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("step", "frame", "tolerance", "learned"):
        return _prepare_fluid(case, seed)
    if kind == "batch":
        from natrix_amd.batch import BatchedScenes
        sizes, scenes = _batch_sizes(case), _batch_inputs(case, seed)
        b = BatchedScenes([w for w, _ in sizes], [h for _, h in sizes], dye=True)
        b.set_params(iterations=case["iterations"], vorticity=0.3, viscosity=0.0,
                     bc_mode="free_slip")
        for i, sc in enumerate(scenes):
            b.set_obstacle_map(i, sc["solid"])
            b.upload(i, "velocity", sc["flow"].cpu().numpy())
            b.upload(i, "dye", sc["dye"].cpu().numpy())
        b.set_step_splats([(i,) + sp for i, sc in enumerate(scenes) for sp in sc["splats"]])
        b.use_graph = case["graph"]
        b.synchronize()
        return {"case": case, "batch": b}
    from natrix_amd.learned.unet import Conv, UNet, pack_input
    inp = _network_inputs(case, seed)
    if kind == "conv":
        layer = Conv(case["cin"], case["cout"]).cuda()
        with torch.no_grad():
            layer.w.copy_(inp["w"])
            layer.b.copy_(inp["b"])
        return {"case": case, "layer": layer, "x": inp["x"].requires_grad_(True),
                "dy": inp["dy"]}
    net = UNet()
    with torch.no_grad():
        for p, q in zip(net.parameters(), _unet_parameters(seed)):
            p.copy_(q)
    return {"case": case, "net": net.cuda(), "x": pack_input(inp["rhs"], inp["solid"]),
            "target": inp["target"], "fluid": ~inp["solid"]}


def _run_fluid(s):
    case, sim, f, inp = s["case"], s["sim"], s["fields"], s["inputs"]
    if case["kind"] == "step":
        if case["drag"]:
            pos, vel = inp["drag"]
            sim.add_velocity(pos, vel, 0.08 * case["width"])
        if inp["splats"]:
            sim.add_splats(inp["splats"] if case["dye"] else
                           [sp[:5] + (0.0,) for sp in inp["splats"]])
        sim.update(DT)
        out = {"velocity": f["velocity"], "pressure": f["pressure"]}
        if case["dye"]:
            out["dye"] = f["dye"]
        return out
    if case["kind"] == "frame":
        pos, vel = inp["drag"]
        sim.add_velocity(pos, vel, 32.0)
        s["area"].add_particles(pos, 40.0, 0.5)
        sim.update(DT)
        s["area"].update(DT)
        return {"image": sim.dye_rgba8(device=True),
                "arrows": sim.quiver_rgba8(case["width"], case["height"], case["arrows"],
                                           device=True),
                "velocity": f["velocity"], "dye": f["dye"]}
    # a step from a given flow, as each member of an ensemble or each sample of
    # a data set takes it
    with torch.cuda.stream(s["stream"]):
        f["velocity"].copy_(inp["flow"])
    if case["kind"] == "learned" and case["mid"]:
        from natrix_amd.learned.solver import solve_step
        solve_step(sim, s["guess"], DT, tol=1e-4, smooth=case["smooth"])
    else:
        sim.update(DT)
    return {"velocity": f["velocity"], "pressure": f["pressure"]}


def run(s):
    kind = s["case"]["kind"]
    if kind in ("step", "frame", "tolerance", "learned"):
        return _run_fluid(s)
    if kind == "batch":
        b = s["batch"]
        for _ in range(s["case"]["steps"]):
            b.update(DT)
        return [[b.download(i, f) for f in ("velocity", "pressure", "dye")]
                for i in range(len(b))]
    if kind == "conv":
        layer, x = s["layer"], s["x"]
        y = layer(x)
        dx, dw, db = torch.autograd.grad(y, (x, layer.w, layer.b), s["dy"])
        return {"y": y.detach(), "dx": dx, "dw": dw, "db": db}
    from natrix_amd.learned.train import masked_loss
    net = s["net"]
    out = net(s["x"])
    grads = torch.autograd.grad(masked_loss(out, s["target"], s["fluid"]), list(net.parameters()))
    return {"out": out.detach(), "grads": list(grads)}


# ------------------------------------------------------------------ work
_CHANNELS = ((8, 32, 0), (32, 32, 0), (32, 64, 1), (64, 64, 1), (64, 128, 2), (128, 128, 2),
             (128, 256, 3), (256, 256, 3), (384, 128, 2), (128, 128, 2), (192, 64, 1),
             (64, 64, 1), (96, 32, 0), (32, 32, 0))


def work(case):
    """Inputs read once and outputs written once; operations of the stencils (5 a cell and
    pressure sweep, about 100 a cell for the other stages), of the sweeps a solve to a
    tolerance needs at least, and of the convolutions."""
    kind = case["kind"]
    if kind == "batch":
        cells = sum(w * h for w, h in _batch_sizes(case))
        return {"bytes": cells * (8 + 4 + 1 + 8 + 4 + 4),
                "flops": cells * case["steps"] * (5 * case["iterations"] + 100)}
    if kind in ("step", "frame", "tolerance", "learned"):
        cells = case["width"] * case["height"]
        if kind == "step":
            e = BYTES[case["storage"]]
            per = 2 * e + 1 + 2 * e + e + (2 * e if case["dye"] else 0)
            return {"bytes": cells * per, "flops": cells * (5 * case["iterations"] + 100)}
        if kind == "frame":  # velocity on a quarter of the cells; two images
            return {"bytes": cells // 4 * 17 + cells * (8 + 8),
                    "flops": cells // 4 * (5 * case["iterations"] + 100) + cells * 100}
        if kind == "tolerance":
            return {"bytes": cells * 21, "flops": cells * 5 * max(case["width"], case["height"])}
        # three refinements of a cycle with 18 smoothing iterations and one network pass
        return {"bytes": cells * 21, "flops": 3 * (cells * 18 * 9 + 5.4e9)}
    n, h, w = case["batch"], case["height"], case["width"]
    if kind == "conv":
        px, ci, co = n * h * w, case["cin"], case["cout"]
        return {"bytes": 2 * px * (2 * ci + 2 * co) + 2 * 4 * 9 * ci * co,
                "flops": 3 * 2 * 9 * px * ci * co}
    px = n * h * w
    macs = sum(9 * ci * co * px // 4 ** lv for ci, co, lv in _CHANNELS)
    first = 9 * 8 * 32 * px  # the first layer needs no gradient of its input
    params = sum(9 * ci * co for ci, co, _ in _CHANNELS)
    return {"bytes": px * (16 + 4 + 4 + 1) + 8 * params, "flops": 6 * macs - 2 * first}


# ------------------------------------------------------------------ float64
def _neighbours(a):
    """Left, right, below and above of each cell, the cell itself beyond an edge."""
    left = torch.cat((a[:, :1], a[:, :-1]), 1)
    right = torch.cat((a[:, 1:], a[:, -1:]), 1)
    below = torch.cat((a[:1], a[:-1]), 0)
    above = torch.cat((a[1:], a[-1:]), 0)
    return left, right, below, above


def _sample(f, px, py):
    """Bilinear values of f at clamped corners around (px, py)."""
    h, w = f.shape[:2]
    x0, x1 = px.floor().clamp(0, w - 1), px.ceil().clamp(0, w - 1)
    y0, y1 = py.floor().clamp(0, h - 1), py.ceil().clamp(0, h - 1)
    tx, ty = px - x0, py - y0
    if f.ndim == 3:
        tx, ty = tx[..., None], ty[..., None]
    x0, x1, y0, y1 = (t.long() for t in (x0, x1, y0, y1))
    low = f[y0, x0] * (1 - tx) + f[y0, x1] * tx
    high = f[y1, x0] * (1 - tx) + f[y1, x1] * tx
    return low * (1 - ty) + high * ty


def _grid(h, w):
    return (torch.arange(w, device="cuda", dtype=torch.float64).expand(h, w),
            torch.arange(h, device="cuda", dtype=torch.float64)[:, None].expand(h, w))


def _walls(u, mode):
    u = u.clone()
    if mode == "reference":
        u[0], u[-1], u[:, 0], u[:, -1] = 0, 0, 0, 0
        return u
    u[0, 1:-1, 0], u[-1, 1:-1, 0] = u[1, 1:-1, 0], u[-2, 1:-1, 0]
    u[0, 1:-1, 1], u[-1, 1:-1, 1] = 0, 0
    if mode == "inflow":
        u[1:-1, -1] = u[1:-1, -2]
        u[0, -1], u[-1, -1] = 0, 0
        u[:, 0, 0], u[:, 0, 1] = 1, 0
        return u
    u[1:-1, 0, 1], u[1:-1, -1, 1] = u[1:-1, 1, 1], u[1:-1, -2, 1]
    u[1:-1, 0, 0], u[1:-1, -1, 0] = 0, 0
    u[0, 0], u[0, -1], u[-1, 0], u[-1, -1] = 0, 0, 0, 0
    return u


def _replaced(p, sides):
    return [torch.where(s, p, q) for s, q in zip(sides, _neighbours(p))]


def _sweep(p, b, sides):
    x1, x2, y1, y2 = _replaced(p, sides)
    return (x1 + x2 + y1 + y2 - b) * 0.25


def _advected(u, solid, walls, dt=DT):
    u = _walls(u, walls)
    x, y = _grid(*u.shape[:2])
    v = _sample(u, x - u[..., 0] * dt * SPEED, y - u[..., 1] * dt * SPEED).clamp(-1, 1)
    v[solid] = 0
    return v


def _forced(v, solid, vorticity, viscosity, dt=DT):
    """Confinement, viscosity and the divergence that the pressure removes."""
    left, right, below, above = _neighbours(v)
    c = 0.5 * ((right[..., 1] - left[..., 1]) - (above[..., 0] - below[..., 0]))
    left, right, below, above = _neighbours(c.abs())
    fx, fy = 0.5 * (above - below), 0.5 * (right - left)
    scale = vorticity * c / (fx * fx + fy * fy).clamp_min(2.4414e-4).sqrt() * dt
    v = v + torch.stack((fx * scale, -fy * scale), -1)
    if viscosity > 0:
        left, right, below, above = _neighbours(v)
        v = (left + right + below + above + v / viscosity) / (4 + 1 / viscosity)
    left, right, below, above = (
        torch.where(s[..., None], torch.zeros_like(q), q)
        for s, q in zip(_neighbours(solid), _neighbours(v)))
    return v, 0.5 * ((right[..., 0] - left[..., 0]) + (above[..., 1] - below[..., 1]))


def _projected(v, p, sides):
    x1, x2, y1, y2 = _replaced(p, sides)
    return v - 0.5 * torch.stack((x2 - x1, y2 - y1), -1)


def _gaussians(u, dye, splats):
    h, w = u.shape[:2]
    x, y = _grid(h, w)
    for px, py, ax, ay, r, q in splats:
        g = torch.exp(-((px * w - x) ** 2 + (py * h - y) ** 2) / (r * r))
        u = u + torch.stack((ax * g, ay * g), -1)
        dye = None if dye is None else dye + q * g
    return u, dye


def _cone(shape, pos, r):
    x, y = _grid(*shape)
    d = ((pos[0] * shape[1] - x) ** 2 + (pos[1] * shape[0] - y) ** 2).sqrt()
    return ((r - d) / r).clamp_min(0)


def _dye(q, u, solid):
    h, w = q.shape
    vh, vw = u.shape[:2]
    x, y = _grid(h, w)
    gx, gy = x * vw / w, y * vh / h
    # which cell's obstacle a dye cell sees is decided in the type of the fields
    ox, oy = (torch.from_numpy((np.arange(n, dtype=np.float32) / np.float32(n) * np.float32(m))
                               .astype(np.int64)).cuda() for n, m in ((w, vw), (h, vh)))
    v = _sample(u, gx, gy)
    out = _sample(q, x - v[..., 0] * (w / vw) * DT * SPEED, y - v[..., 1] * (h / vh) * DT * SPEED)
    out[solid[oy[:, None], ox[None, :]]] = 0
    return out


def _float64_step(u, dye, solid, case, walls, iterations, extra=0):
    v, b = _forced(_advected(u, solid, walls), solid, case["vorticity"], case["viscosity"])
    sides = _neighbours(solid)
    p = torch.zeros_like(b)
    for _ in range(iterations):
        p = _sweep(p, b, sides)
    used = p
    if extra:  # the residual correction of reduced storage: r = b - A p, then sweeps of A e = r
        for _ in range(extra):
            used = _sweep(used, b, sides)
    v = _projected(v, used, sides)
    return v, p, None if dye is None else _dye(dye, v, solid)


def _solve(b, solid):
    """The pressure of divergence b by conjugate gradients, b made solvable on the fluid."""
    fluid = (~solid).double()
    n = fluid.sum()
    sides = _neighbours(solid)

    def apply(p):
        x1, x2, y1, y2 = _replaced(p, sides)
        return (4 * p - (x1 + x2 + y1 + y2)) * fluid
    r = -(b - (b * fluid).sum() / n) * fluid
    x, d = torch.zeros_like(b), r.clone()
    rr = (r * r).sum()
    stop = float(rr) * 1e-18
    for i in range(20000):
        q = apply(d)
        a = rr / (d * q).sum()
        x += a * d
        r -= a * q
        new = (r * r).sum()
        if i % 64 == 63 and float(new) <= stop:
            return x
        d = r + (new / rr) * d
        rr = new
    return None


def _exact_fluid(case, seed):
    inp = _fluid_inputs(case, seed)
    u = inp["flow"].double()
    dye = None if inp["dye"] is None else inp["dye"].double()
    solid = torch.zeros(u.shape[:2], dtype=torch.bool, device="cuda")
    if inp["solid"] is not None:
        solid |= torch.from_numpy(inp["solid"]).cuda() != 0
    if case["kind"] == "step":
        if case["drag"]:
            pos, vel = inp["drag"]
            g = _cone(u.shape[:2], pos, 0.08 * case["width"])
            u = (u + torch.stack((vel[0] * g, vel[1] * g), -1)).clamp(-1, 1)
        u, dye = _gaussians(u, dye, inp["splats"])
        reduced = case["storage"] != "f32"
        v, p, dye = _float64_step(u, dye, solid, case, case["walls"], case["iterations"],
                                  8 if reduced else 0)
        out = {"velocity": v, "pressure": p}
        if case["dye"]:
            out["dye"] = dye
        return out
    if case["kind"] == "frame":
        pos, vel = inp["drag"]
        g = _cone(u.shape[:2], pos, 32.0)
        u = (u + torch.stack((vel[0] * g, vel[1] * g), -1)).clamp(-1, 1)
        dye = dye + 0.5 * _cone(dye.shape, pos, 40.0)
        v, _, dye = _float64_step(u, dye, solid, {"vorticity": 0.0, "viscosity": 0.1},
                                  "reference", case["iterations"])
        return {"image": None, "arrows": None, "velocity": v, "dye": dye}
    if bool(solid.any()):
        return None  # what a solve leaves inside an obstacle has no such value
    v, b = _forced(_advected(u, solid, "inflow"), solid, 0.3, 0.0)
    p = _solve(b, solid)  # a pressure is known up to a constant
    return None if p is None else {"velocity": _projected(v, p, _neighbours(solid)),
                                   "pressure": None}


def _unet_parameters(seed):
    """Weights, biases and head in the network's order, He initialised, on the host."""
    gen = torch.Generator().manual_seed(seed + 1)
    out = [0.18 * torch.randn(32, generator=gen), 0.1 * torch.randn(1, generator=gen)]
    for ci, co, _ in _CHANNELS:
        out.append(math.sqrt(2.0 / (9 * ci)) * torch.randn((co, 9, ci), generator=gen))
        out.append(0.05 * torch.randn(co, generator=gen))
    return out


def _conv64(x, w, b):
    """ReLU of a 3x3 convolution, NHWC, as nine matrix products."""
    n, h, wd, _ = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    y = b.expand(n, h, wd, w.shape[0])
    for t in range(9):
        y = y + xp[:, t // 3:t // 3 + h, t % 3:t % 3 + wd].reshape(-1, x.shape[3]).matmul(
            w[:, t].t()).view(n, h, wd, -1)
    return y.relu()


def _pool(x):
    n, h, w, c = x.shape
    return x.view(n, h // 2, 2, w // 2, 2, c).mean((2, 4))


def _up(x):
    return x.repeat_interleave(2, 1).repeat_interleave(2, 2)


def _unet64(x, p):
    def two(x, i):
        return _conv64(_conv64(x, p[4 * i + 2], p[4 * i + 3]), p[4 * i + 4], p[4 * i + 5])
    e0 = two(x, 0)
    e1 = two(_pool(e0), 1)
    e2 = two(_pool(e1), 2)
    d = two(_pool(e2), 3)
    for i, skip in ((4, e2), (5, e1), (6, e0)):
        d = two(torch.cat((_up(d), skip), 3), i)
    return d.matmul(p[0]) + p[1]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "frame", "tolerance", "learned"):
        return _exact_fluid(case, seed)
    if kind == "batch":
        out = []
        for sc in _batch_inputs(case, seed):
            u = sc["flow"].double()
            dye = sc["dye"].double()
            solid = torch.from_numpy(sc["solid"]).cuda() != 0
            for _ in range(case["steps"]):
                u, dye = _gaussians(u, dye, sc["splats"])
                u, p, dye = _float64_step(u, dye, solid, {"vorticity": 0.3, "viscosity": 0.0},
                                          "free_slip", case["iterations"])
            out.append([u, p, dye])
        return out
    inp = _network_inputs(case, seed)
    if kind == "conv":
        leaves = [inp[k].double().requires_grad_(True) for k in ("x", "w", "b")]
        y = _conv64(*leaves)
        dx, dw, db = torch.autograd.grad(y, leaves, inp["dy"].double())
        return {"y": y.detach(), "dx": dx, "dw": dw, "db": db}
    x = torch.zeros(inp["rhs"].shape + (8,), dtype=torch.float64, device="cuda")
    x[..., 0], x[..., 1] = inp["rhs"].double(), inp["solid"].double()
    params = [q.cuda().double().requires_grad_(True) for q in _unet_parameters(seed)]
    out = _unet64(x, params)
    # the trainer's loss: relative mean-free error over the fluid cells
    fluid = (~inp["solid"]).double()
    n = fluid.sum((1, 2), keepdim=True)
    a = (out - (out * fluid).sum((1, 2), keepdim=True) / n) * fluid
    t = inp["target"].double()
    t = (t - (t * fluid).sum((1, 2), keepdim=True) / n) * fluid
    loss = (((a - t) ** 2).sum((1, 2)) / (t * t).sum((1, 2))).mean()
    grads = list(torch.autograd.grad(loss, params))
    grads[1] = None  # the loss is free of the mean: the head's bias has no gradient but round-off
    return {"out": out.detach(), "grads": grads}
