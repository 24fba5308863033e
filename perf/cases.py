"""What is timed of the particle step: one dict per case, how its inputs are made, one pass of it through the
public entry points (wrach_amd.World, the ctypes binding of include/wrach.h), the bytes and operations that a
pass cannot do without, and its values in 64 bits where they exist.

Kinds of pass:
  tick      the reference's host loop, WrachAPI::tick: one frame, then the packed triple read back.
  noalloc   one frame on a packed triple in the caller's device memory (wrach_frame_noalloc).
  render    one frame, then the canonical device buffers, waited for: what a renderer draws each frame.
  rollout   restart from the store (an upload of no particles re-packs it), `frames` frames of the reference's
            step, the canonical device buffers.
  separate  the same with mode S: `passes` separation passes over the 3x3 cells in every frame, and its report.
  learned   the same with mode L: the network's warm start, then `passes` passes.
  batch     the rollout of many worlds of different sizes in one context.
  train     `steps` Adam steps of the warm start's network on the device.

The particles of one world lie in its lower half ("uniform", "lattice": pixel centres with a jitter of 0.1) or in
64 Gaussian blobs over all of it ("blobs").  Gravity is 0, the reference's own step, or the (0, -0.1) of the
workloads here; `settle` frames under it, run once in prepare, let the world fall and pile up on its floor, and
the store then holds the settled particles."""
import ctypes
import math

import numpy as np
import torch

from wrach_amd import World, WrachConfig, _lib
from wrach_amd._lib import check

FEATURES, HIDDEN = 64, 128
PARAMS = FEATURES * HIDDEN + HIDDEN + HIDDEN * HIDDEN + HIDDEN + HIDDEN * 2 + 2
LEARNING_RATE = 1e-3


def listed():
    def world(name, kind, n, width, height, **more):
        return {"name": name, "kind": kind, "n": n, "width": width, "height": height, "cell": 1, "fill": "uniform",
                "gravity": -0.1, "frames": 1, "passes": 0, "tol": 0.0, "settle": 0, **more}
    return [
        # The reference's default view and cell size and its own physics (no gravity), a few thousand particles:
        # an interactive loop, all launches and latency.
        world("tick-4k", "tick", 4_000, 480, 352, cell=3, gravity=0.0),
        # One frame of the smallest workload on a caller's own device memory: a serving loop.
        world("noalloc-16k", "noalloc", 16_384, 512, 512, gravity=0.0),
        # The smallest workload, whole: 16,384 particles, 512 x 512, 100 frames.
        world("rollout-16k", "rollout", 16_384, 512, 512, frames=100),
        # The headline workload, whole: the falling lattice, 1,000 frames, half of them after its collapse.
        world("rollout-1m", "rollout", 1_000_000, 2048, 1024, fill="lattice", frames=1000),
        # The large-grid workload: crowded blobs in 16.8 M cells (200 of its 500 frames).
        world("rollout-4m", "rollout", 4_000_000, 4096, 4096, fill="blobs", frames=200),
        # A million particles at the reference's own step, drawn every frame.
        world("render-1m", "render", 1_000_000, 2048, 1024, fill="lattice", gravity=0.0),
        # 512 worlds of sides 256, 512 and 1024 and 1,000 to 65,536 particles in one context, 100 frames.
        {"name": "batch-512", "kind": "batch", "worlds": 512, "least": 1000, "most": 65536, "side": 256, "cell": 1,
         "gravity": -0.1, "frames": 100},
        # Separation passes that stop at a tolerance, on a small world: launches in every frame.
        world("separate-16k", "separate", 16_384, 512, 512, frames=50, passes=4, tol=0.01),
        # Two passes per frame on the dense lattice, as the frame-time figures of mode S are quoted.
        world("separate-1m", "separate", 1_000_000, 2048, 1024, fill="lattice", frames=50, passes=2),
        # One pass per frame on the collapsed lattice: hundreds of particles per cell.
        world("pile-1m", "separate", 1_000_000, 2048, 1024, fill="lattice", frames=20, passes=1, settle=600),
        # The learned frame with the passes that its warm start leaves to do.
        world("learned-1m", "learned", 1_000_000, 2048, 1024, fill="lattice", frames=10, passes=9, settle=12),
        # One epoch over a lattice's particles at the training batch used here.
        {"name": "train-8k", "kind": "train", "width": 256, "rows": 256, "batch": 8192, "steps": 8, "target": 8},
    ]


def draw(rng):
    def log(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    kind = rng.choice(["tick", "noalloc", "render", "rollout", "rollout", "batch", "separate", "learned", "train"])
    if kind == "train":
        steps = rng.randrange(4, 13)
        batch = 64 * log(4, 128)
        width = rng.randrange(100, 257)
        rows = max(16, min(256, -(-batch * steps // width)))
        return {"kind": kind, "width": width, "rows": rows, "batch": batch,
                "steps": max(1, min(steps, width * rows // batch)), "target": rng.randrange(2, 9)}
    if kind == "batch":
        return {"kind": kind, "worlds": log(4, 256), "least": log(300, 3000), "most": log(4000, 65536),
                "side": rng.randrange(96, 257), "cell": rng.choice([1, 1, 2]), "gravity": rng.choice([-0.1, 0.0]),
                "frames": log(10, 60)}
    small = kind in ("tick", "noalloc")
    n = log(500, 60_000) if small else log(2_000, 300_000) if kind == "learned" else log(2_000, 1_500_000)
    fill = rng.choice(["uniform", "lattice", "blobs"]) if kind in ("rollout", "render") else rng.choice(["uniform", "lattice"])
    # Area per particle: the lattice needs two pixels, one row of every two being empty space above it.
    area = n * (rng.uniform(2.05, 4.0) if fill == "lattice" else rng.uniform(1.5, 8.0))
    aspect = math.exp(rng.uniform(-0.7, 0.7))
    width = max(32, min(8192, int(math.sqrt(area * aspect))))
    height = max(32, min(8192, int(area / width) + 3))
    gravity = 0.0 if small or kind == "render" else rng.choice([-0.1, -0.1, 0.0])
    frames = 1 if small or kind == "render" else max(4, min(rng.randrange(20, 300), 100_000_000 // n))
    c = {"kind": kind, "n": n, "width": width, "height": height, "cell": rng.choice([1, 1, 2, 3]), "fill": fill,
         "gravity": gravity, "frames": frames, "passes": 0, "tol": 0.0, "settle": 0}
    if kind in ("separate", "learned"):
        c["cell"] = rng.choice([1, 1, 2]) if kind == "separate" else 1
        c["passes"] = rng.randrange(1, 9)
        c["frames"] = max(3, min(30, 6_000_000 // n))
        if kind == "separate":
            c["tol"] = rng.choice([0.0, 0.0, 0.01])
            if gravity and c["cell"] == 1:
                c["settle"] = rng.choice([0, 0, 300])
    return c


# ---------------------------------------------------------------------------
# Inputs.

def particles(case, seed):
    """Positions and velocities (float32) of a world's particles, in the order of its upload."""
    r = np.random.Generator(np.random.PCG64(seed))
    n, w, h = case["n"], case["width"], case["height"]
    if case["fill"] == "lattice":
        i = np.arange(n)
        pos = np.stack([i % w + 0.5, i // w + 0.5], 1) + r.uniform(-0.1, 0.1, (n, 2))
        vel = r.normal(0.0, 0.5, (n, 2))
    elif case["fill"] == "blobs":
        centres = r.uniform(0.0, 1.0, (64, 2)) * (w, h)
        sigma = r.uniform(1 / 512, 1 / 32, 64) * math.sqrt(w * h)
        which = r.integers(0, 64, n)
        pos = np.clip(centres[which] + r.normal(0.0, 1.0, (n, 2)) * sigma[which, None], 0.0, (w, h))
        vel = r.normal(0.0, 1.0, (n, 2))
    else:
        pos = r.uniform(0.0, 1.0, (n, 2)) * (w, h / 2)
        vel = r.uniform(-1.0, 1.0, (n, 2))
    return pos.astype(np.float32), vel.astype(np.float32)


def batch_shapes(case):
    """(side, particles) of every world: three sides in turn, counts spread over their logarithm."""
    least, most = case["least"], case["most"]
    return [(case["side"] << (w % 3), int(least * (most / least) ** (w * 0.6180339887498949 % 1.0)))
            for w in range(case["worlds"])]


def network(seed):
    """Weights uniform in +-1/sqrt(fan in), the last layer's a tenth of that (a displacement is well below a
    particle's radius), biases zero: the layout of wrach_learn_set_params."""
    r = np.random.Generator(np.random.PCG64(seed))
    parts = []
    for rows, cols, scale in ((FEATURES, HIDDEN, 1.0), (HIDDEN, HIDDEN, 1.0), (HIDDEN, 2, 0.1)):
        bound = scale / math.sqrt(rows)
        parts += [r.uniform(-bound, bound, rows * cols), np.zeros(cols)]
    return np.concatenate(parts).astype(np.float32)


def lattice_of(case):
    return {"n": case["width"] * case["rows"], "width": case["width"], "height": 2 * case["rows"], "fill": "lattice"}


def training_order(case, seed):
    rows = case["width"] * case["rows"]
    r = np.random.Generator(np.random.PCG64([seed, 1]))
    return r.permutation(rows)[: case["batch"] * case["steps"]].astype(np.uint32)


def config(width, height, cell, gravity):
    return WrachConfig(dimensions=(width, height), cell_size=cell, gravity=(0.0, gravity))


NOTHING = np.zeros((0, 2), np.float32)


def prepare(case, seed):
    kind = case["kind"]
    state = {"kind": kind, "case": case}
    if kind == "train":
        c = lattice_of(case)
        world = World(config(c["width"], c["height"], 1, -0.1))
        world.learn_set_params(network(seed))
        world.add_particles(*particles(c, seed))
        world.learn_sample(case["target"])
        return {**state, "world": world, "order": training_order(case, seed)}
    if kind == "batch":
        shapes = batch_shapes(case)
        world = World([config(s, s, case["cell"], case["gravity"]) for s, _ in shapes])
        for w, (s, n) in enumerate(shapes):
            c = {"n": n, "width": s, "height": s, "fill": "uniform"}
            world.add_particles(*particles(c, [seed, w]), world=w)
        world.prepare(case["frames"])
        return {**state, "world": world}
    pos, vel = particles(case, seed)
    cfg = config(case["width"], case["height"], case["cell"], case["gravity"])
    if kind == "noalloc":
        key, _, pos, vel, cells = packed(case, pos, vel)
        settings = _lib.WorldSettingsC()
        settings.view_dimensions[:] = [float(case["width"]), float(case["height"])]
        settings.view_anchor[:] = [0.0, 0.0]
        settings.grid_dimensions[:] = grid(case)
        settings.cell_size = case["cell"]
        settings.particles_in_frame_count = len(pos)
        return {**state, "lib": _lib.load(), "settings": settings, "gravity": (ctypes.c_float * 2)(*cfg.gravity),
                "indices": torch.from_numpy(offsets(key, cells)).cuda(), "pos": torch.from_numpy(pos).cuda(),
                "vel": torch.from_numpy(vel).cuda()}
    world = World(cfg)
    world.add_particles(pos, vel)
    if case["settle"]:
        world.step(case["settle"])
        world.store_write_back()
        world.add_particles(NOTHING, NOTHING)
    if kind == "separate":
        world.set_solver("S", case["passes"], case["tol"])
    elif kind == "learned":
        world.learn_set_params(network(seed))
        world.set_solver("L", case["passes"])
    world.prepare(case["frames"])
    return {**state, "world": world}


# ---------------------------------------------------------------------------
# One pass.

class DeviceArray:
    """A device pointer of a world's as an array that torch takes over without a copy; the tensor keeps this
    object, and so the world whose memory it is."""

    def __init__(self, world, pointer, shape, typestr):
        self.world = world
        self.__cuda_array_interface__ = {"data": (pointer, False), "shape": shape, "typestr": typestr, "version": 2}


def canonical(world):
    v = world.device_state(canonical=True)
    world.sync()
    return [torch.as_tensor(DeviceArray(world, v.indices, (v.n_indices,), "<i4"), device="cuda"),
            torch.as_tensor(DeviceArray(world, v.positions, (v.n_particles, 2), "<f4"), device="cuda"),
            torch.as_tensor(DeviceArray(world, v.velocities, (v.n_particles, 2), "<f4"), device="cuda")]


def run(state):
    kind, case = state["kind"], state["case"]
    if kind == "noalloc":
        indices, pos, vel = state["indices"], state["pos"], state["vel"]
        check(state["lib"].wrach_frame_noalloc(
            ctypes.byref(state["settings"]), state["gravity"], 1.0, indices.data_ptr(), pos.data_ptr(),
            vel.data_ptr(), len(pos), torch.cuda.current_stream().cuda_stream))
        return [indices, pos, vel]
    world = state["world"]
    if kind == "tick":
        world.step(1)
        return list(world.read())
    if kind == "render":
        world.step(1)
        return canonical(world)
    if kind == "train":
        losses = world.learn_train(state["order"], case["batch"], LEARNING_RATE)
        return [losses, world.learn_params()]
    world.add_particles(NOTHING, NOTHING, world=0 if kind == "batch" else None)
    world.step(case["frames"])
    out = canonical(world)
    if kind in ("separate", "learned"):
        out.append(world.solver_stats())
    if kind == "learned":
        out.append(world.learned_stats())
    return out


# ---------------------------------------------------------------------------
# What a pass cannot do without.

def grid(case):
    return [case["width"] // case["cell"] + 1, case["height"] // case["cell"] + 1]


def work(case):
    if case["kind"] == "train":
        rows = case["batch"] * case["steps"]
        weights = FEATURES * HIDDEN + HIDDEN * HIDDEN + 2 * HIDDEN
        # A row's features and target once; the parameters and Adam's moments read and written every step.
        return {"bytes": rows * (2 * FEATURES + 8 + 4) + case["steps"] * 24 * PARAMS,
                "flops": rows * 2 * (3 * weights - FEATURES * HIDDEN)}
    if case["kind"] == "batch":
        n = sum(k for _, k in batch_shapes(case))
        cells = sum((s // case["cell"] + 1) ** 2 for s, _ in batch_shapes(case))
    else:
        n, cells = case["n"], grid(case)[0] * grid(case)[1]
    # A frame: a particle's position, velocity and cell read and written by the collision and by the re-bin
    # (72 bytes), a cell's count and offset (16 bytes); some 40 operations for each particle.
    frames = case["frames"]
    total, flops = 72.0 * n + 16.0 * (cells + 2), 40.0 * n
    passes = case.get("passes", 0)
    if passes:
        # A pass reads and writes the positions and meets the particles of the 3x3 cells: about one a pixel where
        # they have not fallen; piled up, the columns above three cells of the floor.
        side = case["cell"]
        near = 9.0 * side * side * min(1.0, 2.0 * n / (case["width"] * case["height"]))
        if case["settle"] >= 300:
            near = 2.5 * side * n / case["width"]
        total += passes * 16.0 * n
        flops += passes * n * near * 12.0
    if case["kind"] == "learned":
        total += 2 * 2.0 * FEATURES * n
        flops += n * (2.0 * (FEATURES * HIDDEN + HIDDEN * HIDDEN + 2 * HIDDEN) + 24 * 8)
    return {"bytes": frames * total, "flops": frames * flops}


# ---------------------------------------------------------------------------
# The values in 64 bits.  A frame's packed order depends on the cell of every f32 position, and after several
# frames on all of them, so a frame's values exist for one frame from the inputs: evaluated in f32 for the order
# and for what is decided by comparison, and beside it in 64 bits.

def packed(case, pos, vel):
    """The particles sorted by cell, stable: (cell, upload index, positions, velocities, cells)."""
    gx, gy = grid(case)
    c = np.trunc(pos / np.float32(case["cell"])).astype(np.int64)
    inside = (c[:, 0] < gx) & (c[:, 1] < gy)
    key = np.where(inside, c[:, 1] * gx + c[:, 0], -1)
    order = np.argsort(key, kind="stable")[int((~inside).sum()):]
    return key[order], order, pos[order], vel[order], gx * gy


def offsets(key, cells):
    """[0, start of every cell, n] as the packed triple holds them."""
    out = np.zeros(cells + 2, np.int32)
    out[2:] = np.cumsum(np.bincount(key, minlength=cells))
    return out


def plain_frame(case, seed):
    key, _, pos, vel, cells = packed(case, *particles(case, seed))
    starts = np.flatnonzero(np.concatenate([[True], key[1:] != key[:-1]]))
    counts = np.minimum(np.diff(np.concatenate([starts, [len(key)]])), 9)
    p32, p64 = pos.copy(), pos.astype(np.float64)
    for i in range(8):  # the pairs of a cell's first nine particles, in order
        for j in range(i + 1, 9):
            at = starts[counts > j]
            if not len(at):
                continue
            d = p32[at + i] - p32[at + j]
            reach = np.sqrt(d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1])
            a, b = (at + i)[reach <= 1], (at + j)[reach <= 1]
            for p in (p32, p64):
                e = p[b] - p[a]
                d = np.sqrt(e[:, 0] * e[:, 0] + e[:, 1] * e[:, 1])
                d[d == 0] = 0.0001
                e = e * ((p.dtype.type(0.5) * (1 - d)) / d)[:, None]
                p[a] -= e
                p[b] += e
    v32, v64 = vel.copy(), vel.astype(np.float64)
    for v, p in ((v32, p32), (v64, p64)):
        if case["gravity"]:
            v[:, 1] += np.float32(case["gravity"])
        p += v
    for axis, wall in ((0, case["width"]), (1, case["height"])):
        for edge, over in ((wall, p32[:, axis] > wall), (0, p32[:, axis] < 0)):
            for p, v in ((p32, v32), (p64, v64)):
                p[over, axis] = edge
                v[over, axis] *= -1
    for v in (v32, v64):
        np.clip(v, -1, 1, out=v)
    gx = grid(case)[0]
    c = np.floor(p32 / np.float32(case["cell"])).astype(np.int64)
    key = c[:, 1] * gx + c[:, 0]
    order = np.argsort(key, kind="stable")
    return [offsets(key, cells), p64[order], v64[order]]


def neighbours(pos, near, most=0):
    """For each particle the others whose cell lies within `near` cells on both axes: a mask in blocks of rows, or
    with `most` the nearest that many (their indices, and which of them are there)."""
    cell = pos.floor()
    for s in range(0, len(pos), 512):
        block = slice(s, min(s + 512, len(pos)))
        d = pos[None] - pos[block, None]
        mask = ((cell[None] - cell[block, None]).abs() <= near).all(2)
        mask[torch.arange(mask.shape[0]), torch.arange(block.start, block.stop)] = False
        sq = torch.where(mask, (d * d).sum(2), torch.inf)
        if most:
            yield block, torch.topk(sq, most, dim=1, largest=False)
        else:
            yield block, d, sq


def plain_training(case, seed):
    """The same Adam steps in 64 bits: features of the 16 nearest within two cells, the displacement of `target`
    separation passes, the network with its weights, inputs and first activations rounded to bf16."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    pos, vel = (torch.from_numpy(x).double().to(dev) for x in particles(lattice_of(case), seed))
    order = torch.argsort((pos[:, 1].floor() * (case["width"] + 1) + pos[:, 0].floor()), stable=True)
    pos, vel = pos[order], vel[order]

    def rounded(x):
        return x.float().bfloat16().double()
    rows = []
    for block, (sq, j) in neighbours(pos, 2, 16):
        x = torch.cat([pos[j] - pos[block, None], vel[j] - vel[block, None]], 2)
        rows.append(rounded(torch.where(torch.isinf(sq)[..., None], 0.0, x)).flatten(1))
    x = torch.cat(rows)
    at = pos
    near = torch.cat([torch.where(torch.isinf(sq), -1, j) for _, (sq, j) in neighbours(pos, 1, min(16, len(pos) - 1))])
    for _ in range(case["target"]):
        e = at[near.clamp(min=0)] - at[:, None]
        d = e.square().sum(2).sqrt()
        hit = (near >= 0) & (d <= 1)
        d = torch.where(d == 0, 0.0001, d)
        move = torch.where(hit[..., None], -e * (0.5 * (1 - d) / d)[..., None], 0.0).sum(1)
        at = at + move / hit.sum(1).clamp(min=1)[:, None]
    target = at - pos
    w = torch.from_numpy(network(seed)).double().to(dev)
    shapes = ((FEATURES, HIDDEN), (HIDDEN,), (HIDDEN, HIDDEN), (HIDDEN,), (HIDDEN, 2), (2,))
    m, v, losses = torch.zeros_like(w), torch.zeros_like(w), []
    sel = torch.from_numpy(training_order(case, seed).astype(np.int64)).to(dev)
    for step in range(case["steps"]):
        rows = sel[step * case["batch"]:(step + 1) * case["batch"]]
        parts = torch.split(w, [math.prod(s) for s in shapes])
        leaf = [(rounded(q) if len(s) == 2 else q).reshape(s).clone().requires_grad_() for q, s in zip(parts, shapes)]
        a1 = torch.nn.functional.silu(x[rows] @ leaf[0] + leaf[1])
        a1 = a1 + (rounded(a1) - a1).detach()
        a2 = torch.nn.functional.silu(a1 @ leaf[2] + leaf[3])
        loss = (a2 @ leaf[4] + leaf[5] - target[rows]).square().sum() / (2 * len(rows))
        losses.append(loss.detach())
        g = torch.cat([q.flatten() for q in torch.autograd.grad(loss, leaf)])
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        t = step + 1
        w = w - LEARNING_RATE * (m / (1 - 0.9 ** t)) / ((v / (1 - 0.999 ** t)).sqrt() + 1e-8)
    return [torch.stack(losses).cpu(), w.cpu()]


def exact(case, seed):
    if case["kind"] in ("tick", "noalloc", "render"):
        return plain_frame(case, seed)
    if case["kind"] == "train":
        return plain_training(case, seed)
    return None  # many frames: no value beyond the f32 one
