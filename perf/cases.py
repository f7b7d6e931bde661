"""Cases that time the framework at its public entry points.

A case is one call pattern of a program that uses the step: a world built
through the box2d:: API (the scene runner of libbox2d.so), advanced by a few
steps, its bodies read back (b2g_get_bodies), or the warm-start network
trained and differentiated (b2g_mlp_train, b2g_mlp_gradient). Worlds are
settled before they are timed, so that a pass repeated many times goes on
meeting the load it is there to measure; the scene whose load is a transient
(bullets) is put back to its start by every pass, as an environment's reset
does.

Kinds:
  pyramid    a box pyramid of `rows` rows stepped frame by frame, the bodies
             read each frame: the interactive small world, where latency and
             the number of launches count
  pile       a random pile of circles and polygons at the spacing of the
             benchmark's (at 100 000 bodies its 300 x 600 m layout): one
             large island, the throughput path
  batch      `worlds` independent piles of `n` bodies in one context: many
             environments advanced together
  stress     a pile on a mat of jointed chains: contacts and joints
  terrain    bodies on chain shapes with continuous collision, the
             reference's default: edge contacts, few events
  bullets    fast bodies and bullets through a column of boxes into a thin
             wall with continuous collision: a chain of events per step,
             replayed from its start by every pass
  reference  the reference-order solver on a pyramid: replays that have to
             match the reference's order
  learned    a pile whose fresh contact points start from a trained network
  train      epochs of Adam over a log of contact points taken from a pile
  gradient   loss and gradient of the network over host rows
"""
import ctypes
import math
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

import box2dpp_amd  # noqa: E402

VP = ctypes.c_void_p
BODY = np.dtype([
    ("type", "<i4"), ("flags", "<i4"), ("xf", "<f4", 4), ("lc", "<f4", 2), ("c0", "<f4", 2), ("a0", "<f4"),
    ("c", "<f4", 2), ("a", "<f4"), ("v", "<f4", 2), ("w", "<f4"), ("force", "<f4", 2), ("torque", "<f4"),
    ("invMass", "<f4"), ("invI", "<f4"), ("linearDamping", "<f4"), ("angularDamping", "<f4"),
    ("gravityScale", "<f4"), ("sleepTime", "<f4"),
])
DYNAMIC = 2
FEATURES, HIDDEN = 16, 64
# b2g_mlp_params as one float array: (name, shape) in layout order
PARAMS = [("W1", (HIDDEN, FEATURES)), ("b1", (HIDDEN,)), ("W2", (HIDDEN, HIDDEN)), ("b2", (HIDDEN,)),
          ("W3", (HIDDEN, HIDDEN)), ("b3", (HIDDEN,)), ("W4", (2, HIDDEN)), ("b4", (2,)),
          ("xmean", (FEATURES,)), ("xstd", (FEATURES,)), ("ymean", (2,)), ("ystd", (2,))]
PARAM_FLOATS = sum(int(np.prod(s)) for _, s in PARAMS)
LEARNED = PARAMS[:8]
LR = 2e-3
BATCH = 65536


def listed():
    return [
        # an interactive level's frame: 210 boxes, one step, read the poses
        {"name": "pyramid_20", "kind": "pyramid", "rows": 20, "steps": 1, "vel": 8, "pos": 3},
        # a mid-sized game world's frame
        {"name": "pile_1493", "kind": "pile", "n": 1493, "steps": 1, "vel": 8, "pos": 3},
        # offline simulation: four steps per recorded frame
        {"name": "pile_9973", "kind": "pile", "n": 9973, "steps": 4, "vel": 8, "pos": 3},
        # the benchmark's size
        {"name": "pile_100000", "kind": "pile", "n": 100000, "steps": 4, "vel": 8, "pos": 3},
        # environments in lockstep, four steps per action
        {"name": "batch_32", "kind": "batch", "worlds": 32, "n": 263, "steps": 4, "vel": 8, "pos": 3},
        # ragdoll-like load: 400 chains of 32 links under 20 011 bodies
        {"name": "stress_20011", "kind": "stress", "n": 20011, "steps": 4, "vel": 8, "pos": 3},
        # a platformer level with the reference's defaults
        {"name": "terrain_200", "kind": "terrain", "n": 200, "steps": 1, "vel": 8, "pos": 3},
        # the impact of a volley: three steps, some hundred events each
        {"name": "bullets_99", "kind": "bullets", "n": 99, "steps": 3, "vel": 8, "pos": 3},
        # a replay in the reference's order
        {"name": "reference_12", "kind": "reference", "rows": 12, "steps": 1, "vel": 8, "pos": 3},
        # the learned start at two thirds of the iterations
        {"name": "learned_9973", "kind": "learned", "n": 9973, "steps": 4, "vel": 6, "pos": 2},
        # training on a pile's log
        {"name": "train_500000", "kind": "train", "points": 500000, "epochs": 2},
        # a gradient for a program's own optimiser
        {"name": "gradient_49999", "kind": "gradient", "n": 49999},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["pyramid", "pile", "pile", "batch", "stress", "terrain", "bullets", "reference", "learned",
                       "train", "gradient"])
    case = {"kind": kind}
    if kind == "pyramid":
        case["rows"] = log(4, 40)
    elif kind == "pile":
        case["n"] = log(64, 60000)
    elif kind == "batch":
        case["worlds"] = log(4, 40)
        case["n"] = log(16, 700)
    elif kind == "stress":
        case["n"] = log(1000, 20000)
    elif kind == "terrain":
        case["n"] = log(30, 300)
    elif kind == "bullets":
        case["n"] = log(24, 150)
    elif kind == "reference":
        case["rows"] = log(3, 14)
    elif kind == "learned":
        case["n"] = log(1000, 30000)
    elif kind == "train":
        case["points"] = log(20000, 500000)
        case["epochs"] = 1
    else:
        case["n"] = log(100, 200000)
    if kind not in ("train", "gradient"):
        case["steps"] = {"pyramid": 1, "reference": 1, "bullets": 3}.get(kind, rng.choice([1, 2, 4]))
        case["vel"], case["pos"] = rng.choice([(8, 3), (6, 2), (10, 4)])
    return case


# ------------------------------------------------------------------ worlds
class World:
    """A box2d:: world behind the scene runner and its device context."""

    def __init__(self, continuous=False):
        self.host, self.b2g = box2dpp_amd.host(), box2dpp_amd.b2g()
        self.b2g.b2g_last_error.restype = ctypes.c_char_p
        self.h = VP(self.host.b2pp_world_create(0.0, -10.0))
        self.host.b2pp_world_set_flags(self.h, 0, 1, int(continuous), 0)
        self.ctx = VP(self.host.b2pp_world_device_context(self.h))

    def __del__(self):
        if getattr(self, "h", None):
            self.host.b2pp_world_destroy(self.h)
            self.h = None

    def check(self, rc):
        if rc:
            raise RuntimeError("rc %d: %s" % (rc, self.b2g.b2g_last_error(self.ctx).decode()))

    def scene(self, kind, n, seed):
        self.check(self.host.b2pp_world_load_scene(self.h, kind.encode(), int(n), ctypes.c_uint(seed)))

    def scenes(self, kind, worlds, n, seed):
        self.check(self.host.b2pp_world_load_worlds(self.h, kind.encode(), int(worlds), int(n), ctypes.c_uint(seed)))

    def step(self, steps, vel, pos):
        self.check(self.host.b2pp_world_step(self.h, ctypes.c_float(1.0 / 60.0), int(vel), int(pos), int(steps)))

    def buffer(self):
        return np.zeros(self.host.b2pp_world_body_count(self.h), BODY)

    def read(self, out):
        self.check(self.b2g.b2g_get_bodies(self.ctx, 0, len(out), out.ctypes.data_as(VP)))
        return out

    def write(self, state):
        self.check(self.b2g.b2g_set_bodies(self.ctx, 0, len(state), state.ctypes.data_as(VP)))

    def params(self):
        p = np.zeros(PARAM_FLOATS, np.float32)
        self.check(self.b2g.b2g_mlp_get_params(self.ctx, p.ctypes.data_as(VP)))
        return p


def split(p, names):
    out, at = {}, 0
    for name, shape in PARAMS:
        k = int(np.prod(shape))
        if (name, shape) in names:
            out[name] = p[at:at + k].reshape(shape)
        at += k
    return out


def pile_height(n):
    """Height of the pile's start layout (columns at 1.34 m, twice as high as wide)."""
    cols = max(4, int(math.ceil(math.sqrt(0.5 * n))))
    return 1.3416 * ((n + cols - 1) // cols)


def fall_steps(height):
    """Steps until a body falling from `height` has landed and the pile has closed up."""
    return int(60.0 * math.sqrt(2.0 * height / 10.0)) + 100


def network(world, points, seed):
    """Logs contact points of the world's next steps and starts a network on them."""
    world.check(world.b2g.b2g_log_fresh(world.ctx, int(points)))
    size = ctypes.c_int(0)
    for _ in range(3000):
        world.step(1, 8, 3)
        world.check(world.b2g.b2g_log_size(world.ctx, ctypes.byref(size)))
        if size.value >= points:
            break
    else:
        raise RuntimeError("the pile gave %d of %d points" % (size.value, points))
    world.check(world.b2g.b2g_mlp_init(world.ctx, ctypes.c_uint(seed)))


def train(world, epochs, seed):
    loss = np.zeros(max(epochs, 1), np.float64)
    world.check(world.b2g.b2g_mlp_train(world.ctx, int(epochs), BATCH, ctypes.c_float(LR), ctypes.c_uint(seed),
                                        loss.ctypes.data_as(VP)))
    return loss


def rows_of(case, seed):
    """Feature rows and targets of a gradient case: standardised features, a smooth target with noise."""
    g = np.random.RandomState(seed)
    n = case["n"]
    x = g.standard_normal((n, FEATURES)).astype(np.float32)
    a, b = g.standard_normal((FEATURES, 2)) / 4.0, g.standard_normal((FEATURES, 2)) / 4.0
    t = (np.tanh(x @ a) + 0.5 * np.sin(x @ b) + 0.1 * g.standard_normal((n, 2))).astype(np.float32)
    return x, t


def weights_of(seed):
    """A network as a program keeps it: uniform weights of the layers' scale, no normalisation."""
    g = np.random.RandomState(seed + 1)
    p = np.zeros(PARAM_FLOATS, np.float32)
    w = split(p, PARAMS)
    for name in ("W1", "W2", "W3", "W4"):
        a = math.sqrt(6.0 / sum(w[name].shape))
        w[name][...] = g.uniform(-a, a, w[name].shape)
    for name in ("b1", "b2", "b3", "b4"):
        w[name][...] = g.uniform(-0.1, 0.1, w[name].shape)
    w["xstd"][...] = 1.0
    w["ystd"][...] = 1.0
    return p


def prepare(case, seed):
    kind, seed = case["kind"], int(seed) & 0x7FFFFFFF
    if kind == "gradient":
        world = World()
        x, t = rows_of(case, seed)
        world.check(world.b2g.b2g_mlp_set_params(world.ctx, weights_of(seed).ctypes.data_as(VP)))
        return {"case": case, "world": world, "x": x, "t": t}
    world = World(continuous=kind in ("terrain", "bullets"))
    state = {"case": case, "world": world}
    if kind in ("pyramid", "reference"):
        world.scene("pyramid", case["rows"], 0)
        if kind == "reference":
            world.host.b2pp_world_set_mode(world.h, 1)
        # every box starts with a small push of its own
        bodies = world.read(world.buffer())
        moving = bodies["type"] == DYNAMIC
        g = np.random.RandomState(seed)
        bodies["v"][moving] = 0.02 * g.standard_normal((int(moving.sum()), 2))
        bodies["w"][moving] = 0.02 * g.standard_normal(int(moving.sum()))
        world.write(bodies)
        world.step(30, 8, 3)
    elif kind in ("pile", "learned"):
        world.scene("world", case["n"], seed)
        world.step(fall_steps(pile_height(case["n"])), 8, 3)
        if kind == "learned":
            network(world, min(BATCH, 8 * case["n"]), seed)
            train(world, 3, seed)
            world.check(world.b2g.b2g_log_fresh(world.ctx, 0))
            world.host.b2pp_world_set_learned(world.h, 1, ctypes.c_float(0.0))
    elif kind == "train":
        world.scene("world", max(2000, case["points"] // 40), seed)
        network(world, case["points"], seed)
    elif kind == "batch":
        world.scenes("world", case["worlds"], case["n"], seed)
        world.step(fall_steps(pile_height(case["n"])), 8, 3)
    elif kind == "stress":
        world.scene("stress", case["n"], seed)
        world.step(fall_steps(600.0), 8, 3)
    elif kind == "terrain":
        world.scene("terrain", case["n"], seed)
        world.step(300, 8, 3)
    else:
        world.scene("bullets", case["n"], seed)
        world.step(8, 8, 3)  # the first bullets reach the column
        state["start"] = world.read(world.buffer())
        world.step(case["steps"], case["vel"], case["pos"])
    state["out"] = world.buffer()
    return state


def run(state):
    case, world = state["case"], state["world"]
    kind = case["kind"]
    if kind == "gradient":
        grad, loss = np.zeros(PARAM_FLOATS, np.float32), np.zeros(1, np.float64)
        world.check(world.b2g.b2g_mlp_gradient(world.ctx, state["x"].ctypes.data_as(VP),
                                               state["t"].ctypes.data_as(VP), case["n"],
                                               grad.ctypes.data_as(VP), loss.ctypes.data_as(VP)))
        return dict(split(grad, LEARNED), loss=loss)
    if kind == "train":
        loss = train(world, case["epochs"], 7)
        return dict(split(world.params(), LEARNED), loss=loss)
    if kind == "bullets":
        world.write(state["start"])
    world.step(case["steps"], case["vel"], case["pos"])
    b = world.read(state["out"])
    # poses now and before the step (a renderer interpolates them), velocities
    return {k: b[k] for k in ("flags", "xf", "c", "a", "c0", "a0", "v", "w", "sleepTime")}


# ------------------------------------------------------------------- sizes
def work(case):
    """Bytes of a step: the bodies' state in and out (and read once by the
    caller), the fixtures' shapes, boxes and materials in and the boxes out,
    the contacts' table rows and manifolds in and out. Flops of the network:
    one forward product chain, twice that for its gradient."""
    kind = case["kind"]
    chain = 2 * (FEATURES * HIDDEN + 2 * HIDDEN * HIDDEN + 2 * HIDDEN)
    if kind == "gradient":
        return {"bytes": 4 * (FEATURES + 2) * case["n"] + 8 * PARAM_FLOATS, "flops": 3 * chain * case["n"]}
    if kind == "train":
        rows = case["points"] * case["epochs"]
        return {"bytes": 4 * (FEATURES + 2) * rows + 8 * PARAM_FLOATS, "flops": 3 * chain * rows}
    contacts = 4.0
    if kind in ("pyramid", "reference"):
        n, contacts = case["rows"] * (case["rows"] + 1) // 2, 2.8
    elif kind == "batch":
        n = case["worlds"] * case["n"]
    elif kind == "stress":
        n = case["n"] + 32 * (case["n"] // 50)
    else:
        n, contacts = case["n"], 2.0 if kind in ("terrain", "bullets") else 4.0
    a_step = n * (2 * 112 + 176 + 32 + 2 * 16) + n * contacts * 2 * (64 + 32)
    # velocity and position passes: about 135 flops a constraint and pass
    flops = n * contacts * 0.6 * 135 * (case["vel"] + case["pos"])
    return {"bytes": int(case["steps"] * a_step + 112 * n), "flops": int(case["steps"] * flops)}


def tolerance(case):
    """Worlds: about four times what one unit in the last place of every
    start velocity changes in the results. Contacts amplify it, more so the
    larger and the less settled the pile. Network: BF16 products."""
    kind = case["kind"]
    if kind in ("gradient", "train"):
        return {"rel": 1e-2}
    if kind in ("pyramid", "reference", "terrain"):
        return {"rel": 5e-5, "max": 5e-4}
    if kind in ("stress", "bullets") or case.get("n", 0) > 20000:
        return {"rel": 1e-2, "max": 0.99}
    return {"rel": 5e-4, "max": 2e-2}


# ------------------------------------------------------------------- exact
def exact(case, seed):
    """The gradient in 64 bits; a step has no reference in plain numpy."""
    if case["kind"] != "gradient":
        return None
    import torch

    x, t = (torch.from_numpy(v.astype(np.float64)) for v in rows_of(case, int(seed) & 0x7FFFFFFF))
    p = weights_of(int(seed) & 0x7FFFFFFF).astype(np.float64)
    w = {k: torch.from_numpy(v.copy()).requires_grad_(True) for k, v in split(p, LEARNED).items()}
    h = x
    for i in ("1", "2", "3"):
        h = torch.nn.functional.gelu(h @ w["W" + i].T + w["b" + i])
    y = h @ w["W4"].T + w["b4"]
    loss = ((y - t) ** 2).sum() / (2.0 * case["n"])
    loss.backward()
    out = {k: v.grad.numpy() for k, v in w.items()}
    out["loss"] = np.array([float(loss)], np.float64)
    return out
