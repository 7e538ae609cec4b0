"""What this framework is timed on: steps of worlds through `StepWorlds`, read back the way their callers read
them, and the learned warm start's network and the device broadphase through their own entry points.

A case is a dict of plain values:

  scene     what a world holds, by the generators of dbox_amd.scenes: "hello", "pyramid", "container" (one mixed
            container), "containers" (a batch of containers of lognormal sizes), "terrain", "joints", "room",
            "stacks"; or "network" / "broadphase" for the stand-alone entry points
  worlds    independent worlds of the handle
  size      bodies of a world (rows for "pyramid" up to 40, boxes above), rows of "network", proxies of "broadphase"
  steps     b2World.Step calls of one pass
  lead      steps taken in prepare(), so that a pass starts from contacts and piles and not from free fall
  solver    "exact" (the reference's solve order), "coloured" (this binding's default) or "learned" (exact order,
            iterated to a residual, new points started by the network)
  ccd       continuous physics
  read      "frame": every step is synchronised and its bodies and contacts read, as a game's loop does;
            "listener": the same with the PreSolve split and the listener's callbacks, as the hook in b2World.Step
            does; "end": the bodies of every world after the last step, as a batch of simulations does
  again     every pass first puts all bodies back to where prepare() left them (an episode, a rollout from a
            snapshot); without it a pass goes on from where the last one ended

All steps are dbox's defaults otherwise: 1/60 s, 8 velocity and 3 position iterations, warm starting and sleeping.
"""
from __future__ import annotations

import os

import numpy as np
import torch

import dbox_amd
from dbox_amd import native, scenes, warmstart

DT, VEL, POS = 1.0 / 60.0, 8, 3
NETWORK = os.path.join(os.path.dirname(os.path.abspath(dbox_amd.__file__)), "learned", "warmstart_c12.npz")


def _case(name, scene, worlds, size, steps, lead, solver, ccd, read, again):
    c = {"scene": scene, "worlds": worlds, "size": size, "steps": steps, "lead": lead, "solver": solver, "ccd": ccd,
         "read": read, "again": again}
    return dict(c, name=name) if name else c


def listed():
    return [
        # examples/hello_world: one box dropped on a ground box, its position printed after each of 60 steps.  The
        # smallest call there is: every step is launches, one wait and read-backs.
        _case("hello_world", "hello", 1, 2, 60, 0, "exact", True, "frame", True),
        # the demo's pyramid (20 rows, 210 boxes), drawn every frame: the ordinary single world.
        _case("pyramid_20_rows", "pyramid", 1, 20, 60, 0, "exact", True, "frame", True),
        # a game level: bodies on a terrain of chains, with a contact listener that gets PreSolve.
        _case("terrain_listener", "terrain", 1, 60, 45, 0, "exact", True, "listener", True),
        # 64 worlds of all the joint kinds (bridge, car, pulley, ...), run as episodes of a second.
        _case("joint_worlds_64", "joints", 64, 43, 60, 0, "exact", True, "end", True),
        # 64 closed rooms of 40 fast projectiles: the continuous pass does the work.
        _case("projectile_rooms_64", "room", 64, 40, 40, 0, "exact", True, "end", True),
        # step()'s own defaults: coloured solver, no continuous physics, a batch of a few hundred small worlds.
        _case("containers_256_coloured", "containers", 256, 64, 60, 240, "coloured", False, "end", False),
        # the benchmark: 4096 containers of 8 to 1024 bodies, from step 300 on.
        _case("containers_4096", "containers", 4096, 64, 60, 300, "exact", True, "end", False),
        # 128 worlds of tall stacks started by the network and iterated to a residual: the learned warm start in use.
        _case("stacks_128_learned", "stacks", 128, 104, 10, 20, "learned", False, "end", False),
        # one world too big for one workgroup: 20,000 bodies, many small islands over a growing pile.
        _case("container_20000", "container", 1, 20000, 12, 180, "exact", True, "end", True),
        # the other kind of big world: 50,000 boxes that are one island once they touch.
        _case("pyramid_50000", "pyramid", 1, 50000, 6, 36, "exact", True, "end", True),
        # the network alone, forward and gradients, at the training batch of the shipped network.
        _case("network_8192", "network", 1, 8192, 1, 0, "learned", False, "end", False),
        # the stand-alone device broadphase near its largest size.
        _case("broadphase_16000", "broadphase", 1, 16000, 1, 0, "exact", False, "end", False),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["pyramid", "container", "terrain", "joints", "room", "containers", "containers", "stacks",
                       "big container", "big pyramid", "network", "broadphase"])
    ccd = rng.random() < 0.75
    exact = "exact" if rng.random() < 0.75 else "coloured"
    read = rng.choice(["frame", "listener", "end"])
    if kind == "pyramid":
        return _case(None, "pyramid", 1, rng.randint(2, 32), rng.randint(20, 60), 0, exact, ccd, read, True)
    if kind == "container":
        return _case(None, "container", 1, _log_int(rng, 9, 900), rng.randint(20, 60), 0, exact, ccd, read, True)
    if kind == "terrain":
        return _case(None, "terrain", 1, rng.randint(5, 150), rng.randint(20, 60), 0, "exact", True, read, True)
    if kind == "joints":
        return _case(None, "joints", _log_int(rng, 1, 200), 43, rng.randint(20, 60), 0, exact, ccd, "end", True)
    if kind == "room":
        return _case(None, "room", _log_int(rng, 1, 200), rng.randint(8, 70), rng.randint(20, 40), 0, "exact", True,
                     "end", True)
    if kind == "containers":
        return _case(None, "containers", _log_int(rng, 3, 2000), 64, rng.randint(20, 60), rng.randint(120, 300), exact,
                     ccd, "end", False)
    if kind == "stacks":
        return _case(None, "stacks", _log_int(rng, 1, 250), 104, rng.randint(5, 10), rng.randint(5, 40),
                     rng.choice(["learned", "exact"]), False, "end", False)
    if kind == "big container":
        return _case(None, "container", 1, _log_int(rng, 1500, 20000), rng.randint(6, 12), rng.randint(20, 180), "exact",
                     ccd, "end", True)
    if kind == "big pyramid":
        return _case(None, "pyramid", 1, _log_int(rng, 1500, 50000), rng.randint(3, 6), rng.randint(5, 36), "exact",
                     ccd, "end", True)
    if kind == "network":
        return _case(None, "network", 1, _log_int(rng, 17, 120000), 1, 0, "learned", False, "end", False)
    return _case(None, "broadphase", 1, _log_int(rng, 50, 16384), 1, 0, "exact", False, "end", False)


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _scenes(c, seed):
    kind, n, worlds = c["scene"], c["size"], c["worlds"]
    base = 0x9E3779B1 * (seed + 1) & 0x7FFFFFFFFFFF
    if kind == "hello":  # the example's box, dropped from a little higher and turned a little
        s = scenes.hello_world()
        u = scenes.Stream(base).uniform(2)
        s.bodies[1]["py"] = 4.0 + u[0]
        s.bodies[1]["angle"] = 0.4 * u[1]
        return [s]
    if kind == "pyramid":
        return [scenes.pyramid(n, seed=base) if n <= 40 else scenes.big_pyramid(n, seed=base)]
    if kind == "container":
        if n > 1000:  # at the density of 20,000 bodies in 200 m x 400 m
            return [scenes.mixed_container(n, 200.0 * (n / 20000.0) ** 0.5, 400.0 * (n / 20000.0) ** 0.5, base)]
        return [scenes.mixed_container(n, 40.0, 80.0, base)]
    if kind == "containers":  # the benchmark's sizes, filled anew
        return scenes.batched_worlds(worlds, seed=base, sizes=scenes.world_sizes(worlds, scenes.config_seed(3)))
    if kind == "stacks":  # the stack workload's boxes, each a little off its place
        out = scenes.stack_worlds(worlds)
        for w, s in enumerate(out):
            s.bodies["px"][1:] += scenes.Stream(base ^ (w + 1)).uniform(len(s.bodies) - 1, -0.01, 0.01)
        return out
    make = {"terrain": lambda s: scenes.chain_terrain(n, seed=s), "room": lambda s: scenes.projectile_room(n, seed=s),
            "joints": lambda s: scenes.joint_world(s)}[kind]
    return [make(base ^ (w + 1) * 0x632BE5AB) for w in range(worlds)]


def _flags(c):
    f = native.WARM | native.SLEEP | (native.CCD if c["ccd"] else 0)
    if c["solver"] == "exact":
        f |= native.ORDERED
    if c["solver"] == "learned":
        f |= native.ORDERED | native.RESIDUAL | native.LEARNED
    return f


def _network_rows(n, seed):
    """Feature rows and labels with the mean and spread that the shipped network was fitted to."""
    params, norm, _ = warmstart.load_network(NETWORK)
    g = np.random.default_rng(seed)
    x = norm[:14] + g.standard_normal((n, 14), np.float32) / norm[14:28]
    t = norm[28:30] + g.standard_normal((n, 2), np.float32) * norm[30:32]
    return params, norm, x.astype(np.float32), t.astype(np.float32)


def prepare(case, seed):
    c = case
    h = native.StepWorlds()
    if c["scene"] == "network":
        params, norm, x, t = _network_rows(c["size"], seed)
        h.mlp_set(params, norm)
        return {"case": c, "h": h, "x": x, "t": t}
    if c["scene"] == "broadphase":
        # the fat AABBs of bodies of 0.2 to 1 m at the density of a pile, two thirds of them moved
        n, g = c["size"], torch.Generator(device="cuda").manual_seed(seed)
        side = (1.6 * n) ** 0.5
        centre = torch.rand((n, 2), generator=g, device="cuda") * side
        half = 0.2 + 0.8 * torch.rand((n, 2), generator=g, device="cuda")
        moved = (torch.rand(n, generator=g, device="cuda") < 2.0 / 3.0).to(torch.int32)
        cap = 32 * n
        s = {"case": c, "h": h, "fat": torch.cat([centre - half, centre + half], 1).contiguous(), "moved": moved,
             "pairs": torch.zeros((cap, 2), dtype=torch.int32, device="cuda"),
             "count": torch.zeros(1, dtype=torch.int32, device="cuda")}
        torch.cuda.synchronize()
        return s
    for s in _scenes(c, seed):
        h.add_scene(s)
    h.finalize()
    if c["solver"] == "learned":
        params, norm, _ = warmstart.load_network(NETWORK)
        h.mlp_set(params, norm)
        h.set_residual(1e-3, 100)
    state = {"case": c, "h": h, "flags": _flags(c)}
    if c["lead"]:
        h.step(DT, VEL, POS, state["flags"], n=c["lead"])
        h.sync()
    if c["again"]:
        state["start"] = [h.bodies(w) for w in range(h.world_count)]
    return state


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------
def _floats(bodies):
    """Body states as 16 floats each (the flags column keeps its bits)."""
    return bodies.view(np.float32).reshape(-1, 16)


def _rows(frames, per_frame):
    """The records of all frames one after the other, as the 32-bit words they are, and each frame's count; a fixed
    number of rows, zeros after the last."""
    words = frames[0].dtype.itemsize // 4
    out, at = np.zeros((per_frame * len(frames), words), np.int32), 0
    for f in frames:
        out[at:at + len(f)] = f.view(np.int32).reshape(len(f), words)
        at += len(f)
    return {"rows": out, "counts": np.array([len(f) for f in frames])}


def run(state):
    c, h = state["case"], state["h"]
    if c["scene"] == "network":
        y = h.mlp_forward(state["x"])
        grad, loss = h.mlp_gradients(state["x"], state["t"])
        return {"y": y, "grad": grad, "loss": loss}
    if c["scene"] == "broadphase":
        h._check(h.L.dbx_broadphase_pairs_noalloc(h.h, state["fat"].data_ptr(), state["moved"].data_ptr(), c["size"],
                                                  state["pairs"].data_ptr(), len(state["pairs"]),
                                                  state["count"].data_ptr()))
        h.sync()
        return {"pairs": state["pairs"], "count": state["count"]}
    flags = state["flags"]
    if c["again"]:
        for w, b in enumerate(state["start"]):
            h.write_bodies(w, b)
    if c["read"] == "end":
        h.step(DT, VEL, POS, flags, n=c["steps"])
        h.sync()
        return {"bodies": _floats(np.concatenate([h.bodies(w) for w in range(h.world_count)]))}
    bodies, contacts, events = [], [], []
    for _ in range(c["steps"]):
        if c["read"] == "listener":
            h.step(DT, VEL, POS, flags | native.PRESOLVE)
            events.append(h.events())
            h.step_finish()
        else:
            h.step(DT, VEL, POS, flags)
        h.sync()
        bodies.append(h.bodies())
        if c["read"] == "listener":
            events.append(h.events())
        else:
            contacts.append(h.contacts())
    out, n = {"bodies": _floats(np.concatenate(bodies))}, h.fixture_counts[0]
    if contacts:
        out["contacts"] = _rows(contacts, 8 * n + 64)
    if events:
        out["events"] = _rows(events, 16 * n + 64)
    return out


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def work(case):
    c = case
    if c["scene"] == "network":  # rows read once, predictions and gradients written; forward twice, backward twice
        n = c["size"]
        return {"bytes": n * (14 + 2 + 2) * 4 + 3 * 5250 * 4, "flops": n * 2 * 5120 * 4}
    if c["scene"] == "broadphase":  # AABBs and flags read, about six pairs a proxy written
        n = c["size"]
        return {"bytes": n * (16 + 4 + 6 * 8), "flops": n * 6 * 4}
    bodies = c["worlds"] * c["size"]
    if c["scene"] == "pyramid" and c["size"] <= 40:
        bodies = c["size"] * (c["size"] + 1) // 2
    if c["scene"] == "containers":
        bodies = c["worlds"] * 88  # mean of the lognormal sizes
    contacts = 2 * bodies
    # a step: body state (92 B read, 76 B written), contacts (84 B read, 16 B written), shapes; about 100 operations a
    # contact and velocity iteration, 150 a position iteration, 300 for its manifold
    per_step = bodies * (92 + 76 + 84) + contacts * (84 + 16)
    flops = contacts * (300 + 100 * VEL + 150 * POS)
    reads = bodies * 64 * (1 if c["read"] == "end" else c["steps"])
    return {"bytes": c["steps"] * per_step + reads, "flops": c["steps"] * flops}


def tolerance(case):
    if case["scene"] == "network":
        return {"rel": 1e-4}
    return "exact"  # a step is the reference's sequence of float operations, to the bit; pairs are whole numbers


def exact(case, seed):
    """The network in 64 bits; a step has no 64-bit value (its floats are the reference's sequence of roundings)."""
    if case["scene"] != "network":
        return None
    params, norm, x, t = _network_rows(case["size"], seed)
    p, m = params.astype(np.float64), norm.astype(np.float64)
    w1, b1, w2, b2, w3, b3 = np.split(p, [896, 960, 5056, 5120, 5248])
    w1, w2, w3 = w1.reshape(64, 14), w2.reshape(64, 64), w3.reshape(2, 64)
    xn = (x.astype(np.float64) - m[:14]) * m[14:28]
    h1 = np.maximum(xn @ w1.T + b1, 0.0)
    h2 = np.maximum(h1 @ w2.T + b2, 0.0)
    y = h2 @ w3.T + b3
    e = y - (t.astype(np.float64) - m[28:30]) / m[30:32]
    dy = 2.0 * e / len(x)
    dz2 = (dy @ w3) * (h2 > 0.0)
    dz1 = (dz2 @ w2) * (h1 > 0.0)
    grad = np.concatenate([(dz1.T @ xn).ravel(), dz1.sum(0), (dz2.T @ h1).ravel(), dz2.sum(0), (dy.T @ h2).ravel(),
                           dy.sum(0)])
    return {"y": y * m[30:32] + m[28:30], "grad": grad, "loss": float(np.sum(e * e) / len(x))}
