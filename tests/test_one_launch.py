"""A small world's step in one launch against the same step in a launch per phase, bit for
bit: the same worlds in a handle of their own and in one with more worlds than the
one-launch step takes.  Every solver mode, split steps, steps of no time and sizes on both
sides of the body limit; the phase times of the profile."""
import os

import numpy as np
import pytest

import dbox_amd
from dbox_amd import native, scenes, warmstart

pytestmark = pytest.mark.gpu
DT = 1.0 / 60.0
NETWORK = os.path.join(os.path.dirname(os.path.abspath(dbox_amd.__file__)), "learned", "warmstart_c12.npz")
BASE = native.WARM | native.SLEEP
MODES = {
    "default": BASE | native.CCD | native.ORDERED,
    "no continuous pass": BASE | native.ORDERED,
    "coloured": BASE | native.CCD,
    "cold": native.CCD | native.ORDERED,
    "residual": BASE | native.ORDERED | native.RESIDUAL,
    "learned": BASE | native.ORDERED | native.RESIDUAL | native.LEARNED,
    "learned, fixed iterations": BASE | native.CCD | native.ORDERED | native.LEARNED,
    "split": BASE | native.CCD | native.ORDERED | native.PRESOLVE,
}


def _worlds():
    return [scenes.mixed_container(n, 2.0 + n ** 0.5, 4.0 + 2.0 * n ** 0.5, n) for n in (1, 15, 16, 47, 63, 64, 100, 126)] + [
        scenes.hello_world(), scenes.chain_terrain(), scenes.sensor_container(60), scenes.projectile_room(),
        scenes.joint_world(3), scenes.joint_world(4, debris=30), scenes.pyramid(9, seed=2)]


def _handle(ws, fill=0, graph=False):
    h = native.StepWorlds(contacts_per_fixture=16, use_graph=graph)
    for s in ws:
        h.add_scene(s)
    for _ in range(fill):
        h.add_scene(scenes.hello_world())
    h.finalize()
    return h


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("mode", list(MODES))
def test_one_launch_equals_separate_launches(mode, graph):
    print(f"case: one launch per step, {mode}, graph {graph}", flush=True)
    ws = _worlds()
    hs = _handle(ws, graph=graph), _handle(ws, fill=1100)
    flags = MODES[mode]
    for h in hs:
        h.set_residual(1e-3, 30)
        if flags & native.LEARNED:
            h.mlp_set(*warmstart.load_network(NETWORK)[:2])
    events = 0
    for i in range(40):
        for h in hs:
            h.step(0.0 if i == 25 else DT, 8, 3, flags)
            if flags & native.PRESOLVE:
                h.step_finish()
        if i % 8 == 7 or i == 25:
            one, many = hs
            assert np.array_equal(one.toi_events(), many.toi_events()[:len(ws)])
            assert one.residuals().tobytes() == many.residuals()[:len(ws)].tobytes()
            events += int(one.toi_events().sum())
            for w in range(len(ws)):
                for read in ("bodies", "contacts", "events", "joints", "fat_aabbs", "pairs"):
                    a, b = (getattr(h, read)(w) for h in hs)
                    assert a.tobytes() == b.tobytes(), f"step {i + 1}, world {w}: {read}"
    assert events > 0 or not flags & native.CCD


@pytest.mark.parametrize("bodies", [127, 128, 129, 130])  # up to 128 a world alone steps in one launch
def test_worlds_around_the_body_limit(bodies):
    print(f"case: a world of {bodies} bodies alone and among others", flush=True)
    s = scenes.mixed_container(bodies - 1, 2.0 + bodies ** 0.5, 4.0 + 2.0 * bodies ** 0.5, bodies)
    assert len(s.bodies) == bodies
    one, many = _handle([s]), _handle([s], fill=1100)
    for mode in ("default", "coloured", "residual"):
        for h in (one, many):
            h.set_residual(1e-3, 30)
            h.step(DT, 8, 3, MODES[mode], n=12)
            h.sync()
        for read in ("bodies", "contacts", "events", "fat_aabbs", "pairs"):
            assert getattr(one, read)(0).tobytes() == getattr(many, read)(0).tobytes(), (mode, read)
    one.close()
    many.close()


def test_profile_of_a_one_launch_step():
    h = _handle([scenes.mixed_container(40, 14.0, 30.0, 3)])
    for _ in range(3):
        h.step(DT, flags=MODES["default"], n=20)
        h.sync()
        p = h.profile()
        parts = [v for k, v in p.items() if k != "step"]
        assert min(parts) >= 0.0 and 0.0 < p["solve"] < p["step"], p
        assert p["collide"] > 0.0 and p["solveTOI"] > 0.0 and p["broadphase"] > 0.0, p
    ms, n = h.phase_totals()
    assert n > 0 and all(v > 0.0 for v in ms.values()), ms
