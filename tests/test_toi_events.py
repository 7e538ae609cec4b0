"""Events of the continuous pass against the oracle, bit for bit, where the work an event
spreads over a wave has its edges: bodies with fewer and more contacts than a wave has
lanes, islands up to the contact limit (b2_maxTOIContacts), bodies the event wakes, and
more contacts to look at again than one wave takes at once."""
import numpy as np
import pytest

from dbox_amd import native, scenes
from oracle import pyoracle as po
from tests.helpers import body_mismatch, contact_mismatch

pytestmark = pytest.mark.gpu
DT = 1.0 / 60.0


def _plate(n, bullets, asleep=0):
    """A plate with n small boxes on it, thrown onto the ground; the last `asleep` boxes lie
    sleeping where it lands."""
    b = scenes.body_defs(2 + n)
    b[0]["type"] = scenes.STATIC
    b[1:]["type"] = scenes.DYNAMIC
    hx = 0.06 * n + 0.5
    b[1]["py"], b[1]["vy"] = 3.0, -100.0
    x = (np.arange(n) - 0.5 * (n - 1)) * 0.1
    b[2:]["px"], b[2:]["py"], b[2:]["vy"] = x, 3.14, -100.0
    b[2:2 + bullets]["bullet"] = 1
    if asleep:
        b[-asleep:]["py"], b[-asleep:]["vy"], b[-asleep:]["awake"] = 0.045, 0.0, 0
    f = scenes.fixture_defs(2 + n)
    f["body"] = np.arange(2 + n)
    scenes._edge(f[0], 0, -50.0, 0.0, 50.0, 0.0, 0.6)
    f[1:]["shape"], f[1:]["density"], f[1:]["friction"] = scenes.SHAPE_BOX, 1.0, 0.4
    f[1]["p"][:2] = (hx, 0.1)
    f[2:]["p"][:, :2] = 0.04
    return scenes.Scene(b, f, name=f"plate{n}")


WORLDS = [_plate(1, 0), _plate(31, 31), _plate(62, 0), _plate(63, 4), _plate(64, 0), _plate(65, 40), _plate(130, 70),
          _plate(40, 10, asleep=12), _plate(200, 0, asleep=70), scenes.projectile_room(40, seed=5),
          scenes.projectile_room(9, seed=6, speed=300.0), scenes.mixed_container(60, 9.0, 40.0, 8)]


@pytest.mark.parametrize("alone", [True, False])
def test_events_equal_the_oracle(alone):
    groups = [[s] for s in WORLDS] if alone else [WORLDS]
    events = 0
    for ws in groups:
        print(f"case: TOI events of {[s.name for s in ws]}", flush=True)
        orc = [po.OracleWorld(s, continuous=True, exact_rot=True) for s in ws]
        h = native.StepWorlds(contacts_per_fixture=24)
        for s in ws:
            h.add_scene(s)
        h.finalize()
        for i in range(20):
            h.step(DT, flags=native.WARM | native.SLEEP | native.CCD | native.ORDERED)
            got = h.toi_events()
            for w, o in enumerate(orc):
                o.step(DT)
                label = f"step {i + 1}, {ws[w].name}"
                assert int(got[w]) == o.toi_events(), f"{label}: {int(got[w])} events, the oracle {o.toi_events()}"
                events += o.toi_events()
                m = body_mismatch(h.bodies(w), o.bodies(), o.bodies_def["type"]) or contact_mismatch(h.contacts(w),
                                                                                                       o.contacts())
                assert m is None, f"{label}: {m}"
    assert events > 300
