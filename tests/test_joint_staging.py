"""Joint worlds on both sides of the LDS limits of the island search and of the solve,
and with one to many islands per wave, against the oracle, bit for bit: each alone and
all in one handle, where the same launch serves both sides."""
import numpy as np
import pytest

from dbox_amd import native, scenes
from oracle import pyoracle as po
from tests.helpers import body_mismatch, contact_mismatch

pytestmark = pytest.mark.gpu
DT = 1.0 / 60.0
SIZES = [0, 1, 12, 150, 200, 500, 900]  # debris; solved from LDS up to about 180, searched from LDS up to about 750


def _scattered(n):
    s = scenes.joint_world(n + 1, debris=n)
    r = np.random.default_rng(n)
    d = s.bodies[13:13 + n]  # after the ground and the twelve planks
    d["px"], d["py"] = r.uniform(-29.0, -19.0, n), r.uniform(7.0, 8.0 + n / 40.0, n)
    return s


@pytest.mark.parametrize("warm", [True, False])
@pytest.mark.parametrize("sizes", [[n] for n in SIZES] + [SIZES])
def test_joint_worlds_equal_the_oracle(sizes, warm):
    print(f"case: joint worlds with {sizes} pieces of debris, warm {warm}", flush=True)
    ws = [_scattered(n) for n in sizes]
    orc = [po.OracleWorld(s, continuous=False, warm_starting=warm, exact_rot=True) for s in ws]
    h = native.StepWorlds(contacts_per_fixture=16)
    for s in ws:
        h.add_scene(s)
    h.finalize()
    for i in range(12):
        h.step(DT, flags=native.SLEEP | native.ORDERED | (native.WARM if warm else 0))
        for w, o in enumerate(orc):
            o.step(DT)
            label = f"step {i + 1}, {sizes[w]} pieces"
            m = body_mismatch(h.bodies(w), o.bodies(), o.bodies_def["type"])
            assert m is None, f"{label}: {m}"
            assert h.joints(w).tobytes() == o.joints().tobytes(), f"{label}: joints"
            m = contact_mismatch(h.contacts(w), o.contacts())
            assert m is None, f"{label}: {m}"
