"""The workgroup broadphase against the oracle's UpdatePairs, exactly, on both sides of
each of its rules: direct tests or sort and sweep (moved proxies times proxies per
thread), pairs ordered by counting or by the sorting network, more pairs than the LDS
stages, and no moved proxy at all.  The sizes lie around the wave and the workgroup."""
import numpy as np
import pytest

from dbox_amd import native, scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu
DT = 1.0 / 60.0

CASES = {  # bodies, width, height of the container
    "small": [(1, 4.0, 4.0), (2, 4.0, 4.0), (60, 14.0, 30.0), (61, 14.0, 30.0), (62, 14.0, 30.0)],
    "ordinary": [(125, 14.0, 30.0), (253, 20.0, 40.0), (254, 20.0, 40.0)],
    "many pairs": [(40, 4.0, 5.0), (100, 7.0, 7.0), (300, 12.0, 12.0)],
    "large": [(700, 40.0, 60.0), (1100, 50.0, 70.0)],
}


@pytest.mark.parametrize("name", list(CASES))
def test_pairs_equal_the_oracles(name):
    print(f"case: workgroup broadphase, {name}", flush=True)
    ws = [scenes.mixed_container(n, w, h, 7 * n) for n, w, h in CASES[name]]
    still = scenes.mixed_container(90, 14.0, 30.0, 5)  # every proxy moved in the first step, none later
    still.bodies["type"] = scenes.STATIC
    ws.append(still)
    orc = [po.OracleWorld(s, continuous=False, exact_rot=True) for s in ws]
    h = native.StepWorlds(contacts_per_fixture=24)
    for s in ws:
        h.add_scene(s)
    h.finalize()
    seen = []
    for i in range(12):
        h.step(DT, flags=native.WARM | native.SLEEP | native.ORDERED)
        for w, o in enumerate(orc):
            o.step(DT)
            assert np.array_equal(h.pairs(w), o.last_pairs()), f"step {i + 1}, world {w}: pairs"
            seen.append(len(o.last_pairs()))
    print(f"{name}: {min(seen)} to {max(seen)} pairs", flush=True)
    assert min(seen) == 0 and max(seen) > {"small": 10, "many pairs": 1000}.get(name, 100)
