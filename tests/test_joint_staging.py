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


# joint worlds beside others in the same tier: (other worlds, their bodies, debris of the joint
# worlds), so that each form of the solve is chosen: together with LDS for the joint worlds'
# state, together without it, a launch each
MIXES = {
    "few": (300, 20, [0, 12, 40]),
    "larger LDS for all": (280, 200, [150, 170]),
    "too many rounds for that": (2000, 200, [150, 170]),
    "many joint worlds": (1000, 60, [96 + k % 4 for k in range(700)]),
}


@pytest.mark.parametrize("mode", ["exact", "coloured", "residual"])
@pytest.mark.parametrize("mix", list(MIXES))
def test_joint_worlds_among_others_equal_them_alone(mix, mode):
    print(f"case: joint worlds in a mixed tier, {mix}, {mode}", flush=True)
    others, size, debris = MIXES[mix]
    box = [scenes.mixed_container(size, 3.0 + size ** 0.5, 6.0 + 2.0 * size ** 0.5, k) for k in range(4)]
    joint = {n: _scattered(n) for n in debris}
    ws = [joint[n] for n in debris] + [box[k % 4] for k in range(others)]
    flags = native.WARM | native.SLEEP | {"exact": native.ORDERED, "coloured": 0,
                                          "residual": native.ORDERED | native.RESIDUAL}[mode]

    def run(ws):
        h = native.StepWorlds(contacts_per_fixture=16)
        for s in ws:
            h.add_scene(s)
        h.finalize()
        h.set_residual(1e-2, 20)
        h.step(DT, 8, 3, flags, n=15)
        h.sync()
        return h

    mixed = run(ws)
    for w in [*range(0, len(debris), max(1, len(debris) // 8)), *range(len(debris), len(debris) + 4)]:
        alone = run([ws[w]])
        for read in ("bodies", "contacts", "joints"):
            assert getattr(mixed, read)(w).tobytes() == getattr(alone, read)(0).tobytes(), f"world {w}: {read}"
        assert mixed.solver_stats()[0][w] == alone.solver_stats()[0][0] and mixed.residuals()[w] == alone.residuals()[0]
        alone.close()
    mixed.close()


# joint worlds alone, as many as each form of their launch is chosen for: state in LDS, from
# global memory on four, two and one wave
@pytest.mark.parametrize("worlds,debris", [(300, 60), (512, 100), (700, 100), (1500, 40)])
def test_many_joint_worlds_equal_them_alone(worlds, debris):
    print(f"case: {worlds} joint worlds with {debris} pieces of debris", flush=True)
    kinds = [_scattered(debris + k) for k in range(4)]
    hs = []
    for ws in [[kinds[k % 4] for k in range(worlds)]] + [[k] for k in kinds]:
        h = native.StepWorlds(contacts_per_fixture=16)
        for s in ws:
            h.add_scene(s)
        h.finalize()
        h.step(DT, 8, 3, native.WARM | native.SLEEP | native.ORDERED, n=12)
        h.sync()
        hs.append(h)
    for w in [0, 1, 2, 3, worlds - 4, worlds - 3, worlds - 2, worlds - 1]:
        for read in ("bodies", "contacts", "joints"):
            assert getattr(hs[0], read)(w).tobytes() == getattr(hs[1 + w % 4], read)(0).tobytes(), (w, read)
    for h in hs:
        h.close()
