"""The coloured mode against the oracle's colour order, bit for bit, for worlds around the
wave and the workgroup sizes and on both sides of the LDS limit of the solve; a residual
that never ends the iterations gives the fixed count's result."""
import pytest

from dbox_amd import native, scenes
from oracle import pyoracle as po
from tests.helpers import body_mismatch, contact_mismatch

pytestmark = pytest.mark.gpu
DT = 1.0 / 60.0


def _worlds(dense):
    w = 1.0 if dense else 2.0
    return [scenes.mixed_container(n, w * (2.0 + n ** 0.5), w * (2.0 + n ** 0.5), n)
            for n in (1, 2, 7, 31, 32, 61, 64, 65, 127, 160, 260, 420, 700)] + [scenes.pyramid(12, seed=4)]


@pytest.mark.parametrize("dense", [False, True])
@pytest.mark.parametrize("warm,residual", [(True, False), (False, False), (True, True)])
def test_coloured_worlds_equal_the_colour_order_oracle(dense, warm, residual):
    print(f"case: coloured worlds, dense {dense}, warm {warm}, residual {residual}", flush=True)
    ws = _worlds(dense)
    orc = [po.OracleWorld(s, warm_starting=warm, colour_order=True, exact_rot=True) for s in ws]
    h = native.StepWorlds(contacts_per_fixture=16)
    for s in ws:
        h.add_scene(s)
    h.finalize()
    if residual:
        h.set_residual(-1.0, 8)
    flags = native.SLEEP | (native.WARM if warm else 0) | (native.RESIDUAL if residual else 0)
    for i in range(20):
        h.step(DT, 8, 3, flags)
        for w, o in enumerate(orc):
            o.step(DT)
            if i % 5 == 4:
                m = body_mismatch(h.bodies(w), o.bodies(), o.bodies_def["type"]) or contact_mismatch(h.contacts(w),
                                                                                                       o.contacts())
                assert m is None, f"step {i + 1}, world {w}: {m}"


@pytest.mark.parametrize("fill", [0, 1100])  # in one launch, and a launch per phase
def test_iterations_reported_without_a_constraint(fill):
    print(f"case: iteration counts of coloured worlds in free fall, {fill} more worlds", flush=True)
    h = native.StepWorlds()
    for s in [scenes.hello_world(), scenes.pyramid(3)] + [scenes.hello_world()] * fill:
        h.add_scene(s)
    h.finalize()
    h.step(DT, 5, 3, native.WARM, n=1)
    it, _ = h.solver_stats()
    assert len(h.contacts(0)) == 0 and it[0] == 5 and it[1] == 5 and h.residuals()[0] == -1.0
    for tol, most, want in ((-1.0, 7, 7), (0.0, 7, 1), (1e-3, 1, 1), (1e-3, 30, 1)):
        h.set_residual(tol, most)
        h.step(DT, 8, 3, native.WARM | native.RESIDUAL, n=1)
        it, _ = h.solver_stats()
        assert it[0] == want and h.residuals()[0] == 0.0, (tol, most, it[0])
        assert tol >= 0.0 or it[1] == most
    h.close()
