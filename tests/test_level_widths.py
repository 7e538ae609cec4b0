"""Level sweeps over levels of 1 to 300 constraints, around the 32 lane pairs and the 64
lanes of a wave, with one- and two-point contacts mixed, against the oracle, bit for bit,
in every form of the sweeps: one wave, overlapped, to a residual, colours."""
import numpy as np
import pytest

from dbox_amd import native, scenes
from oracle import pyoracle as po
from tests.helpers import body_mismatch, contact_mismatch

pytestmark = pytest.mark.gpu
DT = 1.0 / 60.0
WIDTHS = [1, 2, 31, 32, 33, 63, 64, 65, 97, 128, 129, 300]


def _row(n):
    """n bodies side by side on the ground, every third a ball, every fourth with a box on top."""
    top = [k for k in range(n) if k % 4 == 1]
    b = scenes.body_defs(1 + n + len(top))
    b[0]["type"] = scenes.STATIC
    b[1:]["type"] = scenes.DYNAMIC
    x = 1.5 * (np.arange(n) - 0.5 * n)
    b[1:1 + n]["px"], b[1:1 + n]["py"] = x, 0.52
    b[1:1 + n]["vx"] = np.linspace(-1.0, 1.0, n)
    b[1 + n:]["px"], b[1 + n:]["py"] = x[top] + 0.1, 1.5
    f = scenes.fixture_defs(len(b))
    f["body"] = np.arange(len(b))
    scenes._edge(f[0], 0, -2.0 * n - 5.0, 0.0, 2.0 * n + 5.0, 0.0, 0.6)
    f[1:]["density"], f[1:]["friction"], f[1:]["shape"] = 1.0, 0.4, scenes.SHAPE_BOX
    f[1:]["p"][:, :2] = 0.5
    ball = np.zeros(len(b), bool)
    ball[1:1 + n:3] = True
    f["shape"][ball], f["radius"][ball], f["p"][ball] = scenes.SHAPE_CIRCLE, 0.5, 0.0
    return scenes.Scene(b, f, name=f"row{n}")


@pytest.mark.parametrize("form", ["default", "sequential", "always", "residual", "residual always", "coloured"])
@pytest.mark.parametrize("warm", [True, False])
def test_levels_of_every_width_equal_the_oracle(form, warm, monkeypatch):
    print(f"case: level widths, {form}, warm {warm}", flush=True)
    for var, on in (("DBX_SWEEPS_SEQUENTIAL", form == "sequential"), ("DBX_SWEEPS_OVERLAP_ALWAYS", "always" in form)):
        monkeypatch.setenv(var, "1") if on else monkeypatch.delenv(var, raising=False)
    ws = [_row(n) for n in WIDTHS]
    orc = [po.OracleWorld(s, warm_starting=warm, colour_order=form == "coloured", exact_rot=True) for s in ws]
    h = native.StepWorlds(contacts_per_fixture=16)
    for s in ws:
        h.add_scene(s)
    h.finalize()
    flags = native.SLEEP | (native.WARM if warm else 0) | (0 if form == "coloured" else native.ORDERED)
    if "residual" in form:
        h.set_residual(-1.0, 8)  # never ends early: the fixed count's result
        flags |= native.RESIDUAL
    for i in range(30):
        h.step(DT, 8, 3, flags)
        for w, o in enumerate(orc):
            o.step(DT)
            if i % 6 == 5:
                m = body_mismatch(h.bodies(w), o.bodies(), o.bodies_def["type"]) or contact_mismatch(h.contacts(w),
                                                                                                       o.contacts())
                assert m is None, f"step {i + 1}, {ws[w].name}: {m}"
    widest = max(int(np.bincount(h.schedule(w)[:, 3]).max()) for w in range(len(ws)))
    assert widest >= 300
