"""A world too big for one workgroup's LDS: its islands' velocity sweeps overlapped on several
waves, with the impulses in global memory, against the sweeps one after the other, bit
for bit."""
import pytest

from dbox_amd import native, scenes
from tests.test_sweep_waves import _handles, _same, _step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vel,pos,warm", [(8, 3, True), (8, 3, False), (1, 1, True), (2, 3, False), (21, 3, True)])
def test_overlapped_sweeps_of_a_big_world_equal_sequential(vel, pos, warm, monkeypatch):
    print(f"case: big world, {vel} / {pos} iterations, warm {warm}", flush=True)
    hs = _handles([scenes.mixed_container(6000, 100.0, 120.0, 3)])
    flags = native.SLEEP | native.ORDERED | (native.WARM if warm else 0)
    for i in range(60):
        _step(hs, monkeypatch, vel, pos, flags)
        if i % 15 == 14:
            _same(hs, f"step {i + 1}")
    sched = hs["sequential"].schedule(0)
    assert len(sched) > 2000  # a pile with islands of many levels
