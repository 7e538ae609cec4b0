"""The stand-alone broadphase against the brute-force pair set, bit for bit, at the
edges of its tiles and segments, and in the layouts that load one row with every pair."""
import ctypes as C

import numpy as np
import pytest

from dbox_amd import native
from oracle import pyoracle as po
from tests.test_zz_no_alloc import _Dev, _hip_runtime

pytestmark = pytest.mark.gpu


def _boxes(rng, n, layout):
    side = 1.0 + 1.3 * n ** 0.5
    lo = rng.uniform(0, side, (n, 2))
    sz = rng.uniform(0.05, 2.0, (n, 2))
    if layout == "wall":  # the first and the last proxy overlap everything
        lo[[0, -1]], sz[[0, -1]] = -1.0, side + 4.0
    if layout == "stack":  # every box starts at the same x, equal bounds in y
        lo[:, 0], lo[:, 1] = 3.0, np.arange(n)
        sz[:] = 1.0
    fat = np.concatenate([lo, lo + sz], 1).astype(np.float32)
    if layout == "infinite":
        fat[n // 2] = -np.inf, -np.inf, np.inf, np.inf
    return fat


@pytest.mark.parametrize("layout", ["spread", "wall", "stack", "infinite"])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 63, 64, 65, 255, 256, 257, 511, 513, 1025, 4097, 16384, 16385])
def test_pairs_equal_brute_force(n, layout):
    print(f"case: broadphase {n} proxies, {layout}", flush=True)
    rng = np.random.default_rng(1000 + n)
    fat = _boxes(rng, n, layout)
    h = native.StepWorlds()
    for frac in (1.0, 0.3, 0.0):
        moved = (rng.random(n) < frac).astype(np.uint8)
        got = native.broadphase_pairs(h, fat, moved)
        want = po.brute_force_pairs(fat, moved)
        assert np.array_equal(got, want)
    h.close()


@pytest.mark.parametrize("cap", [0, 16])
def test_no_proxies_give_a_count_of_zero(cap):
    print(f"case: broadphase without proxies, capacity {cap}", flush=True)
    h = native.StepWorlds()
    fat = _boxes(np.random.default_rng(5), 400, "wall")
    assert len(native.broadphase_pairs(h, fat, np.ones(400, np.uint8))) > 700  # its count lay in memory handed out again
    out, n = np.full((max(cap, 1), 2), -7, np.int32), C.c_int32(-1)
    assert h.L.dbx_broadphase_pairs(h.h, None, None, 0, out.ctypes.data, cap, C.byref(n)) == native.DBX_OK
    assert n.value == 0 and (out == -7).all()
    rt = _hip_runtime()
    pairs, count = _Dev(rt, out), _Dev(rt, np.full(1, 55, np.int32))
    assert h.L.dbx_broadphase_pairs_noalloc(h.h, None, None, 0, pairs.ptr, cap, count.ptr) == native.DBX_OK
    h.sync()
    assert count.read()[0] == 0 and (pairs.read() == -7).all()
    for d in (pairs, count):
        d.free()
    h.close()
