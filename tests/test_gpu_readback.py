"""Read-backs and body writes through pinned memory: writes back to back, and so many that
they fill the staging memory several times over, reads that outgrow it, and short output buffers."""
import ctypes as C

import numpy as np
import pytest

from dbox_amd import native, scenes

pytestmark = pytest.mark.gpu
FLAGS = native.WARM | native.SLEEP | native.ORDERED | native.CCD


def _handle(ws):
    h = native.StepWorlds()
    for s in ws:
        h.add_scene(s)
    h.finalize()
    return h


@pytest.mark.parametrize("forces", [False, True])
def test_writes_back_to_back_equal_writes_one_at_a_time(forces):
    print(f"case: 300 worlds written back to back, forces {forces}", flush=True)
    ws = [scenes.pyramid(5, seed=w) for w in range(300)]
    a, b = _handle(ws), _handle(ws)
    rng = np.random.default_rng(3)
    for w in range(300):
        st = a.bodies(w)
        st["vx"][1:] += rng.uniform(-1, 1, len(st) - 1).astype(np.float32)
        st["flags"][1] &= ~2  # asleep
        f = rng.uniform(-5, 5, (len(st), 3)).astype(np.float32) if forces else None
        for h in (a, b):
            h.write_bodies(w, st, f)
        b.sync()
        if w % 37 == 0:
            got = a.bodies(w)
            assert got.tobytes() == st.tobytes()
    for h in (a, b):
        h.step(flags=FLAGS, n=3)
        h.sync()
    for w in range(0, 300, 7):
        assert a.bodies(w).tobytes() == b.bodies(w).tobytes()
    a.close()
    b.close()


def test_writes_without_a_read_between_them_wrap_and_grow_the_staging_memory():
    # 300 small worlds and one whose states alone outgrow the first 256 KiB, four times over
    ws = [scenes.pyramid(5, seed=w) for w in range(300)] + [scenes.mixed_container(5000, 100.0, 120.0, 3)]
    order = list(range(150)) + [300] + list(range(150, 300))
    a, b = _handle(ws), _handle(ws)
    states = [b.bodies(w) for w in range(len(ws))]
    print(f"case: {4 * sum(s.nbytes for s in states) >> 10} KiB of body states written without a read", flush=True)
    rng = np.random.default_rng(4)
    for k in range(4):
        for w in order:
            st = states[w]
            st["vx"][1:] = rng.uniform(-1, 1, len(st) - 1).astype(np.float32)
            f = rng.uniform(-5, 5, (len(st), 3)).astype(np.float32) if (w + k) % 3 == 0 else None
            a.write_bodies(w, st, f)
            b.write_bodies(w, st, f)
            b.sync()
            st["vx"][1:] = 99.0  # the calls have copied their input
    for h in (a, b):
        h.step(flags=FLAGS & ~native.CCD, n=2)
        h.sync()
    for w in range(len(ws)):
        assert a.bodies(w).tobytes() == b.bodies(w).tobytes(), w
    a.close()
    b.close()


def test_bad_states_change_nothing():
    h = _handle([scenes.pyramid(4)])
    st = h.bodies()
    bad = st.copy()
    bad["px"][2] = np.nan
    with pytest.raises(native.DbxError):
        h.write_bodies(0, bad)
    with pytest.raises(native.DbxError):
        h.write_bodies(0, st, np.full((len(st), 3), np.inf, np.float32))
    assert h.bodies().tobytes() == st.tobytes()
    h.close()


def test_reads_that_outgrow_the_pinned_memory():
    print("case: 4000-body container read small, large and truncated", flush=True)
    h = _handle([scenes.mixed_container(4000, 90.0, 60.0, 5), scenes.hello_world()])
    h.step(flags=FLAGS & ~native.CCD, n=40)  # the continuous pass changes touching flags after the count
    small = h.contacts(1)
    c = h.contacts(0)
    assert len(c) == h.info(0)[2] > 3200 and len(small) == h.info(1)[2]
    fixtures = h.fixture_counts[0]
    assert (c["fixture_a"] >= 0).all() and (c["fixture_b"] < fixtures).all()
    assert np.count_nonzero(c["flags"] & 2) == h.info(0)[3]
    assert c.tobytes() == h.contacts(0).tobytes()
    n = C.c_int32()
    part = np.zeros(10, native.CONTACT_DTYPE)
    assert h.L.dbx_read_contacts(h.h, 0, part.ctypes.data_as(C.c_void_p), 10, C.byref(n)) == native.DBX_OK
    assert n.value == len(c) and part.tobytes() == c[:10].tobytes()
    ev = h.events(0)
    assert len(ev) > 1000 and ev.tobytes() == h.events(0).tobytes()
    assert h.L.dbx_read_events(h.h, 0, None, 0, C.byref(n)) == native.DBX_OK and n.value == len(ev)
    short = np.zeros(5, native.EVENT_DTYPE)
    st = h.L.dbx_read_events(h.h, 0, short.ctypes.data_as(C.c_void_p), 5, C.byref(n))
    assert st == native.DBX_E_CAPACITY and n.value == len(ev) and not short.view(np.uint8).any()
    assert len(h.bodies(0)) == 4001
    h.close()


def test_reads_of_a_world_that_is_not_there_are_refused_by_the_library():
    h = _handle([scenes.pyramid(3)])
    for world in (1, 7, -1):
        for read in (h.contacts, h.events):
            with pytest.raises(native.DbxError):
                read(world)
    assert len(h.contacts(0)) == 0 and len(h.events(0)) == 0
    h.close()
