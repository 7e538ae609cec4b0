"""The workgroup width that a tier gets by default, and that results do not depend on it:
worlds around the rule's body limit, one bigger than a workgroup's LDS, and a tier with
more worlds than the device has compute units, in both solver modes."""
import pytest

from dbox_amd import native, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ordered", [True, False])
@pytest.mark.parametrize("name", ["small", "large", "big", "many"])
def test_default_width_keeps_results(name, ordered):
    print(f"case: default workgroup width, {name}, ordered {ordered}", flush=True)
    box = lambda n, k: scenes.mixed_container(n, 3.0 + n ** 0.5, 6.0 + 2.0 * n ** 0.5, k)
    ws = {"small": [box(127, 1), box(60, 2)], "large": [box(128, 1), box(700, 2), box(20, 3)],
          "big": [box(7000, 4), box(100, 5)], "many": [box(140, k % 7) for k in range(600)]}[name]
    flags = native.WARM | native.SLEEP | native.CCD | (native.ORDERED if ordered else 0)
    hs = [native.StepWorlds(block_size=b) for b in (0, 256)]
    for h in hs:
        for s in ws:
            h.add_scene(s)
        h.finalize()
        h.step(1.0 / 60.0, 8, 3, flags, n=25)
        h.sync()
    rows, _ = hs[0].tiers()
    assert set(hs[1].tiers()[0][:, 3]) == {256}
    assert rows[0][3] == (1024 if name == "large" else 256), rows
    for w in range(0, len(ws), 17 if name == "many" else 1):
        for read in ("bodies", "contacts", "pairs"):
            assert getattr(hs[0], read)(w).tobytes() == getattr(hs[1], read)(w).tobytes(), (w, read)


def test_autotuner_leaves_one_launch_tiers_alone():
    box = lambda n, k: scenes.mixed_container(n, 3.0 + n ** 0.5, 6.0 + 2.0 * n ** 0.5, k)
    flags = native.WARM | native.SLEEP | native.CCD | native.ORDERED
    # only one-launch tiers, and one beside a tier with a width to tune
    for ws, tuned in (([box(100, 1), box(20, 2)], 0), ([box(700, 3), box(20, 4)], 1)):
        print(f"case: autotuner over {[len(s.bodies) for s in ws]} bodies", flush=True)
        hs = [native.StepWorlds(), native.StepWorlds()]
        for h in hs:
            for s in ws:
                h.add_scene(s)
            h.finalize()
        rows, _ = hs[0].tiers()
        for width in (64, 512, 1024, 128, 64, 1024):
            hs[0].set_tier_blocks([width] * len(rows))
            hs[0].autotune(1)
            for h in hs:
                h.step(1.0 / 60.0, 8, 3, flags, n=5)
                h.sync()
            assert set(hs[0].tiers()[0][tuned:, 3]) == {width}
        for w in range(len(ws)):
            assert hs[0].bodies(w).tobytes() == hs[1].bodies(w).tobytes()
        for h in hs:
            h.close()
