"""The network's entry points over row counts around their tiles (16 and 32 rows) and their
chunk (65,536 rows): a row's outputs do not depend on the rows around it, and gradients
and loss equal the reference's within the bounds of its bf16 products."""
import numpy as np
import pytest

from dbox_amd import native, scenes
from oracle import mlp_ref
from tests.test_gpu_mlp import _norm

pytestmark = pytest.mark.gpu
ROWS = [1, 2, 15, 16, 17, 31, 32, 33, 255, 4099, 65535, 65536, 65537, 70001]


def _net(rng):
    p, norm = mlp_ref.he_init(5), _norm(rng)
    h = native.StepWorlds()
    h.mlp_set(p, norm)
    return h, p, norm


def test_forward_rows_are_independent():
    rng = np.random.default_rng(11)
    h, p, norm = _net(rng)
    x = rng.normal(0, 2, (max(ROWS), 14)).astype(np.float32)
    ref = mlp_ref.forward(p, norm, x[:4099])["out"]
    first = h.mlp_forward(x[:4099])
    assert np.abs(first - ref).max() < 2e-2 * np.abs(ref).max()
    for n in ROWS:
        print(f"case: forward, {n} rows", flush=True)
        y = h.mlp_forward(x[:n])
        assert y.shape == (n, 2) and y[:4099].tobytes() == first[:n].tobytes()
        k = min(n, 20)
        assert y[n - k:].tobytes() == h.mlp_forward(x[n - k:n]).tobytes()


def test_gradients_over_chunks():
    rng = np.random.default_rng(12)
    h, p, norm = _net(rng)
    x = rng.normal(0, 1.5, (max(ROWS), 14)).astype(np.float32)
    t = rng.normal(0, 1, (max(ROWS), 2)).astype(np.float32)
    for n in ROWS:
        print(f"case: gradients, {n} rows", flush=True)
        g, loss = h.mlp_gradients(x[:n], t[:n])
        again, loss2 = h.mlp_gradients(x[:n], t[:n])
        gref, lref = mlp_ref.gradients(p, norm, x[:n], t[:n])
        assert abs(loss - lref) < 1e-3 * max(1.0, lref), (n, loss, lref)
        # sums in another order: float32 rounding of n terms at most
        assert np.abs(g - again).max() <= 1e-5 * np.abs(g).max() and abs(loss - loss2) <= 1e-5 * loss
        assert np.linalg.norm(g - gref) <= 1e-2 * np.linalg.norm(gref) + 1e-7, n


def test_body_writes_and_rows_share_the_staging_memory():
    rng = np.random.default_rng(13)
    h, _, _ = _net(rng)
    h.add_scene(scenes.mixed_container(60, 14.0, 30.0, 4))
    h.finalize()
    x, t = rng.normal(0, 2, (3000, 14)).astype(np.float32), rng.normal(0, 1, (3000, 2)).astype(np.float32)
    y, (g, _) = h.mlp_forward(x), h.mlp_gradients(x, t)
    for i in range(5):
        s = h.bodies()
        s["vx"][1:] = 0.25 * (i + 1)
        h.write_bodies(0, s)
        assert h.mlp_forward(x).tobytes() == y.tobytes()
        h.write_bodies(0, s)
        assert np.abs(h.mlp_gradients(x, t)[0] - g).max() <= 1e-5 * np.abs(g).max()
        assert np.array_equal(h.bodies()["vx"], s["vx"])
