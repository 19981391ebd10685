"""Face-pair and grid weights of small awkward meshes against the oracle, bit for bit: pairs that
share one, two or three vertices, duplicated and nearly coincident triangles, pair counts around the
seven pairs and the 64 pairs a wave takes at once, and time steps so short that the exponentials
leave the range of the shared-reciprocal divisions (|Im k| r > 600)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
N, H, C = 16, 0.01, 343.0


def _mesh(name):
    rng = np.random.default_rng(3)
    mid = N * H / 2
    if name.startswith("soup"):  # n separate triangles around the centre: n * n regular pairs
        n = int(name[4:])
        c = mid + rng.uniform(-0.015, 0.015, (n, 1, 3))
        v = (c + rng.uniform(-0.004, 0.004, (n, 3, 3))).reshape(-1, 3)
        return v, np.arange(3 * n).reshape(n, 3)
    p = mid + 0.008 * rng.standard_normal((6, 3))
    if name == "corner":
        return p, np.array([[0, 1, 2], [2, 3, 4]])
    if name == "edge":
        return p, np.array([[0, 1, 2], [1, 2, 3], [3, 4, 5]])
    if name == "duplicate":  # the same triangle again, turned and flipped
        return p, np.array([[0, 1, 2], [1, 2, 0], [0, 2, 1], [3, 4, 5]])
    q = np.concatenate([p[:3], p[:3] + 1e-5, p[3:]])  # unconnected, centroids closer than 0.1 h
    return q, np.array([[0, 1, 2], [3, 4, 5], [6, 7, 8]])


@pytest.mark.parametrize("dt_scale", [1.0, 0.02])
@pytest.mark.parametrize("name", ["soup1", "soup2", "soup3", "soup8", "soup23", "corner", "edge", "duplicate",
                                  "coincident", "sphere"])
def test_weights_bitexact(amd, oracle_mod, scenes_mod, name, dt_scale):
    _compare(amd, oracle_mod, scenes_mod, name, dt_scale, 1.0)


# cells of 1e-15 and 2e4: distances on both sides of either end of the shared reciprocals' range
@pytest.mark.parametrize("scale", [1e-13, 2e6])
@pytest.mark.parametrize("name", ["soup8", "duplicate", "sphere"])
def test_weights_bitexact_at_scale(amd, oracle_mod, scenes_mod, name, scale):
    _compare(amd, oracle_mod, scenes_mod, name, 1.0, scale)


def _compare(amd, oracle_mod, scenes_mod, name, dt_scale, scale):
    if name == "sphere":
        v, f = scenes_mod.icosphere(1, 0.03, (N * H / 2,) * 3)
    else:
        v, f = _mesh(name)
    v, f = (np.asarray(v, np.float64) * scale).astype(np.float32), f.astype(np.int32)
    h = H * scale
    dt = np.float32(dt_scale * h / (np.sqrt(3.0) * C))
    g = amd.PPPMSolver(N, h, dt, (0, 0, 0), 0, 0.83, C)
    o = oracle_mod.Oracle(N, h, dt, (0, 0, 0), C, 0.83, oracle_mod.FP64)
    g.set_mesh(v, f)
    o.set_mesh(v, f)
    sa, na, ra = g.get_face_weights()
    sb, nb, rb = o.face_weights()
    assert np.array_equal(sa, sb) and np.array_equal(na, nb)
    assert ra.tobytes() == rb.tobytes()
    assert g.get_grid_weights().tobytes() == o.grid_weights().tobytes()
