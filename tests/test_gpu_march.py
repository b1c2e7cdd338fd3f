"""Soft-shadow marches: a wave for each march (small launches, and the long
marches that a lane hands over) against marches kept on lanes.  Both answer
every distance query with the minimum of the same triangle distances, so
factors and step counts are equal bit for bit."""
import numpy as np
import pytest

from helpers import Device

pytestmark = pytest.mark.gpu

N = 3001  # queries; repeated, a launch exceeds the size up to which every march takes a wave
COPIES = 50


def soup(kind, rng):
    if kind == "crowd":  # far more than a wave's lanes of triangles in reach of any point
        c = rng.uniform(-0.4, 0.4, (6000, 1, 3))
        return (c + rng.uniform(-0.05, 0.05, (6000, 3, 3))), 0.6
    if kind == "walls":  # long faces that marches creep along
        t = []
        for k in range(40):
            o = rng.uniform(-6, 6, 3)
            o[k % 2] = np.round(o[k % 2])
            d = np.eye(3) * rng.uniform(3, 9)
            u, v = d[(k + 1) % 2], d[2]
            t += [[o, o + u, o + u + v], [o, o + u + v, o + v]]
        return np.array(t), 6.0
    if kind == "far":  # large coordinates: margins and cells at a kilometre
        c = rng.uniform(-30, 30, (3000, 1, 3)) + [[[900.0, -1200.0, 40.0]]]
        return (c + rng.uniform(-1.5, 1.5, (3000, 3, 3))), 30.0
    return np.zeros((0, 3, 3)), 3.0  # nothing to hit


@pytest.mark.parametrize("kind", ["crowd", "walls", "far", "empty"])
def test_wave_and_lane_marches_agree(lib, kind):
    dev, a, b, k = workload(lib, kind)
    one, steps = dev.shadow(a, b, k)
    many, steps2 = dev.shadow(np.tile(a, (COPIES, 1)), np.tile(b, (COPIES, 1)), np.tile(k, COPIES))
    dev.close()
    many, steps2 = many.reshape(COPIES, N), steps2.reshape(COPIES, N)
    same = (many.view(np.uint32) == one.view(np.uint32)).all(0) & (steps2 == steps).all(0)
    assert same.all(), (kind, np.flatnonzero(~same)[:5], one[~same][:5], many[0][~same][:5])
    if kind == "walls":
        assert steps.max() > 128  # some were handed over


def test_more_long_marches_than_the_list_holds(lib):
    """A launch whose every march is long: more of them reach the limit than
    the list of long marches takes (524,288)."""
    dev, a, b, k = workload(lib, "walls")
    one, steps = dev.shadow(a, b, k)
    at = np.flatnonzero(steps >= 112)
    assert len(at) >= 8
    at = np.resize(at, 1_500_000)
    many, steps2 = dev.shadow(a[at], b[at], k[at])
    dev.close()
    assert np.array_equal(many.view(np.uint32), one[at].view(np.uint32))
    assert np.array_equal(steps2, steps[at])


def workload(lib, kind):
    """The device and N marches on it: from, to, k."""
    rng = np.random.default_rng(len(kind))
    tris, ext = soup(kind, rng)
    tris = tris.astype(np.float32).reshape(-1, 9)
    mid = np.array([900.0, -1200.0, 40.0]) if kind == "far" else np.zeros(3)
    a = (mid + rng.uniform(-ext, ext, (N, 3))).astype(np.float32)
    b = (mid + rng.uniform(-ext, ext, (N, 3))).astype(np.float32)
    if len(tris):  # a third start on a face, 5 mm off, and run along it
        n = N // 3
        t = tris[rng.integers(0, len(tris), n)].reshape(n, 3, 3).astype(np.float64)
        w = rng.dirichlet([1, 1, 1], n)
        nrm = np.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0])
        nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
        p = (t * w[:, :, None]).sum(1)
        a[:n] = p + 0.005 * nrm
        b[:n] = p + (t[:, 1] - t[:, 0]) * rng.uniform(1, 4, (n, 1)) + 0.02 * nrm
    b[-1] = a[-1]
    k = rng.choice([0.0, -0.1, 1e-3, 0.05, 0.5, 3.0], N).astype(np.float32)
    return Device(lib, tris), a, b, k
