"""The link search over clusters of 64 patches against the all-pairs
enumeration, bit for bit: patch counts at the edges of clusters and
super-clusters, normals of any direction and length, flat, crowded and
far-away patch sets."""
import ctypes as C

import numpy as np
import pytest

from helpers import Device, P
from lighter_amd import _lib

pytestmark = pytest.mark.gpu
u32p = C.POINTER(C.c_uint32)


def links(lib, dev, pos, nrm, mode):
    _lib.check(lib.lgx_SetLinkSearch(dev.h, mode), lib)
    nl = C.c_size_t(0)
    _lib.check(lib.lgx_RadLinks(dev.h, P(pos), P(nrm), len(pos), C.byref(nl)), lib)
    rowmap = np.zeros(2 * len(pos), np.uint32)
    other = np.zeros(max(nl.value, 1), np.uint32)
    fac = np.zeros(max(nl.value, 1), np.float32)
    _lib.check(lib.lgx_RadReadLinks(dev.h, rowmap.ctypes.data_as(u32p), other.ctypes.data_as(u32p), P(fac)), lib)
    return rowmap, other, fac


def patches(kind, n, rng):
    d = rng.normal(size=(n, 3))
    nrm = d / np.linalg.norm(d, axis=1, keepdims=True)
    if kind == "ball":  # crowded: every pair within reach
        pos = rng.uniform(-2, 2, (n, 3))
    elif kind == "far":  # a kilometre from the origin, several linking distances wide
        pos = rng.uniform(-40, 40, (n, 3)) + [1500.0, -900.0, 200.0]
    elif kind == "lengths":  # normals from zero to five metres long
        pos = rng.uniform(-30, 30, (n, 3))
        nrm = nrm * rng.choice([0.0, 0.01, 0.3, 1.0, 5.0], (n, 1))
    elif kind == "planes":  # floor and ceiling, axis-aligned normals, repeated positions
        pos = rng.integers(0, 24, (n, 3)).astype(float)
        pos[:, 2] = np.where(rng.random(n) < 0.5, 0.0, 2.5)
        nrm = np.where(pos[:, 2:3] == 0, [0.0, 0.0, 1.0], [0.0, 0.0, -1.0])
    return pos.astype(np.float32), nrm.astype(np.float32)


@pytest.mark.parametrize("kind", ["ball", "far", "lengths", "planes"])
@pytest.mark.parametrize("n", [2, 63, 64, 65, 1000, 4097])
def test_clusters_find_the_all_pairs_links(lib, kind, n):
    rng = np.random.default_rng(n)
    pos, nrm = patches(kind, n, rng)
    ext = float(np.ptp(pos, axis=0).max()) + 1
    c = pos[rng.integers(0, n, 300)][:, None] + rng.uniform(-0.1, 0.1, (300, 1, 3)) * ext
    tris = (c + rng.uniform(-0.1, 0.1, (300, 3, 3)) * ext).astype(np.float32).reshape(-1, 9)
    dev = Device(lib, tris)
    a, b = links(lib, dev, pos, nrm, 1), links(lib, dev, pos, nrm, 2)
    dev.close()
    for x, y in zip(a, b):
        assert x.shape == y.shape
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
    if n >= 1000:  # only that there is something to compare (an unlinked set leaves one unused entry)
        assert len(a[1]) > 1


@pytest.mark.parametrize("n", [2, 6144, 6145, 20_000])
def test_automatic_choice_and_waves_per_patch(lib, n):
    """Mode 0 on both sides of the count up to which it takes all pairs, and
    the clusters with 16, 8 and 2 waves to a patch."""
    rng = np.random.default_rng(n)
    pos, nrm = patches("planes", n, rng)
    pos[:, :2] += rng.uniform(0.0, 0.9, (n, 2)).astype(np.float32)
    tris = rng.uniform(0.0, 24.0, (200, 9)).astype(np.float32)
    tris[:, 2::3] *= 0.1
    dev = Device(lib, tris)
    a, b, c = (links(lib, dev, pos, nrm, m) for m in (1, 0, 2))
    dev.close()
    for x, y, z in zip(a, b, c):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
        assert np.array_equal(x.view(np.uint32), z.view(np.uint32))
    assert n == 2 or len(a[1]) > 1000


@pytest.mark.parametrize("n", [1500, 9000, 40_000])
def test_kept_candidates_are_the_all_pairs_ones(lib, n):
    """With counting on, the clusters' candidates (16, 4 and 1 waves to a
    patch) are those of all pairs: as many, and the canonical walk of each
    visits as much in sum and finds the links that were kept."""
    rng = np.random.default_rng(n)
    pos, nrm = patches("far", n, rng)
    tris = (pos[rng.integers(0, n, 400), None] + rng.uniform(-4, 4, (400, 3, 3))).astype(np.float32).reshape(-1, 9)
    dev = Device(lib, tris)
    out = []
    for mode in (1, 2):
        _lib.check(lib.lgx_SetCounting(dev.h, 1), lib)
        found = len(links(lib, dev, pos, nrm, mode)[1])
        _lib.check(lib.lgx_SetCounting(dev.h, 0), lib)
        c = (C.c_uint64 * 5)()
        _lib.check(lib.lgx_ReferenceCountsLinks(dev.h, P(tris), len(tris), c), lib)
        assert c[3] == 0 and c[4] == found and c[2] > found > 50
        out.append(list(c))
    dev.close()
    assert out[0] == out[1]


@pytest.mark.parametrize("run", [1, 37, 500])
def test_runs_of_cluster_pairs(lib, run):
    """A search that takes its pairs of clusters in many runs (one first
    cluster each, a few, some more) against one run: links, factors and
    the candidates kept with counting on."""
    n = 9000
    rng = np.random.default_rng(run)
    pos, nrm = patches("far", n, rng)
    tris = (pos[rng.integers(0, n, 400), None] + rng.uniform(-4, 4, (400, 3, 3))).astype(np.float32).reshape(-1, 9)
    dev = Device(lib, tris)
    out = []
    for pairs in (0, run):
        _lib.check(lib.lgx_SetLinkRunPairs(dev.h, pairs), lib)
        got = links(lib, dev, pos, nrm, 2)
        _lib.check(lib.lgx_SetCounting(dev.h, 1), lib)
        links(lib, dev, pos, nrm, 2)
        _lib.check(lib.lgx_SetCounting(dev.h, 0), lib)
        c = (C.c_uint64 * 5)()
        _lib.check(lib.lgx_ReferenceCountsLinks(dev.h, P(tris), len(tris), c), lib)
        out.append((*got, np.array(list(c), np.uint64).view(np.uint32)))
    dev.close()
    assert len(out[0][1]) > 1000
    for x, y in zip(*out):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
