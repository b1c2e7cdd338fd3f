"""Queries and link searches of changing size on one device, whose scratch
blocks one call takes over from another, against a new device for each."""

import ctypes as C

import numpy as np
import pytest

from helpers import Device, P
from lighter_amd import _lib

pytestmark = pytest.mark.gpu


def _links(lib, dev, pos, nrm):
    nl = C.c_size_t(0)
    _lib.check(lib.lgx_RadLinks(dev.h, P(pos), P(nrm), len(pos), C.byref(nl)), lib)
    rowmap = np.zeros(2 * len(pos), np.uint32)
    other = np.zeros(nl.value, np.uint32)
    fac = np.zeros(nl.value, np.float32)
    u32p = C.POINTER(C.c_uint32)
    _lib.check(lib.lgx_RadReadLinks(dev.h, rowmap.ctypes.data_as(u32p), other.ctypes.data_as(u32p), P(fac)), lib)
    return rowmap, other, fac


def test_scratch_passes_between_calls(lib):
    rng = np.random.default_rng(11)
    c = rng.uniform(-3, 3, (200, 1, 3))
    tris = (c + rng.uniform(-0.5, 0.5, (200, 3, 3))).astype(np.float32).reshape(-1, 9)
    dev = Device(lib, tris)
    for n in (4000, 3, 1025, 700, 4001, 64, 2500):
        a = rng.uniform(-3, 3, (n, 3)).astype(np.float32)
        b = rng.uniform(-3, 3, (n, 3)).astype(np.float32)
        k = rng.uniform(0, 1, n).astype(np.float32)
        nrm = rng.normal(size=(n, 3)).astype(np.float32)
        nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
        one = Device(lib, tris)
        out = [[d.distance(a), *d.shadow(a, b, k), *_links(lib, d, a, nrm), d.distance(b)] for d in (dev, one)]
        one.close()
        for x, y in zip(*out):
            assert np.array_equal(x.view(np.uint32), y.view(np.uint32)), n
    dev.close()
