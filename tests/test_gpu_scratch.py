"""Queries and link searches of changing size on one device, whose scratch
blocks one call takes over from another, against a new device for each."""

import ctypes as C

import numpy as np
import pytest

from helpers import Device, P
from hipmem import hip
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


def test_failed_allocation_gives_spare_blocks_back(lib):
    """The scratch that one device keeps (1.6 GB after a query of 100 M
    points) is there for a call of another that finds no memory: it is given
    back before that call fails (a dense matrix of 360 GB here)."""
    h = hip()
    h.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]

    def free_memory():
        free, total = C.c_size_t(0), C.c_size_t(0)
        assert h.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        assert total.value < 360e9
        return free.value

    rng = np.random.default_rng(12)
    tris = rng.uniform(-3, 3, (20, 9)).astype(np.float32)

    def dense_solve(n):
        dev = Device(lib, tris)
        pos = np.zeros((n, 3), np.float32)
        pos[:, :2] = np.stack(np.divmod(np.arange(n), 1000), 1)
        nrm = np.tile(np.array([0, 0, 1], np.float32), (n, 1))
        nl = C.c_size_t(0)
        _lib.check(lib.lgx_RadLinks(dev.h, P(pos), P(nrm), n, C.byref(nl)), lib)
        E, diff, area = np.ones((n, 1)), np.ones((n, 3), np.float32), np.ones(n, np.float32)
        dp = C.POINTER(C.c_double)
        ok = lib.lgx_RadSolve(dev.h, E.ctypes.data_as(dp), 1, P(diff), P(area), 2, 1, 0,
                              np.zeros_like(E).ctypes.data_as(dp), None)
        dev.close()
        return ok

    assert dense_solve(1000) == 1
    dev = Device(lib, tris)
    dev.distance(np.zeros((1000, 3), np.float32))
    before = free_memory()
    dev.distance(np.zeros((100_000_000, 3), np.float32))
    assert before - free_memory() > 1.5e9  # kept
    assert dense_solve(300_000) == 0
    assert "allocating" in _lib.last_error(lib)
    assert before - free_memory() < 0.5e9
    dev.close()
