"""Radiosity solver forms over right-hand-side counts at the edges of the
kernels' column groups and over ragged patch counts, against the same series
in FP64 (numpy) on the links the device returns."""
import ctypes as C

import numpy as np
import pytest

from helpers import Device, P, prepared, prod_samples, prod_tris, u32p
from lighter_amd import _lib, scenes

pytestmark = pytest.mark.gpu

dp = C.POINTER(C.c_double)
BOUNCES = 3
# Positive factors and operands: a product's relative error is at most its
# operands' rounding (2 x half an ulp of the 16-bit type; FP32 forms: the sum
# of up to some hundred terms in FP32), a total's at most BOUNCES times that.
BOUND = {0: 1e-13, 1: BOUNCES * 64 * 2.0 ** -24, 2: BOUNCES * 256 * 2.0 ** -24, 3: BOUNCES * 2 * 2.0 ** -9,
         4: BOUNCES * 2 * 2.0 ** -12, 5: BOUNCES * 256 * 2.0 ** -24, 6: BOUNCES * 256 * 2.0 ** -24,
         7: BOUNCES * 256 * 2.0 ** -24}


@pytest.fixture(scope="module")
def room(lib):
    b = prepared(lib, scenes.room_scene(lm=64, n_boxes=6, wall_tess=4, bounce_count=0))
    pos, nrm, _, rad = prod_samples(lib, b.scene, 1)
    tris = prod_tris(lib, b.scene, 1)
    b.destroy()
    return pos, scenes.normalize_rows_f32(nrm), np.ascontiguousarray(rad[:, 3]), tris


def links(lib, dev, pos, nrm):
    n, nl = len(pos), C.c_size_t(0)
    _lib.check(lib.lgx_RadLinks(dev.h, P(pos), P(nrm), n, C.byref(nl)), lib)
    rowmap, other, fac = np.zeros((n, 2), np.uint32), np.zeros(max(nl.value, 1), np.uint32), np.zeros(max(nl.value, 1), np.float32)
    _lib.check(lib.lgx_RadReadLinks(dev.h, rowmap.ctypes.data_as(u32p), other.ctypes.data_as(u32p), P(fac)), lib)
    F = np.zeros((n, n))
    for i in range(n):
        o, c = rowmap[i]
        F[i, other[o:o + c]] = fac[o:o + c]
    return F + F.T


@pytest.mark.parametrize("n", [1, 257, 1500])
@pytest.mark.parametrize("R", [1, 3, 16, 17, 33, 64, 65, 129, 192])
def test_forms_against_fp64(lib, room, n, R):
    pos, nrm, area, tris = room
    sel = np.sort(np.random.default_rng(n).choice(len(pos), n, replace=False))
    pos, nrm, area = pos[sel].copy(), nrm[sel].copy(), area[sel].copy()
    dev = Device(lib, tris)
    F = links(lib, dev, pos, nrm)
    rng = np.random.default_rng(R)
    diff = rng.uniform(0.2, 0.9, (n, 3)).astype(np.float32)
    E = rng.uniform(0.02, 1.0, (n, R))
    g = rng.uniform(0.1, 1.0, (n, R))
    mul = diff[:, np.arange(R) % 3].astype(np.float64)
    a = area.astype(np.float64)[:, None]
    S, z = [E], E
    for _ in range(BOUNCES):
        z = F @ (z * mul * a)
        S.append(S[-1] + z)
    lam, dalb, y = g.copy(), np.zeros_like(E), g
    for k in range(BOUNCES, 0, -1):
        u = a * (F @ y)
        dalb += u * S[k - 1]
        y = mul * u
        lam = lam + y
    for form, bound in BOUND.items():
        total, t2, l2, d2 = (np.zeros_like(E) for _ in range(4))
        for _ in range(2):  # the second on kept buffers
            _lib.check(lib.lgx_RadSolve(dev.h, E.ctypes.data_as(dp), R, P(diff), P(area), form, BOUNCES, 0,
                                        total.ctypes.data_as(dp), None), lib)
        _lib.check(lib.lgx_RadSolveGrad(dev.h, E.ctypes.data_as(dp), R, P(diff), P(area), form, BOUNCES,
                                        g.ctypes.data_as(dp), t2.ctypes.data_as(dp), l2.ctypes.data_as(dp),
                                        d2.ctypes.data_as(dp), None), lib)
        for name, got, want in (("total", total, S[-1]), ("grad total", t2, S[-1]), ("lam", l2, lam), ("dalb", d2, dalb)):
            err = np.linalg.norm(got - want) / max(np.linalg.norm(want), 1e-30)
            assert err <= 2 * bound, (form, name, err)
    dev.close()
