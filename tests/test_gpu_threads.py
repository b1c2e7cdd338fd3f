"""Queries from several host threads on one device, beside a direct-light run
on it: a launch's claims and the long marches that its lanes hand over are
its own, so every call answers as it does by itself.  The sizes are above
those up to which a launch needs neither (131,072 queries, 98,304 marches of
the direct light), and one below them."""
import ctypes as C
import threading

import numpy as np
import pytest

from helpers import Device, P, all_samples_and_tris, bits, prepared
from lighter_amd import _lib, scenes, workloads

pytestmark = pytest.mark.gpu
u32p = C.POINTER(C.c_uint32)
ROUNDS = 6


def test_queries_beside_each_other_and_a_light_pass(lib):
    spec = scenes.room_scene(lm=256, n_boxes=12, n_point=3)
    b = prepared(lib, spec)
    pos, nrm, tris = all_samples_and_tris(lib, b)
    N = len(pos)
    dev = Device(lib, tris)
    _lib.check(lib.lgx_SetSamples(dev.h, P(pos), P(nrm), N, None), lib)
    lights = workloads.make_lights(spec)
    L = len(lights)
    items = np.concatenate([(np.uint32(l) << np.uint32(26)) | np.arange(N, dtype=np.uint32) for l in range(L)])
    off = np.arange(L + 1, dtype=np.uint32) * N
    _lib.check(lib.lgx_DirectLightSetup(dev.h, lights, L, items.ctypes.data_as(u32p), len(items),
                                        off.ctypes.data_as(u32p), 1), lib)

    def light():
        _lib.check(lib.lgx_DirectLightRun(dev.h), lib)
        w = np.zeros(len(items), np.float32)
        v = np.zeros(len(items), np.float32)
        _lib.check(lib.lgx_ReadWeights(dev.h, P(w), P(v), len(items)), lib)
        return w, v

    rng = np.random.default_rng(8)

    def query(n):
        at = rng.integers(0, N, n)
        p = pos[at] + nrm[at] * rng.uniform(0.005, 1.0, (n, 1))
        q = p + rng.normal(0.0, 4.0, (n, 3))
        k = rng.uniform(0.05, 0.5, n)
        return lambda: dev.shadow(p, q, k)

    calls = [light, query(200_001), query(150_003), query(1_001)]
    want = [c() for c in calls]
    assert np.count_nonzero(want[0][1] < 1.0) > 1000 and want[1][1].max() > 64
    marches = np.count_nonzero((want[0][0] != 0.0) & ~np.isnan(want[0][0]))
    assert marches + np.count_nonzero(want[0][1] == 0.0) > 98_304
    wrong = []

    def loop(i):
        try:
            for r in range(ROUNDS):
                got = calls[i]()
                for g, w in zip(got, want[i]):
                    if not np.array_equal(g.view(np.uint32), w.view(np.uint32)):
                        wrong.append((i, r, int(np.count_nonzero(g.view(np.uint32) != w.view(np.uint32)))))
        except Exception as e:  # the thread's error is this test's
            wrong.append((i, repr(e)))

    threads = [threading.Thread(target=loop, args=(i,)) for i in range(len(calls))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    dev.close()
    b.destroy()
    assert not wrong, wrong
