"""Abort of the direct-light march from inside the persistent kernel.

The reference's ltr_Abort is a no-op (lighter.cpp:1154-1157); here a bake's
worker raises a flag in pinned host memory, one claim of work in 64 relays
it to a device flag, and every wave reads the device flag at each claim, so
a long march stops within about one claim per wave instead of at the next
stage boundary.  The device-level switch lgx_DeviceAbort raises the device
flag before the launch, which makes the outcome deterministic: every wave leaves at its first claim (no march finishes and
no distance query runs, by the kernel's own counters), the run returns 0
with "direct light aborted", the lightmap keeps its colours, and once the
switch is cleared the same work gives the same weights bit for bit as
before.
(The stage-boundary abort of a whole bake runs on the CPU in test_abi.py.)
"""
import ctypes as C
import time

import numpy as np
import pytest

from helpers import Device, P, all_samples_and_tris, bits, prepared
from lighter_amd import _lib, api, scenes, workloads

pytestmark = pytest.mark.gpu
u32p = C.POINTER(C.c_uint32)


def test_device_abort_stops_the_march_and_leaves_the_lightmap(lib):
    spec = scenes.room_scene(lm=64, n_boxes=12, n_point=3)
    b = prepared(lib, spec)
    pos, nrm, tris = all_samples_and_tris(lib, b)
    N = len(pos)
    dev = Device(lib, tris)
    lm0 = np.full((N, 3), 0.125, np.float32)
    _lib.check(lib.lgx_SetSamples(dev.h, P(pos), P(nrm), N, P(lm0)), lib)
    lights = workloads.make_lights(spec)
    L = len(lights)
    items = np.concatenate([(np.uint32(l) << np.uint32(26)) | np.arange(N, dtype=np.uint32) for l in range(L)])
    off = np.arange(L + 1, dtype=np.uint32) * N

    def run():
        return lib.lgx_DirectLight(dev.h, lights, L, items.ctypes.data_as(u32p), len(items),
                                   off.ctypes.data_as(u32p), 1)

    def lightmap():
        out = np.zeros((N, 3), np.float32)
        _lib.check(lib.lgx_ReadLightmap(dev.h, P(out)), lib)
        return out

    def weights():
        w = np.zeros(len(items), np.float32)
        _lib.check(lib.lgx_ReadWeights(dev.h, P(w), None, len(items)), lib)
        return w

    assert run() == 1, _lib.last_error(lib)
    w1, lm1 = weights(), lightmap()
    assert (lm1 > 0.125).mean() > 0.2  # the lights reached the room
    _lib.check(lib.lgx_DeviceAbort(dev.h, 1), lib)
    lib.lgx_SetCounting(dev.h, 1)
    cnt = (C.c_uint64 * 6)()
    for _ in range(2):  # the switch stays on until cleared
        assert run() == 0
        assert "direct light aborted" in _lib.last_error(lib)
        assert np.array_equal(bits(lightmap()), bits(lm1))
        lib.lgx_ReadCounters(dev.h, cnt)
        assert cnt[4] == 0 and cnt[3] == 0, list(cnt)  # no march finished, no distance query ran
    lib.lgx_SetCounting(dev.h, 0)
    _lib.check(lib.lgx_DeviceAbort(dev.h, 0), lib)
    assert run() == 1, _lib.last_error(lib)
    assert np.array_equal(bits(weights()), bits(w1))
    lm2 = lightmap()
    assert np.all(lm2 >= lm1) and np.any(lm2 > lm1)  # the second run added its light
    dev.close()
    b.destroy()


def _grazing(extent, lm):
    """A flat square of extent m under a sun 0.02 degrees above its plane: every
    texel's march creeps thousands of steps along it, a wave's for
    milliseconds."""
    chart = scenes.Chart(np.zeros(3), np.array([extent, 0.0, 0.0]), np.array([0.0, extent, 0.0]), 1, 1, 0)
    parts = scenes.charts_to_part_arrays([chart], lm, lm)
    mesh = scenes.Mesh("ground", parts, [scenes.Instance(scenes.IDENTITY.copy(), 1.0, 1, "ground0")])
    d = np.array([1.0, 0.3, 3e-4])
    sun = scenes.dir_light(d / np.linalg.norm(d), np.ones(3), 2.0 * extent)
    return scenes.SceneSpec("ground", [mesh], [sun], dict(bounce_count=0, blur_size=0.0, max_num_threads=4), lm_size=lm)


def _bake(lib, spec, abort):
    """Seconds from the first look at the running light stage (with abort:
    from ltr_Abort then) to the bake's end, and the fractions seen between."""
    b = scenes.BuiltScene(lib, spec)
    st = api.WorkStatus()
    seen, t0 = [], None
    lib.ltr_Start(b.scene)
    while lib.ltr_GetStatus(b.scene, C.byref(st)):
        if st.stage == b"rendering lightmaps":
            if t0 is None:
                # a few looks: the march has begun
                time.sleep(0.02)
                t0 = time.perf_counter()
                if abort:
                    lib.ltr_Abort(b.scene)
            seen.append(st.completion)
        time.sleep(0.0005)
    t = time.perf_counter() - t0
    outputs = len(b.outputs())
    b.destroy()
    return t, seen, outputs


@pytest.mark.parametrize("extent,lm", [(2000.0, 256), (700.0, 512)])
def test_abort_and_progress_of_a_bake_inside_a_march(lib, extent, lm):
    """At most 65,536 marches, a wave for each from the start, which takes its
    next ones while the stage runs: the fraction rises and ltr_Abort ends the
    stage long before its time.  262,144 marches, all begun by lanes at once:
    an abort still leaves the bake without outputs."""
    spec = _grazing(extent, lm)
    _bake(lib, spec, False)
    full, seen, outputs = _bake(lib, spec, False)
    assert outputs == 1 and full > 0.05, (full, outputs)
    assert all(0.0 <= f <= 1.0 for f in seen) and seen == sorted(seen)
    part, _, outputs = _bake(lib, spec, True)
    assert outputs == 0
    if lm == 256:
        assert any(0.1 < f < 0.9 for f in seen), seen
        assert part < 0.5 * full, (part, full)
