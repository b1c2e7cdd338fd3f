"""Ambient occlusion with several texels to a wave (at most 32 rays each)
against a wave per texel, which a device that counts its queries takes for
every ray count (from 2,049 texels on, the more texels the more to a wave): the same rays and the same order of their sum, so the colours
agree bit for bit (Job_AORender_Inner, lighter.cpp:799-841)."""

import ctypes as C

import numpy as np
import pytest

from helpers import Device, P
from lighter_amd import _lib

pytestmark = pytest.mark.gpu


def _soup(rng, n):
    c = rng.uniform(-4, 4, (n, 1, 3))
    return (c + rng.uniform(-0.8, 0.8, (n, 3, 3))).astype(np.float32).reshape(n, 9)


@pytest.mark.parametrize("rays", [1, 2, 3, 17, 21, 22, 31, 32, 33, 64, 65])
@pytest.mark.parametrize("texels", [1, 5, 1001, 7001, 140_001])
def test_packed_texels_match_wave_per_texel(lib, rays, texels):
    rng = np.random.default_rng(100 * rays + texels)
    dev = Device(lib, _soup(rng, 300))
    pos = rng.uniform(-4, 4, (texels, 3)).astype(np.float32)
    nrm = rng.normal(size=(texels, 3)).astype(np.float32)
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    ro = rng.uniform(0, 1, texels).astype(np.float32)
    lm0 = rng.uniform(0, 1, (texels, 3)).astype(np.float32)
    col = np.array([0.1, 0.2, 0.3], np.float32)
    out = []
    for count in (0, 1):
        _lib.check(lib.lgx_SetCounting(dev.h, count), lib)
        _lib.check(lib.lgx_SetSamples(dev.h, P(pos), P(nrm), texels, P(lm0)), lib)
        _lib.check(lib.lgx_AmbientOcclusion(dev.h, P(ro), rays, 3.0, 1.2, 1.5, 0.4, P(col)), lib)
        got = np.zeros_like(lm0)
        _lib.check(lib.lgx_ReadLightmap(dev.h, P(got)), lib)
        out.append(got)
    dev.close()
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
    assert texels < 1000 or np.any(out[0] != lm0)


def test_sample_sets_of_changing_size(lib):
    """One device given sample sets that grow and shrink, against a
    new device for each."""
    rng = np.random.default_rng(3)
    tris = _soup(rng, 300)
    dev = Device(lib, tris)
    col = np.ones(3, np.float32)
    for n in (2000, 1, 499, 2001, 700, 64, 0, 65):
        pos = rng.uniform(-4, 4, (n, 3)).astype(np.float32)
        nrm = rng.normal(size=(n, 3)).astype(np.float32)
        ro = rng.uniform(0, 1, n).astype(np.float32)
        one = Device(lib, tris)
        out = []
        for d in (dev, one):
            _lib.check(lib.lgx_SetSamples(d.h, P(pos), P(nrm), n, None), lib)
            _lib.check(lib.lgx_AmbientOcclusion(d.h, P(ro), 24, 2.0, 1.0, 1.0, 0.0, P(col)), lib)
            got = np.zeros((n, 3), np.float32)
            if n:
                _lib.check(lib.lgx_ReadLightmap(d.h, P(got)), lib)
            out.append(got)
        one.close()
        assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32)), n
    dev.close()
