"""The work that users of this library have it do, as timed cases.

A caller drives the library in three ways: it bakes a whole scene (`ltr_Start`
.. `ltr_GetWorkOutput`), it runs single stages on a device scene that it keeps
(`lgx_DirectLightNoAlloc`, `lgx_AmbientOcclusion`, `lgx_RadLinks`, ..), or it
asks single points and segments (`lgx_Query*`).  The cases below take each of
these through its public entry points: `prepare` makes what the caller holds
before the call (the scene's samples, the device scene, links, buffers), `run`
is one pass, `exact` the same in 64 bits by brute force where that is cheap.

Scenes are the seeded rooms, terrains and city blocks of lighter_amd.scenes;
`scale` shrinks a terrain or city in extent while its triangles and texels per
square metre stay (1.0 is the 200 m terrain of 548,288 triangles or the 1 km
city of 1,991,072 triangles).
"""
from __future__ import annotations

import ctypes as C
import math
import time

import numpy as np
import torch

from lighter_amd import _lib, api, scenes, workloads

fp = C.POINTER(C.c_float)
dp = C.POINTER(C.c_double)
u32p = C.POINTER(C.c_uint32)
u8p = C.POINTER(C.c_uint8)

ROOM_TRIANGLES = 968  # 6 walls of 8 x 8 quads and 20 boxes of 10 triangles, about
FORMS = {"f64_links": 0, "f32_links": 1, "bf16_tiles": 3, "f16_tiles": 4, "f32_tiles": 5, "f16x3_tiles": 6}
AO_DISTANCE, AO_MULTIPLIER, AO_FALLOFF, AO_EFFECT = 2.0, 1.2, 1.0, 0.0
NO_ALLOC_ITEMS = 1 << 22  # lgx_DirectLightNoAlloc takes at most this many


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # an editor placing a few probes: distance, soft shadow, closest hit
        # and visibility of 64 points in a room; latency of four small calls
        dict(name="probe_room", kind="probe", scene="room", scale=1.0, points=64),
        # light probes over a terrain, an odd count
        dict(name="probe_terrain", kind="probe", scene="terrain", scale=0.25, points=100_003),
        # relighting one small atlas in a loop with the caller's own buffers
        dict(name="direct_room", kind="direct", scene="room", scale=1.0, items=8_001, lights=3),
        # the terrain's lights and its sun: nearly every item marches
        dict(name="direct_terrain", kind="direct", scene="terrain", scale=0.5, items=3_500_000, lights=4),
        # city lights: the largest batch the call takes, few items march
        dict(name="direct_city", kind="direct", scene="city", scale=0.25, items=NO_ALLOC_ITEMS, lights=8),
        # ambient occlusion of a part of the city, 64 rays a texel
        dict(name="ao_city", kind="ao", scene="city", scale=0.25, texels=700_001, rays=64),
        # radiosity links among a room's texels (everything sees everything)
        dict(name="links_room", kind="links", scene="room", scale=1.0, patches=32_768, bounces=2),
        # radiosity links of a part of the city (links reach 18 m), one bounce
        dict(name="links_city", kind="links", scene="city", scale=0.2, patches=440_003, bounces=1),
        # 64 lighting set-ups x RGB through a room's links at once
        dict(name="solve_bf16", kind="solve", scene="room", scale=1.0, patches=32_768, rhs=192, bounces=8,
             form="bf16_tiles"),
        # one RGB set-up on the sparse FP32 form
        dict(name="solve_rgb", kind="solve", scene="room", scale=1.0, patches=5_003, rhs=3, bounces=4,
             form="f32_links"),
        # the gradient of one RGB set-up (forward and reverse sweep)
        dict(name="grad_f16", kind="grad", scene="room", scale=1.0, patches=24_001, rhs=3, bounces=4,
             form="f16_tiles"),
        # a whole bake through the drop-in API: direct light, one bounce, AO,
        # export
        dict(name="bake_city", kind="bake", scene="city", scale=0.25, lights=8, bounces=1, rays=64, normals=False,
             half=False),
    ]


def _log(rng, lo, hi):
    """An odd whole number, its logarithm spread over [lo, hi]."""
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi)))) | 1))


def draw(rng):
    kind = rng.choice(["probe", "direct", "ao", "links", "solve", "grad", "bake"])
    scene = rng.choice(["room", "terrain", "city"])
    scale = {"room": 1.0, "terrain": round(rng.uniform(0.125, 0.5), 3), "city": round(rng.uniform(0.0625, 0.25), 4)}[scene]
    if kind == "probe":
        return dict(kind=kind, scene=scene, scale=scale, points=_log(rng, 17, 150_001))
    if kind == "direct":
        return dict(kind=kind, scene=scene, scale=scale, lights=rng.randint(1, 8),
                    items=_log(rng, 1_001, 200_001 if scene == "room" else 3_500_001))
    if kind == "ao":
        return dict(kind=kind, scene=scene, scale=scale, rays=rng.choice([17, 33, 64, 100]),
                    texels=_log(rng, 501, 60_001 if scene == "room" else 150_001))
    if kind == "links":
        return dict(kind=kind, scene=scene, scale=scale, bounces=rng.randint(1, 4),
                    patches=_log(rng, 401, 32_769 if scene == "room" else 100_001))
    if kind in ("solve", "grad"):
        return dict(kind=kind, scene="room", scale=1.0, patches=_log(rng, 401, 24_001),
                    rhs=rng.choice([3, 3, 6, 24, 48, 96, rng.randint(1, 192)]), bounces=rng.randint(1, 8),
                    form=rng.choice(sorted(FORMS)))
    return dict(kind=kind, scene=scene, scale=scale if scene == "city" else min(scale, 0.25) if scene == "terrain" else 1.0,
                lights=rng.randint(1, 8), bounces=rng.randint(0, 1), rays=rng.choice([0, 17, 64]),
                normals=rng.random() < 0.3, half=rng.random() < 0.3)


# ---------------------------------------------------------------------------
# scenes and their samples
# ---------------------------------------------------------------------------
def _spec(case, seed, lights=1, room_lm=64, extra_texels=1.0):
    """The case's scene; extra_texels scales the atlas area."""
    s = float(case["scale"])
    if case["scene"] == "room":
        spec = scenes.room_scene(seed=seed, lm=room_lm, n_point=max(1, lights - 1), with_sun=lights > 1, bounce_count=0)
    elif case["scene"] == "terrain":
        tiles = max(1, round(16 * s))
        lm = max(32, int(128 * math.sqrt(extra_texels)))
        spec = scenes.terrain_scene(seed=seed, grid=32 * tiles, extent=200.0 * tiles / 16, n_boxes=max(1, round(2000 * (tiles / 16) ** 2)),
                                    tiles=tiles, lm_total=lm * tiles, n_lights=max(1, lights - 1), sun=lights > 1)
    else:
        tiles = max(1, round(16 * s))
        lm = max(32, int(256 * math.sqrt(extra_texels)))
        spec = scenes.city_scene(seed=seed, extent=1000.0 * tiles / 16, grid=16 * tiles, n_boxes=max(1, round(155_000 * (tiles / 16) ** 2)),
                                 tiles=tiles, lm_total=lm * tiles, n_lights=lights)
    spec.albedo = None  # part colours come from arrays here, not from a callback
    return spec


def _triangles(case):
    """About how many triangles the case's scene has."""
    s = round(16 * float(case["scale"])) / 16
    return {"room": ROOM_TRIANGLES, "terrain": 548_288 * s * s, "city": 1_991_072 * s * s}[case["scene"]]


def _samples(case, seed, n, lights=1, want=0):
    """The scene's first n texels (positions, normals, uv/part/area rows), its
    shadow triangles, and the work items of its lights (`want` of them at
    least) with the texels that they number."""
    lib = _lib.load()
    threads = workloads.host_cores()[0]
    room_lm, extra = max(64, int(math.sqrt(n / 0.7))), max(1.0, n / (0.68 * (65536 if case["scene"] == "city" else 16384) * max(1, round(16 * float(case["scale"]))) ** 2))
    while True:
        spec = _spec(case, seed, lights, room_lm, extra)
        rad = []
        b, pos, nrm, tris, items, off = workloads.direct_workload(lib, spec, threads, radinfo=rad)
        b.destroy()
        if len(pos) >= n and len(items) >= want:
            break
        more = 1.05 * max(n / len(pos), want / max(1, len(items)))
        room_lm, extra = int(room_lm * math.sqrt(more)) + 4, extra * more
    return spec, pos[:n].copy(), nrm[:n].copy(), np.concatenate(rad)[:n].copy(), tris, items, off, pos, nrm


class _State:
    """What a caller keeps: the device scene or the scene, and the arrays."""

    dev = None
    built = None
    destroy = None

    def __del__(self):
        if self.dev:
            self.destroy(self.dev)
            self.dev = None


def _P(a):
    return a.ctypes.data_as(fp)


def _D(a):
    return a.ctypes.data_as(dp)


def _device(st, tris):
    lib = _lib.load()
    st.dev = lib.lgx_DeviceCreate(_P(tris), len(tris))
    _lib.check(st.dev, lib)
    st.tris, st.destroy = tris, lib.lgx_DeviceDestroy


def _inputs(case, seed):
    """The case's arrays (host memory), from the seed alone."""
    rng = np.random.default_rng(seed)
    k = case["kind"]
    x = _State()
    x.rays, x.bounces, x.form = case.get("rays", 0), case.get("bounces", 0), FORMS.get(case.get("form"), 0)
    if k == "probe":
        n = case["points"]
        m = min(n, 20_000)
        spec, pos, nrm, _, x.tris, _, _, _, _ = _samples(case, seed, m)
        # points 1 cm to 2 m off the surfaces, and segments and marches from
        # them to points in the scene's air
        at = rng.integers(0, m, n)
        x.p = np.ascontiguousarray(pos[at] + nrm[at] * rng.uniform(0.01, 2.0, (n, 1)), dtype=np.float32)
        x.q = np.ascontiguousarray(x.p + rng.normal(0.0, 4.0, (n, 3)) + [0.0, 0.0, 3.0], dtype=np.float32)
        x.k = rng.uniform(0.05, 0.5, n).astype(np.float32)
    elif k == "direct":
        n = case["items"]
        spec, _, _, _, x.tris, items, off, x.pos, x.nrm = _samples(case, seed, n // case["lights"], case["lights"], n)
        x.items, x.off = np.ascontiguousarray(items[:n]), np.minimum(off, n).astype(np.uint32)
        x.lights = workloads.make_lights(spec)
    elif k == "ao":
        _, x.pos, x.nrm, _, x.tris, _, _, _, _ = _samples(case, seed, case["texels"])
        x.ro = rng.uniform(0.0, 1.0, case["texels"]).astype(np.float32)
        x.lm0 = rng.uniform(0.1, 1.0, (case["texels"], 3)).astype(np.float32)
    elif k in ("links", "solve", "grad"):
        n = case["patches"]
        _, x.pos, nrm, rad, x.tris, _, _, _, _ = _samples(case, seed, n)
        x.nrm = scenes.normalize_rows_f32(nrm)
        x.area = np.ascontiguousarray(rad[:, 3])
        part = rng.uniform(0.2, 0.9, (64, 3)).astype(np.float32)
        x.diff = np.ascontiguousarray(part[rad[:, 2].astype(np.int64) % 64])
        # light of a few point lights in the air above the patches
        r = case.get("rhs", 3)
        lo, hi = x.pos.min(0).astype(np.float64), x.pos.max(0).astype(np.float64)
        at = lo + (hi - lo) * rng.uniform([0.1, 0.1, 0.6], [0.9, 0.9, 0.95], (4, 3))
        W = np.zeros((n, 4))
        for i in range(4):
            d = at[i] - x.pos
            l = np.sqrt((d * d).sum(1)) + 0.1
            W[:, i] = np.maximum(0.0, (d * x.nrm).sum(1) / l) * np.maximum(0.0, 1.0 - l / np.linalg.norm(hi - lo))
        E = W @ rng.uniform(0.3, 1.0, (4, r)) + 0.02
        if k == "links":
            x.emit = np.ascontiguousarray(E, dtype=np.float32)
        else:
            x.E = np.ascontiguousarray(E)
            x.g = np.ascontiguousarray(E * rng.uniform(-0.3, 0.3, E.shape))
    return x


def prepare(case, seed):
    lib = _lib.load()
    k = case["kind"]
    if k == "bake":
        st = _State()
        st.seed = seed % (1 << 31)
        spec = _spec(case, seed, case["lights"], room_lm=128)
        spec.config.update(bounce_count=case["bounces"], ao_distance=AO_DISTANCE if case["rays"] else 0.0,
                           ao_num_samples=max(1, case["rays"]), blur_size=0.5, ds2x=int(case["half"]),
                           generate_normalmap_data=int(case["normals"]))
        st.built = scenes.BuiltScene(lib, spec, dict(max_num_threads=workloads.host_cores()[0]))
        return st
    st = _inputs(case, seed)
    _device(st, st.tris)
    if k == "probe":
        n = len(st.p)
        st.dist, st.fac, st.steps = np.zeros(n, np.float32), np.zeros(n, np.float32), np.zeros(n, np.uint32)
        st.hit, st.occ = np.zeros(n, np.float32), np.zeros(n, np.uint8)
    elif k == "direct":
        _lib.check(lib.lgx_SetSamples(st.dev, _P(st.pos), _P(st.nrm), len(st.pos), None), lib)
        st.d_items = torch.from_numpy(st.items.view(np.int32)).cuda()
        st.d_w = torch.empty(len(st.items), device="cuda")
        st.d_vis = torch.empty(len(st.items), device="cuda")
    elif k == "ao":
        st.lm = np.zeros_like(st.lm0)
        st.black = np.zeros(3, np.float32)
    elif k == "links":
        st.total = np.zeros_like(st.emit)
    else:
        links = C.c_size_t(0)
        _lib.check(lib.lgx_RadLinks(st.dev, _P(st.pos), _P(st.nrm), len(st.pos), C.byref(links)), lib)
        st.total = np.zeros_like(st.E)
        if k == "grad":
            st.lam, st.dalb = np.zeros_like(st.E), np.zeros_like(st.E)
    return st


def run(st):
    lib = _lib.load()
    if st.built:  # bake: start, wait, take the images
        C.CDLL(None).srand(st.seed)  # the AO rotations come from the C library's generator
        status = api.WorkStatus()
        lib.ltr_Start(st.built.scene)
        while lib.ltr_GetStatus(st.built.scene, C.byref(status)):
            time.sleep(0.0005)
        if status.stage != b"finished":
            raise RuntimeError("the bake ended as " + repr(status.stage))
        outs = st.built.outputs()
        return dict(rgb=np.concatenate([o[3].reshape(-1, 3) for o in outs]),
                    normals=np.concatenate([o[4].reshape(-1, 4) for o in outs if o[4] is not None] or [np.zeros((1, 4), np.float32)]))
    if hasattr(st, "occ"):  # probe
        n = len(st.p)
        _lib.check(lib.lgx_QueryDistance(st.dev, _P(st.p), n, _P(st.dist)), lib)
        _lib.check(lib.lgx_QueryShadow(st.dev, _P(st.p), _P(st.q), _P(st.k), n, _P(st.fac), st.steps.ctypes.data_as(u32p)), lib)
        _lib.check(lib.lgx_QueryClosest(st.dev, _P(st.p), _P(st.q), n, _P(st.hit)), lib)
        _lib.check(lib.lgx_QueryOccluded(st.dev, _P(st.p), _P(st.q), n, st.occ.ctypes.data_as(u8p)), lib)
        return dict(dist=st.dist, fac=st.fac, steps=st.steps.astype(np.int64), hit=st.hit, occ=st.occ)
    if hasattr(st, "d_items"):  # direct
        _lib.check(lib.lgx_DirectLightNoAlloc(st.dev, st.lights, len(st.lights), st.d_items.data_ptr(), len(st.items),
                                              st.off.ctypes.data_as(u32p), st.d_w.data_ptr(), st.d_vis.data_ptr()), lib)
        return dict(weights=st.d_w, vis=st.d_vis)
    if hasattr(st, "ro"):  # ao: the lightmap so far up, occluded, down
        n = len(st.ro)
        _lib.check(lib.lgx_SetSamples(st.dev, _P(st.pos), _P(st.nrm), n, _P(st.lm0)), lib)
        _lib.check(lib.lgx_AmbientOcclusion(st.dev, _P(st.ro), st.rays, AO_DISTANCE, AO_MULTIPLIER, AO_FALLOFF,
                                            AO_EFFECT, _P(st.black)), lib)
        _lib.check(lib.lgx_ReadLightmap(st.dev, _P(st.lm)), lib)
        return st.lm
    if hasattr(st, "emit"):  # links and bounces
        links = C.c_size_t(0)
        _lib.check(lib.lgx_RadLinks(st.dev, _P(st.pos), _P(st.nrm), len(st.pos), C.byref(links)), lib)
        _lib.check(lib.lgx_RadBounce(st.dev, _P(st.diff), _P(st.emit), _P(st.area), st.bounces, _P(st.total)), lib)
        return dict(total=st.total, links=int(links.value))
    if hasattr(st, "lam"):  # gradient
        _lib.check(lib.lgx_RadSolveGrad(st.dev, _D(st.E), st.E.shape[1], _P(st.diff), _P(st.area), st.form, st.bounces,
                                        _D(st.g), _D(st.total), _D(st.lam), _D(st.dalb), None), lib)
        return dict(total=st.total, lam=st.lam, dalb=st.dalb)
    _lib.check(lib.lgx_RadSolve(st.dev, _D(st.E), st.E.shape[1], _P(st.diff), _P(st.area), st.form, st.bounces, 0,
                                _D(st.total), None), lib)
    return st.total


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """Inputs once in and outputs once out; operations: the tests and sums
    that any method does, without a walk's or a search's overhead."""
    k, t = case["kind"], _triangles(case)
    if k == "probe":
        n = case["points"]
        return dict(bytes=36 * t + n * (12 + 28 + 24 + 24 + 4 + 8 + 4 + 1), flops=300 * n)
    if k == "direct":
        n = case["items"]
        return dict(bytes=36 * t + n * (4 + 4 + 4) + 24 * n / max(1, case["lights"]), flops=30 * n)
    if k == "ao":
        n = case["texels"]
        return dict(bytes=36 * t + n * (24 + 12 + 4 + 12), flops=n * case["rays"] * 60)
    if k == "bake":
        tiles = max(1, round(16 * float(case["scale"])))
        n = {"room": 14_000, "terrain": 11_700 * tiles * tiles, "city": 46_500 * tiles * tiles}[case["scene"]]
        return dict(bytes=36 * t + 120 * n, flops=n * (30 * case["lights"] + 60 * case["rays"] + (case["bounces"] and 6000 * 20)))
    n, r = case["patches"], case.get("rhs", 3)
    # pairs within the linking distance, links among them (as measured on the
    # room of 32,768 patches and the city of 12 patches per square metre)
    pairs = n * n / 2 if case["scene"] == "room" else 6000 * n
    nnz = 0.11 * n * n if case["scene"] == "room" else 500 * n
    if k == "links":
        return dict(bytes=36 * t + n * (24 + 12 + 12 + 4 + 12) + 8 * nnz, flops=20 * pairs + 6 * nnz * case["bounces"])
    times = 1 if k == "solve" else 2
    return dict(bytes=16 * n * r * (1 if k == "solve" else 2.5) + 8 * nnz + 16 * n, flops=times * 2 * nnz * r * case["bounces"])


# ---------------------------------------------------------------------------
# tolerances
# ---------------------------------------------------------------------------
def tolerance(case):
    """About four times what the path was seen to be off `exact` where both
    take the same decisions: 3e-6 for AO factors (FP32 hit parameters), 2e-6
    for FP32 sums over links, 7e-5 for BF16 and 7e-6 for FP16 matrices.  A
    soft-shadow march decides on thresholds of its distances, so single
    factors differ by as much as they are (a room's weights: 4.5e-3)."""
    k = case["kind"]
    if k == "probe":
        return dict(rel=1e-3, max=0.99, differ=2e-3)
    if k == "direct":
        return dict(rel=6e-3, max=0.99)
    if k == "ao":
        return dict(rel=1.5e-5, max=1e-3)
    if k == "links":
        return dict(rel=1e-5, max=1e-4, differ=0.0)
    if k == "bake":
        return dict(rel=2e-5, max=1e-3)
    return {"f64_links": dict(rel=1e-12, max=1e-10), "f32_links": dict(rel=1.5e-5, max=1e-4),
            "bf16_tiles": dict(rel=3e-4, max=0.02), "f16_tiles": dict(rel=5e-5, max=5e-3),
            "f32_tiles": dict(rel=1e-5, max=1e-4), "f16x3_tiles": dict(rel=1e-5, max=1e-4)}[case["form"]]


# ---------------------------------------------------------------------------
# the same in 64 bits, by brute force over the triangles
# ---------------------------------------------------------------------------
def _t64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda().double()


def _unit(v):
    l = v.norm(dim=-1, keepdim=True)
    return torch.where(l > 0, v / l, torch.zeros_like(v))


def _distance(p, tri):
    """min(2, distance to the nearest triangle) of points p (n, 3)."""
    a, b, c = tri[:, 0], tri[:, 1], tri[:, 2]
    nrm = _unit(torch.linalg.cross(b - a, c - a))
    out = []
    for q in p.split(max(1, (1 << 23) // len(tri))):
        inside = torch.ones(len(q), len(tri), dtype=torch.bool, device=q.device)
        edge = torch.full((len(q), len(tri)), math.inf, dtype=torch.float64, device=q.device)
        for s, e in ((a, b), (b, c), (c, a)):
            d = e - s
            t = ((q @ d.T - (s * d).sum(1)) / (d * d).sum(1)).clamp(0, 1)
            o = q[:, None] - s - t[..., None] * d
            edge = torch.minimum(edge, (o * o).sum(2))
            out_dir = torch.linalg.cross(d, nrm)
            inside &= (q @ out_dir.T - (s * out_dir).sum(1)) <= 0
        plane = (q @ nrm.T - (a * nrm).sum(1)).abs()
        out.append(torch.where(inside, plane, edge.sqrt()).min(1).values.clamp(max=2.0))
    return torch.cat(out)


def _march(a, b, k, tri):
    """Soft-shadow factor of the march from a to b."""
    rd, end = _unit(b - a), (b - a).norm(dim=1)
    t, res = torch.full_like(end, 0.001), torch.ones_like(end)
    live = t < end
    while live.any():
        i = live.nonzero()[:, 0]
        h = _distance(a[i] + rd[i] * t[i, None], tri)
        dark = h < 0.001
        res[i] = torch.where(dark, torch.zeros_like(h), torch.minimum(res[i], h / (t[i] * k[i]).clamp(max=2.0)))
        t[i] += h.clamp(max=0.99)
        live[i] = ~dark & (t[i] < end[i])
    return res


def _closest(a, b, tri):
    """Closest hit on a -> b shrunk by 0.001 at both ends, 2 for none."""
    d = _unit(b - a)
    o, d = a + 0.001 * d, (b - 0.001 * d) - (a + 0.001 * d)
    p1, u, v = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    n = torch.linalg.cross(u, v)
    uu, uv, vv = (u * u).sum(1), (u * v).sum(1), (v * v).sum(1)
    D = uv * uv - uu * vv
    pn, pu, pv = (p1 * n).sum(1), (p1 * u).sum(1), (p1 * v).sum(1)
    out = []
    for o_, d_ in zip(o.split(max(1, (1 << 25) // len(tri))), d.split(max(1, (1 << 25) // len(tri)))):
        den = d_ @ n.T
        r = (pn - o_ @ n.T) / den
        wu = o_ @ u.T + r * (d_ @ u.T) - pu
        wv = o_ @ v.T + r * (d_ @ v.T) - pv
        s, t = (uv * wv - vv * wu) / D, (uv * wu - uu * wv) / D
        ok = (den.abs() >= 0.001) & (r >= 0) & (r <= 1) & (s >= 0) & (s <= 1) & (t >= 0) & (s + t <= 1)
        out.append(torch.where(ok, r, torch.full_like(r, 2.0)).min(1).values)
    return torch.cat(out)


def _factors(x, tri):
    """Dense symmetric link factors of the patches."""
    pos, nrm = _t64(x.pos), _t64(x.nrm)
    n = len(pos)
    F = torch.zeros(n, n, dtype=torch.float64, device="cuda")
    for i0 in range(0, n, 64):
        i = torch.arange(i0, min(n, i0 + 64), device="cuda")
        d = pos[None] - pos[i, None]
        da, db, l2 = (nrm[i, None] * d).sum(2), -(nrm[None] * d).sum(2), (d * d).sum(2)
        f = da * db / (l2 * l2 * math.pi)
        ok = (da > 0.001) & (db > 0.001) & (f >= 0.001) & (torch.arange(n, device="cuda")[None] > i[:, None])
        r, c = ok.nonzero(as_tuple=True)
        if len(r):
            hit = _closest(pos[i[r]], pos[c], tri) < 1.0
            F[i[r][hit], c[hit]] = f[r, c][hit]
    return F + F.T


def exact(case, seed):
    k, t = case["kind"], _triangles(case)
    if k == "bake" or case["scene"] != "room":
        return None
    if case.get("points", case.get("items", 0)) * t > 1.2e8 or case.get("patches", 0) > 5_100:
        return None
    if k == "ao" and case["texels"] * case["rays"] * t > 2.5e9:
        return None
    x = _inputs(case, seed)
    tri = _t64(x.tris).reshape(-1, 3, 3)
    if k == "probe":
        p, q = _t64(x.p), _t64(x.q)
        return dict(dist=_distance(p, tri).cpu().numpy(), fac=_march(p, q, _t64(x.k), tri).cpu().numpy(), steps=None,
                    hit=_closest(p, q, tri).cpu().numpy(), occ=None)
    if k == "direct":
        pos, nrm = _t64(x.pos), _t64(x.nrm)
        w = torch.full((len(x.items),), math.nan, dtype=torch.float64, device="cuda")
        vis = torch.ones(len(x.items), dtype=torch.float64, device="cuda")
        for l, L in enumerate(x.lights):
            b, e = int(x.off[l]), int(x.off[l + 1])
            s = torch.from_numpy((x.items[b:e] & np.uint32((1 << 26) - 1)).astype(np.int64)).cuda()
            if not len(s):
                continue
            P, N = pos[s], nrm[s]
            ldir, lpos = _t64(np.array(L.dir)), _t64(np.array(L.pos))
            if L.type == api.LTR_LT_DIRECT:
                gate = (N @ ldir).clamp(min=0)
                to = P + ldir * float(L.range)
                wl = torch.zeros_like(gate)
            else:
                d = lpos - P
                dist = d.norm(dim=1)
                d = d / dist[:, None]
                gate = (1 - (dist / float(L.range)).clamp(max=1)).pow(float(L.power)) * (d * N).sum(1).clamp(min=0)
                if L.type == api.LTR_LT_SPOT:
                    ang = (-(d @ ldir)).clamp(max=1).acos()
                    o, i = (math.pi * float(v) / 180 for v in (L.spot_angle_out, L.spot_angle_in))
                    gate = gate * ((ang - o) / (i - o if i != o else -0.001)).clamp(0, 1).pow(float(L.spot_curve))
                to = lpos.expand_as(P)
                wl = torch.full_like(gate, math.nan)
            m = gate > 0
            f = _march((P + N * 0.005)[m], to[m], torch.full((int(m.sum()),), float(L.radius), dtype=torch.float64, device="cuda"), tri)
            wl[m] = gate[m] * f
            w[b:e] = wl
            vis[b:e][m] = f
        return dict(weights=w.cpu().numpy(), vis=vis.cpu().numpy())
    if k == "ao":
        n, rays = case["texels"], case["rays"]
        P, N, ro = _t64(x.pos), _t64(x.nrm), _t64(x.ro)
        dv = torch.stack([N[:, 1], -N[:, 2], N[:, 0]], 1)
        up = _unit(torch.linalg.cross(N, dv))
        rt = torch.linalg.cross(N, up)
        o = P + N * 0.002
        ao = torch.zeros(n, dtype=torch.float64, device="cuda")
        for i in range(rays):
            ang = (i + ro) * (float(np.float32(137.508)) / 180 * math.pi)
            cs = math.sqrt((i + 0.5) / rays)
            sn = math.sqrt(1 - cs * cs)
            d = (ang.cos() * sn)[:, None] * rt + (ang.sin() * sn)[:, None] * up + cs * N
            hit = _closest(o, o + d * AO_DISTANCE, tri)
            ao += torch.where(hit < 1, 1 - hit, torch.zeros_like(hit))
        ao = (ao / rays * AO_MULTIPLIER).clamp(max=1)
        return (_t64(x.lm0) * (1 - ao * (1 - AO_EFFECT))[:, None]).cpu().numpy()
    F = _factors(x, tri)
    diff, area = _t64(x.diff), _t64(x.area)
    E = _t64(x.emit if k == "links" else x.E)
    n, r = E.shape
    mul = diff[:, torch.arange(r, device="cuda") % 3] * area[:, None]  # per column: albedo times area
    total, z, S = E.clone(), E, [E.clone()]
    for _ in range(case["bounces"]):
        z = F @ (z * mul)
        total = total + z
        S.append(total.clone())
    if k == "links":
        return dict(total=total.cpu().numpy(), links=None)
    if k == "solve":
        return total.cpu().numpy()
    y = _t64(x.g)
    lam, dalb = y.clone(), torch.zeros_like(E)
    for b in range(case["bounces"], 0, -1):
        u = area[:, None] * (F @ y)
        dalb += u * S[b - 1]
        y = diff[:, torch.arange(r, device="cuda") % 3] * u
        lam += y
    return dict(total=total.cpu().numpy(), lam=lam.cpu().numpy(), dalb=dalb.cpu().numpy())
