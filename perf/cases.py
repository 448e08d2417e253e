"""The work that programs built on librtx have it do, as cases that can be timed and compared.

Every case goes through the public entry points of `pyrtx` (the binding of the C ABI) with the launch configuration
that a new context has.  Meshes and rays are generated on the GPU from the seed; sizes are those of the repository's
own scenes, tests and benchmark (the reference's quads at 1200x800, the 512-instance query scene of 20M triangles
with 16.7M-ray buffers, the Cornell box with a 1.3M-triangle sphere at 1920x1080, 64 uneven scenes in one batch,
65,536 training paths per radiance-cache frame) and the smaller, odd ones between them.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.abspath(os.getcwd()), "build-up-phase_amd"))
import pyrtx  # noqa: E402
from pyrtx import scenes as S  # noqa: E402

DEV = "cuda:0"
BATCH_FILMS = ((256, 256), (512, 512), (1024, 768))


def listed():
    return [
        # the smallest calls: a handful of rays against one ordinary mesh (picking, a collision test); the time is
        # launches and one ray's latency
        dict(name="rays_pick", kind="rays", scene="field", tris=20480, instances=3, rays=777, coherent=False, any=False),
        # the reference program itself: two quads in two geometries and two instances, one ray per pixel
        dict(name="film_reference", kind="film", width=1200, height=800),
        # the headline ray set: primary rays of a 4096x4096 camera over 20M instanced triangles, closest hit
        dict(name="rays_coherent", kind="rays", scene="field", tris=20000000, instances=512, rays=4096 * 4096,
             coherent=True, any=False),
        # its counterpart: random origins and directions, as gathers and probes make them
        dict(name="rays_incoherent", kind="rays", scene="field", tris=20000000, instances=512, rays=4096 * 4096,
             coherent=False, any=False),
        # visibility queries inside a closed room around one dense mesh, a ragged number of them
        dict(name="rays_shadow", kind="rays", scene="room", tris=1310720, instances=1, rays=3000017, coherent=False,
             any=True),
        # alpha-tested and procedural content: cutout triangles and boxes with a sphere program, shaded into a film
        dict(name="film_cutout", kind="cutout", tris=327680, boxes=5000, instances=24, width=1920, height=1080),
        # loading one mesh: BLAS and TLAS from device buffers, then the first few rays through them
        dict(name="build_mesh", kind="build", tris=1310720, instances=2, rays=8192),
        # a frame over 64 uneven scenes: one batched build of all of them, their TLAS, one sample per pixel
        dict(name="batch_frame", kind="batch", scenes=64, tri_lo=1000, tri_hi=2000000, spp=1, depth=6),
        # an animated frame: a deforming mesh refitted in place, the TLAS rebuilt, the film traced
        dict(name="update_frame", kind="update", tris=327680, instances=64, width=1277, height=719),
        # path tracing, progressive: 4 more samples per pixel of the Cornell box at 1080p, full depth
        dict(name="render", kind="render", tris=1310720, width=1920, height=1080, spp=4, depth=8),
        # a frame of the radiance-cache integrator: 65,536 training paths, their Adam steps, one sample per pixel
        dict(name="nrc_frame", kind="nrc", tris=1310720, width=1920, height=1080, paths=65536, depth=8),
        # the cache as a program of its own: predictions for a film's worth of queries, then training on samples
        dict(name="nrc_cache", kind="cache", queries=2073600, samples=65536, batch=16384),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rays", "rays", "rays", "film", "cutout", "build", "batch", "update", "render", "nrc", "cache"])
    if kind == "rays":
        return dict(kind=kind, scene=rng.choice(["field", "room"]), tris=_log(rng, 2000, 12000000),
                    instances=_log(rng, 1, 512), rays=_log(rng, 500, 16000000) | 1, coherent=rng.random() < 0.5,
                    any=rng.random() < 0.4)
    if kind == "film":
        return dict(kind=kind, width=_log(rng, 60, 3840), height=_log(rng, 60, 2160))
    if kind == "cutout":
        return dict(kind=kind, tris=_log(rng, 2000, 1300000), boxes=_log(rng, 10, 20000), instances=_log(rng, 2, 64),
                    width=_log(rng, 200, 1920), height=_log(rng, 120, 1080))
    if kind == "build":
        return dict(kind=kind, tris=_log(rng, 500, 4000000), instances=_log(rng, 1, 300), rays=_log(rng, 500, 8192))
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randint(3, 48), tri_lo=_log(rng, 500, 2000), tri_hi=_log(rng, 20000, 1500000),
                    spp=rng.randint(1, 2), depth=rng.randint(3, 6))
    if kind == "update":
        return dict(kind=kind, tris=_log(rng, 1000, 1300000), instances=_log(rng, 1, 256), width=_log(rng, 200, 1920),
                    height=_log(rng, 120, 1080))
    if kind == "render":
        return dict(kind=kind, tris=_log(rng, 2000, 1300000), width=_log(rng, 120, 1920), height=_log(rng, 90, 1080),
                    spp=rng.randint(1, 6), depth=rng.randint(3, 8))
    if kind == "nrc":
        return dict(kind=kind, tris=_log(rng, 2000, 1300000), width=_log(rng, 200, 1920), height=_log(rng, 120, 1080),
                    paths=_log(rng, 4096, 65536), depth=rng.randint(4, 8))
    return dict(kind=kind, queries=_log(rng, 1000, 2000000) | 1, samples=_log(rng, 1000, 65536) | 1, batch=16384)


# ---- scenes -------------------------------------------------------------------------------------------------------

@functools.lru_cache(maxsize=1)
def _context():
    return pyrtx.Context(0)  # one context, as a program keeps it


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * int(seed) + 17)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64)


def _noise(p, g, octaves=3):
    """Smooth displacement of points [n, 3] in about [-1, 1]: a few random plane waves per octave."""
    out = torch.zeros(p.shape[0], device=DEV, dtype=torch.float64)
    for k in range(octaves):
        w = (_rand(g, 4, 3) - 0.5) * (8.0 * 2.0 ** k)
        ph = _rand(g, 4) * (2 * math.pi)
        for j in range(4):
            out += (0.5 ** k / 4) * torch.sin(p @ w[j] + ph[j])
    return out / 1.75


def _grid_indices(nu, nv, base=0):
    """Two triangles per cell of an (nu + 1) x (nv + 1) grid of vertices."""
    a = (torch.arange(nv, device=DEV)[:, None] * (nu + 1) + torch.arange(nu, device=DEV)[None, :]).reshape(-1) + base
    b, c, d = a + 1, a + nu + 1, a + nu + 2
    return torch.cat([torch.stack([a, b, c], 1), torch.stack([b, d, c], 1)], 0)


def _sphere(tris, g, radius=1.0, amp=0.1, centre=(0.0, 0.0, 0.0)):
    """A displaced sphere: a cube of 6 n x n grids pushed out to the sphere (12 n^2 triangles, closed surface)."""
    n = max(1, int(round(math.sqrt(tris / 12.0))))
    u = torch.linspace(-1.0, 1.0, n + 1, device=DEV, dtype=torch.float64)
    x, y = torch.meshgrid(u, u, indexing="xy")
    x, y, o = x.reshape(-1), y.reshape(-1), torch.ones((n + 1) ** 2, device=DEV, dtype=torch.float64)
    faces = [(x, y, o), (y, x, -o), (o, x, y), (-o, y, x), (y, o, x), (x, -o, y)]
    p = torch.cat([torch.stack(f, 1) for f in faces], 0)
    p = p / p.norm(dim=1, keepdim=True)
    v = p * (radius * (1.0 + amp * _noise(p, g)))[:, None] + torch.tensor(centre, device=DEV, dtype=torch.float64)
    idx = torch.cat([_grid_indices(n, n, f * (n + 1) ** 2) for f in range(6)], 0)
    return v.to(torch.float32).contiguous(), idx.to(torch.int32).contiguous()


def _terrain(tris, g, size=2.0, height=0.3):
    n = max(1, int(round(math.sqrt(tris / 2.0))))
    u = torch.linspace(-size / 2, size / 2, n + 1, device=DEV, dtype=torch.float64)
    x, z = torch.meshgrid(u, u, indexing="xy")
    p = torch.stack([x.reshape(-1), torch.zeros((n + 1) ** 2, device=DEV, dtype=torch.float64), z.reshape(-1)], 1)
    p[:, 1] = height * _noise(p, g)
    return p.to(torch.float32).contiguous(), _grid_indices(n, n).to(torch.int32).contiguous()


def _geom(mesh, opaque=True, transform=None):
    return {"vertices": mesh[0], "indices": mesh[1], "transform": transform, "opaque": opaque}


def _host_geom(g):
    return _geom((torch.from_numpy(g.vertices.astype(np.float32)).to(DEV),
                  torch.from_numpy(g.indices.astype(np.int32)).to(DEV)), transform=None if g.transform is None else
                 torch.from_numpy(np.ascontiguousarray(g.transform, np.float32)).to(DEV))


def _transforms(n, g, box, scale=(0.5, 2.0)):
    """[n, 3, 4] float32: random rotation, scale and position in [-box, box]^3."""
    q = torch.randn(n, 4, generator=g, device=DEV, dtype=torch.float64)
    w, x, y, z = (q / q.norm(dim=1, keepdim=True)).unbind(1)
    r = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                     2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                     2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], 1).reshape(n, 3, 3)
    s = scale[0] + (scale[1] - scale[0]) * _rand(g, n, 1, 1)
    t = (2 * _rand(g, n, 3, 1) - 1) * box
    return torch.cat([r * s, t], 2).to(torch.float32)


IDENTITY = torch.tensor([[1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 1, 0]], dtype=torch.float32)


def _instances(transforms, addresses, sbt_offset=None, flags=0, custom=None):
    n = transforms.shape[0]
    rec = np.zeros(n, pyrtx.INSTANCE_DTYPE)
    rec["xf"] = transforms.cpu().numpy().reshape(n, 12)
    rec["cm"] = (np.arange(n) if custom is None else custom) | (0xFF << 24)
    rec["sf"] = (0 if sbt_offset is None else np.asarray(sbt_offset)) | (flags << 24)
    rec["addr"] = np.asarray(addresses, np.uint64)
    return torch.from_numpy(rec.view(np.uint8).reshape(-1).copy()).to(DEV)


def _records(rec):
    return torch.from_numpy(np.ascontiguousarray(rec).view(np.uint8).reshape(-1).copy()).to(DEV)


def _world(case, seed):
    """Meshes (a list of meshes), transforms and the mesh of each instance, of the scenes that rays are shot into."""
    g = _gen(seed)
    n, m = case["instances"], case["tris"]
    if case.get("scene") == "room":  # a closed unit box of 12 triangles around one dense mesh per instance
        box = torch.tensor([[x, y, z] for z in (0.0, 1.0) for y in (0.0, 1.0) for x in (0.0, 1.0)], device=DEV)
        quads = [(0, 1, 3, 2), (4, 6, 7, 5), (0, 4, 5, 1), (2, 3, 7, 6), (0, 2, 6, 4), (1, 5, 7, 3)]
        wall = torch.tensor([t for a, b, c, d in quads for t in ((a, b, c), (a, c, d))], device=DEV, dtype=torch.int32)
        meshes = [(box.to(torch.float32).contiguous(), wall), _sphere(m, g, 0.3 if n == 1 else 0.06, 0.1)]
        xf = torch.cat([IDENTITY.to(DEV)[None], _transforms(n, g, 0.08 if n == 1 else 0.4, (0.9, 1.1))], 0)
        xf[1:, :, 3] += 0.5
        return meshes, xf, np.array([0] + [1] * n), (0.0, 1.0)
    if n < 10:  # one mesh of each kind
        meshes = [_sphere(m / 2, g), _terrain(m / 2, g)]
    else:  # ten meshes of uneven sizes: 5 spheres and 5 height fields
        w = (0.026, 0.056, 0.084, 0.11, 0.2)
        meshes = [_sphere(m * f, g, 1.0, 0.05) for f in w] + [_terrain(m * 0.105, g) for _ in range(5)]
    box = 50.0 if n >= 100 else 2.0 * n ** (1.0 / 3.0)
    return meshes, _transforms(n, g, box), np.arange(n) % len(meshes), (-box - 2.0, box + 2.0)


def _rays(case, seed, bounds):
    g = _gen(seed + 7777)
    n = case["rays"]
    lo, hi = bounds
    r = torch.empty(n, 8, device=DEV, dtype=torch.float32)
    if case["coherent"]:
        # the first n pixels of a square camera looking at the scene (from inside a room)
        w = max(1, int(math.ceil(math.sqrt(n))))
        i = torch.arange(n, device=DEV)
        tan = math.tan(math.radians(60.0 if lo < 0 else 75.0) / 2)
        eye = _rand(g, 3) * 0.02 + torch.tensor([0.0, 0.0, 3.0 * hi] if lo < 0 else [0.5, 0.5, 0.97], device=DEV)
        r[:, 0:3] = eye.to(torch.float32)
        r[:, 4] = ((((i % w).double() + 0.5) / w * 2 - 1) * tan).to(torch.float32)
        r[:, 5] = (-((torch.div(i, w, rounding_mode="floor").double() + 0.5) / w * 2 - 1) * tan).to(torch.float32)
        r[:, 6] = -1.0
    else:
        r[:, 0:3] = (lo + (hi - lo) * _rand(g, n, 3)).to(torch.float32)
        z = 1 - 2 * _rand(g, n)
        phi = 2 * math.pi * _rand(g, n)
        s = torch.sqrt(torch.clamp(1 - z * z, min=0))
        r[:, 4:7] = torch.stack([s * torch.cos(phi), s * torch.sin(phi), z], 1).to(torch.float32)
    r[:, 3] = 0.0
    r[:, 7] = 0.5 if case["any"] and lo == 0.0 else math.inf  # shadow rays inside the room end before its walls
    return r


def _cornell(case, seed):
    """The Cornell box of the repository's scenes with a displaced sphere from the GPU; (geometry lists, Scene, lights)."""
    sc, lights = S.cornell_scene(sphere_level=1, seed=seed & 0xFFFF, width=case["width"], height=case["height"])
    sphere = _sphere(case["tris"], _gen(seed), 0.3, 0.1, (0.58, 0.31, 0.36))
    return [[_host_geom(x) for x in sc.blas[0]], [_geom(sphere)]], sc, torch.from_numpy(lights).to(DEV)


def _uneven(case):
    """Triangle counts, log-uniform over the range, and film sizes of a batch's scenes."""
    f = [(k * 0.6180339887498949 + 0.5) % 1.0 for k in range(case["scenes"])]
    lo, hi = math.log(case["tri_lo"]), math.log(case["tri_hi"])
    return [math.exp(lo + (hi - lo) * x) for x in f], [BATCH_FILMS[(5 * k + k // 3) % 3] for k in range(case["scenes"])]


# ---- prepare ------------------------------------------------------------------------------------------------------

def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    st = {"case": case, "ctx": ctx}
    if kind in ("rays", "build"):
        meshes, xf, of, bounds = _world(case, seed)
        st["geoms"] = [[_geom(m)] for m in meshes]
        rc = case if kind == "rays" else dict(case, coherent=False, any=False)
        st["rays"] = _rays(rc, seed, bounds)
        st["mode"] = pyrtx.RTX_QUERY_ANY_HIT if rc["any"] else pyrtx.RTX_QUERY_CLOSEST_HIT
        st["out"] = torch.empty((case["rays"],) if rc["any"] else (case["rays"], 6), dtype=torch.int32, device=DEV)
        st["blas"] = [ctx.build_blas(x) for x in st["geoms"]]
        st["inst"] = _instances(xf, [st["blas"][b].address for b in of])
        st["xf"], st["of"] = xf, of
        st["tlas"] = ctx.build_tlas(st["inst"])
        for b in st["blas"]:
            b.keepalive = ()  # the build's scratch is not kept
    elif kind == "film":
        sc = S.scene_r0()
        blas = [ctx.build_blas([_host_geom(x) for x in geoms]) for geoms in sc.blas]
        st["inst"] = _instances(torch.from_numpy(sc.transforms), [blas[0].address] * 2, sc.sbt_offset, 1, sc.custom_index)
        st["blas"], st["tlas"], st["records"] = blas, ctx.build_tlas(st["inst"]), _records(sc.records)
        st["camera"] = _reference_camera(seed)
        st["film"] = torch.empty(case["height"], case["width"], 4, device=DEV)
    elif kind == "cutout":
        g = _gen(seed)
        n = case["instances"]
        lo = 4 * _rand(g, case["boxes"], 3) - 2
        boxes = torch.cat([lo, lo + 0.02 + 0.08 * _rand(g, case["boxes"], 3)], 1).to(torch.float32).contiguous()
        st["blas"] = [ctx.build_blas([_geom(_sphere(case["tris"], g), opaque=False)]),
                      ctx.build_blas([{"aabbs": boxes, "opaque": True}])]
        xf = torch.cat([_transforms(n, g, 2.0, (0.3, 0.8)), IDENTITY.to(DEV)[None]], 0)
        st["inst"] = _instances(xf, [st["blas"][0].address] * n + [st["blas"][1].address], [0] * n + [1])
        st["tlas"] = ctx.build_tlas(st["inst"])
        st["records"] = _records(S.hit_records(
            [S.PROGRAM_BARYCENTRIC, S.hit_group(S.PROGRAM_BARYCENTRIC, S.INTERSECTION_SPHERE)], np.zeros((2, 3)),
            any_hit=[S.ANY_HIT_CUTOUT | (3 << 8), 0]))
        st["film"] = torch.empty(case["height"], case["width"], 4, device=DEV)
    elif kind == "batch":
        g = _gen(seed)
        tris, films = _uneven(case)
        sc, views, lights = S.batch_scenes(count=case["scenes"], tri_lo=20, tri_hi=21)
        st["geoms"] = []
        for k in range(case["scenes"]):
            views[k]["width"], views[k]["height"] = films[k]
            st["geoms"].append([_geom(_sphere(tris[k], g, 0.3, 0.1, (0.5, 0.35, 0.5)))] +
                               [_host_geom(x) for x in sc.blas[k][1:]])
        st["blas"] = ctx.build_blas_batch(st["geoms"])
        st["scratch"] = st["blas"][0].keepalive[0]
        st["inst"] = _instances(torch.from_numpy(sc.transforms), [b.address for b in st["blas"]], sc.sbt_offset)
        st["tlas"] = ctx.build_tlas(st["inst"])
        st["records"], st["lights"], st["views"] = _records(sc.records), torch.from_numpy(lights).to(DEV), views
        st["films"] = torch.empty(sum(w * h for w, h in films), 4, device=DEV)
        st["seed"] = seed & 0xFFFF
    elif kind == "update":
        g = _gen(seed)
        rest = _sphere(case["tris"], g)
        moved = (rest[0].double() * (1.0 + 0.08 * _noise(2.0 * rest[0].double(), g))[:, None]).to(torch.float32)
        flags = pyrtx.RTX_BUILD_PREFER_FAST_TRACE_BIT | pyrtx.RTX_BUILD_ALLOW_UPDATE_BIT
        st["blas"] = [ctx.build_blas([_geom(rest)], flags), ctx.build_blas([_geom(_terrain(20000, g, 16.0, 1.0))])]
        st["moved"] = [_geom((moved.contiguous(), rest[1]))]
        n = case["instances"]
        xf = torch.cat([_transforms(n, g, 4.0, (0.4, 1.0)), IDENTITY.to(DEV)[None]], 0)
        xf[n, 1, 3] = -3.0
        st["inst"] = _instances(xf, [st["blas"][0].address] * n + [st["blas"][1].address])
        st["tlas"] = ctx.build_tlas(st["inst"])
        st["records"] = _records(S.hit_records([S.PROGRAM_BARYCENTRIC], np.zeros((1, 3))))
        st["film"] = torch.empty(case["height"], case["width"], 4, device=DEV)
    elif kind in ("render", "nrc"):
        geoms, sc, st["lights"] = _cornell(case, seed)
        st["blas"] = [ctx.build_blas(x) for x in geoms]
        st["inst"] = _instances(torch.from_numpy(sc.transforms), [b.address for b in st["blas"]], sc.sbt_offset)
        st["tlas"], st["records"], st["camera"] = ctx.build_tlas(st["inst"]), _records(sc.records), sc.camera
        for b in st["blas"]:
            b.keepalive = ()
        st["film"] = torch.empty(case["height"], case["width"], 4, device=DEV)
        st["seed"] = seed & 0xFFFF
        if kind == "nrc":
            st["nrc"] = pyrtx.Nrc(ctx, (0.0, 0.0, 0.0), (1.0, 1.0, 1.0), seed=1 + (seed & 0xFFFF))
    else:
        st["queries"], st["samples"] = _cache_data(case, seed)
        st["nrc"] = pyrtx.Nrc(ctx, (0.0, 0.0, 0.0), (1.0, 1.0, 1.0), seed=1 + (seed & 0xFFFF), batch_size=case["batch"])
    return st


def _reference_camera(seed):
    r = np.random.default_rng(seed)
    return (float(np.float32(r.uniform(-0.3, 0.3))), float(np.float32(r.uniform(-0.3, 0.3))),
            float(np.float32(r.uniform(9.7, 10.3))), 60.0)


def _cache_data(case, seed):
    """Queries [n, 12] and samples [m, 16] like path vertices in a unit box: positions on its walls and inside, unit
    normals and directions, the albedos of a few materials; targets a smooth radiance of position and normal."""
    g = _gen(seed)

    def vertices(n):
        p = _rand(g, n, 3)
        axis = torch.randint(0, 3, (n, 1), generator=g, device=DEV)
        side = torch.round(_rand(g, n, 1))
        p = torch.where(_rand(g, n, 1) < 0.7, p.scatter(1, axis, side), p)
        nd = torch.randn(n, 2, 3, generator=g, device=DEV, dtype=torch.float64)
        nd = (nd / nd.norm(dim=2, keepdim=True)).reshape(n, 6)
        alb = torch.tensor([[0.75, 0.75, 0.75], [0.75, 0.15, 0.15], [0.15, 0.75, 0.15]], device=DEV, dtype=torch.float64)
        return torch.cat([p, nd, alb[torch.randint(0, 3, (n,), generator=g, device=DEV)]], 1)

    q, s = vertices(case["queries"]), vertices(case["samples"])
    light = 0.4 + 0.6 * s[:, 1:2] + 0.3 * torch.sin(5 * s[:, 0:1]) * s[:, 4:5] + 0.5 * _rand(g, case["samples"], 1)
    s = torch.cat([s, torch.clamp(light * s[:, 9:12], min=0), torch.zeros(case["samples"], 1, device=DEV)], 1)
    return q.to(torch.float32).contiguous(), s.to(torch.float32).contiguous()


# ---- run ----------------------------------------------------------------------------------------------------------

def _hits(out):
    return {"tuv": out[:, :3].view(torch.float32), "ids": out[:, 3:]} if out.dim() == 2 else {"occluded": out}


def run(st):
    ctx, case = st["ctx"], st["case"]
    kind = case["kind"]
    if kind == "rays":
        return _hits(ctx.trace_ray_buffer(st["tlas"], st["rays"], st["mode"], out=st["out"]))
    if kind == "build":
        blas = [ctx.build_blas(x) for x in st["geoms"]]
        inst = _instances(st["xf"], [blas[b].address for b in st["of"]])
        tlas = ctx.build_tlas(inst)
        return _hits(ctx.trace_ray_buffer(tlas, st["rays"], st["mode"], out=st["out"]))
    if kind == "film":
        return ctx.trace_rays(st["tlas"], st["records"], st["camera"], case["width"], case["height"], film=st["film"])
    if kind == "cutout":
        return ctx.trace_rays(st["tlas"], st["records"], (0.0, 0.0, 6.0, 50.0), case["width"], case["height"],
                              film=st["film"], ray_flags=0)
    if kind == "batch":
        ctx.build_blas_batch(st["geoms"], into=st["blas"], scratch=st["scratch"])
        tlas = ctx.build_tlas(st["inst"], into=st["tlas"])
        return ctx.render_batch(tlas, st["records"], st["views"], st["lights"], spp=case["spp"],
                                max_depth=case["depth"], seed=st["seed"], films=st["films"])
    if kind == "update":
        st["blas"][0].keepalive = ()
        ctx.update_blas(st["blas"][0], st["moved"])
        tlas = ctx.build_tlas(st["inst"], into=st["tlas"])
        return ctx.trace_rays(tlas, st["records"], (0.0, 0.0, 9.0, 55.0), case["width"], case["height"], film=st["film"])
    if kind == "render":
        return ctx.render(st["tlas"], st["records"], st["camera"], st["lights"], case["width"], case["height"],
                          spp=case["spp"], max_depth=case["depth"], seed=st["seed"], film=st["film"])
    if kind == "nrc":
        film = ctx.render_nrc(st["tlas"], st["records"], st["camera"], st["lights"], st["nrc"], case["width"],
                              case["height"], spp=1, train_paths=case["paths"], max_depth=case["depth"],
                              seed=st["seed"], film=st["film"])
        return {"film": film, "params": st["nrc"].params()}
    rgb = st["nrc"].infer(st["queries"])
    st["nrc"].train(st["samples"])
    return {"rgb": rgb, "params": st["nrc"].params()}


# ---- work ---------------------------------------------------------------------------------------------------------

def _ray_flops(rays, prims):
    """Boxes of the 8-wide nodes on one path down the tree (18 operations each) and two triangles (60 each)."""
    return rays * (math.log(max(8, prims), 8) * 8 * 18 + 120)


def _structure(prims, rays):
    """Bytes of a structure that the rays have to read: all of it once (75 B a primitive), or the nodes and the
    triangle of one path each (64 B) where that is less."""
    return min(75 * prims, rays * 64 * (math.log(max(8, prims), 8) + 1))


def work(case):
    kind = case["kind"]
    if kind == "rays":
        n = case["rays"]
        return {"bytes": n * (32 + (4 if case["any"] else 24)) + _structure(case["tris"], n),
                "flops": _ray_flops(n, case["tris"])}
    if kind == "film":
        n = case["width"] * case["height"]
        return {"bytes": 16 * n, "flops": _ray_flops(n, 8)}
    if kind == "cutout":
        n, prims = case["width"] * case["height"], case["tris"] + case["boxes"]
        return {"bytes": 16 * n + _structure(prims, n), "flops": _ray_flops(n, prims)}
    if kind == "build":  # 12 B of indices and about 6 B of vertices in per triangle, 75 B of structure out
        return {"bytes": (18 + 75) * case["tris"] + 56 * case["rays"], "flops": _ray_flops(case["rays"], case["tris"])}
    if kind == "update":  # vertices, indices and the kept order and links in, the structure out
        n = case["width"] * case["height"]
        return {"bytes": (18 + 20 + 75) * case["tris"] + 16 * n + _structure(case["tris"], n),
                "flops": _ray_flops(n, case["tris"])}
    if kind == "batch":
        tris, films = _uneven(case)
        n = sum(w * h for w, h in films)
        return {"bytes": 93 * sum(tris) + 16 * n, "flops": _ray_flops(n * case["spp"] * case["depth"] * 0.8, tris[0])}
    if kind == "render":
        n = case["width"] * case["height"]
        return {"bytes": 16 * n + 75 * case["tris"], "flops": _ray_flops(n * case["spp"] * case["depth"], case["tris"])}
    mlp = 2 * (96 * 64 + 4 * 64 * 64 + 64 * 16)
    if kind == "nrc":  # three rays and a query per pixel; a training path traces two rays per vertex
        n, t = case["width"] * case["height"], case["paths"] * case["depth"] // 2
        return {"bytes": 16 * n + 75 * case["tris"] + 4 * 23888,
                "flops": _ray_flops(3 * n + 2 * t, case["tris"]) + mlp * (n + 3 * t)}
    return {"bytes": 60 * case["queries"] + 64 * case["samples"] + 8 * 23888,
            "flops": mlp * (case["queries"] + 3 * case["samples"])}


# ---- exact --------------------------------------------------------------------------------------------------------

def _closest64(rays, tri, want=2 ** 25):
    """Closest hits of rays [n, 8] on triangles [m, 3, 3] (both float64): (t, u, v, index), index -1 for a miss.  Rays
    are taken in chunks against all triangles, coefficients of the ray in each triangle's plane frame."""
    n, m = rays.shape[0], tri.shape[0]
    e1, e2 = tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    nrm = torch.linalg.cross(e1, e2)
    den = (nrm * nrm).sum(1)
    den = torch.where(den > 0, den, torch.full_like(den, math.nan))
    a1, a2 = torch.linalg.cross(e2, nrm) / den[:, None], torch.linalg.cross(nrm, e1) / den[:, None]
    # per triangle rows w, u', v' with: height = w . p - w0, u = a1 . p - u0, v = a2 . p - v0
    rows = torch.cat([nrm, a1, a2], 0)
    off = torch.cat([(nrm * tri[:, 0]).sum(1), (a1 * tri[:, 0]).sum(1), (a2 * tri[:, 0]).sum(1)])
    t_out = torch.zeros(n, 3, device=rays.device, dtype=torch.float64)
    idx = torch.full((n,), -1, device=rays.device, dtype=torch.int64)
    step = max(1, want // m)
    for i in range(0, n, step):
        r = rays[i:i + step]
        P, D = r[:, 0:3] @ rows.T - off, r[:, 4:7] @ rows.T
        t = -P[:, :m] / D[:, :m]
        u, v = P[:, m:2 * m] + t * D[:, m:2 * m], P[:, 2 * m:] + t * D[:, 2 * m:]
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= r[:, 3:4]) & (t <= r[:, 7:8])
        t = torch.where(ok, t, torch.full_like(t, math.inf))
        best, k = t.min(1)
        hit = torch.isfinite(best)
        j = torch.arange(r.shape[0], device=rays.device)
        row = torch.stack([best, u[j, k], v[j, k]], 1)
        t_out[i:i + step] = torch.where(hit[:, None], row, torch.zeros_like(row))
        idx[i:i + step] = torch.where(hit, k, torch.full_like(k, -1))
    return t_out, idx


def _triangles64(meshes, xf, of):
    out = []
    for i, b in enumerate(of):
        v = meshes[b][0].double() @ xf[i, :, :3].double().T + xf[i, :, 3].double()
        out.append(v[meshes[b][1].long()])
    return torch.cat(out, 0)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("rays", "build") and not case.get("any", False):
        meshes, xf, of, bounds = _world(case, seed)
        total = sum(meshes[b][1].shape[0] for b in of)
        if total * case["rays"] > 1.5e10:
            return None  # too many pairs to look at one by one
        rays = _rays(dict(case, coherent=case.get("coherent", False), any=False), seed, bounds)
        tuv, _ = _closest64(rays.double(), _triangles64(meshes, xf, of))
        return {"tuv": tuv, "ids": None}
    if kind == "film":
        sc = S.scene_r0()  # its arrays are the reference's literals
        w, h = case["width"], case["height"]
        tri, colour, bary = [], [], []
        for i in range(2):
            for gi, geom in enumerate(sc.blas[0]):
                v = geom.vertices.astype(np.float64) + geom.transform[:, 3].astype(np.float64) + sc.transforms[i][:, 3]
                for p, ix in enumerate(geom.indices):
                    tri.append(v[ix])
                    colour.append(sc.records["color"][int(sc.sbt_offset[i]) + gi].astype(np.float64))
                    bary.append((p, i, gi) == (1, 1, 1))
        cam = _reference_camera(seed)
        ay = math.tan(math.radians(cam[3]) / 2)
        x = (torch.arange(w, device=DEV, dtype=torch.float64) + 0.5) / w * 2 - 1
        y = (torch.arange(h, device=DEV, dtype=torch.float64) + 0.5) / h * 2 - 1
        rays = torch.zeros(h, w, 8, device=DEV, dtype=torch.float64)
        rays[..., 0:3] = torch.tensor(cam[:3], device=DEV, dtype=torch.float64)
        rays[..., 4], rays[..., 5], rays[..., 6], rays[..., 7] = (x * ay * w / h)[None, :], (-y * ay)[:, None], -1.0, 100.0
        tuv, k = _closest64(rays.reshape(-1, 8), torch.from_numpy(np.stack(tri)).to(DEV), 2 ** 23)
        table = torch.from_numpy(np.concatenate([np.stack(colour), [[0.0, 0.0, float(np.float32(0.2))]]])).to(DEV)
        c = table[k]
        b = torch.tensor(bary + [False], device=DEV)[k]
        c = torch.where(b[:, None], torch.stack([1 - tuv[:, 1] - tuv[:, 2], tuv[:, 1], tuv[:, 2]], 1), c)
        return torch.cat([c, torch.zeros_like(c[:, :1])], 1).reshape(h, w, 4)
    if kind == "cache":
        q, s = _cache_data(case, seed)
        p = _initial_parameters(1 + (seed & 0xFFFF)).to(DEV).requires_grad_(True)
        with torch.no_grad():
            rgb = torch.cat([torch.clamp(_mlp64(p, x.double()), min=0) for x in q.split(262144)])
        m, v = torch.zeros_like(p), torch.zeros_like(p)
        for k, x in enumerate(s.double().split(case["batch"])):
            y = _mlp64(p, x[:, :12])
            loss = ((y - x[:, 12:15]) ** 2 / (y.detach() ** 2 + 0.01)).sum(1).mean()
            (g,) = torch.autograd.grad(loss, p)
            with torch.no_grad():
                m, v = 0.9 * m + 0.1 * g, 0.99 * v + 0.01 * g * g
                p -= 1e-3 * (m / (1 - 0.9 ** (k + 1))) / (torch.sqrt(v / (1 - 0.99 ** (k + 1))) + 1e-8)
        return {"rgb": rgb, "params": p.detach().cpu().numpy()}
    return None


def _initial_parameters(seed):
    """The weights a new cache starts from: He-uniform, drawn from splitmix64 (Steele, Lea & Flood 2014)."""
    dims, fan = [(64, 96)] + [(64, 64)] * 4 + [(16, 64)], [81, 64, 64, 64, 64, 64]
    n = sum(r * c for r, c in dims)
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + np.arange(1, n + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    u = (z >> np.uint64(11)).astype(np.float64) / 9007199254740992.0
    out, at = [], 0
    for l, (r, c) in enumerate(dims):
        w = (2 * u[at:at + r * c] - 1).reshape(r, c) * math.sqrt(6.0 / fan[l])
        w[:, fan[l]:] = 0
        if l == 5:
            w[3:] = 0
        out += [w.astype(np.float32).astype(np.float64).reshape(-1), np.zeros(r)]
        at += r * c
    return torch.from_numpy(np.concatenate(out))


def _mlp64(p, q):
    f = 2.0 ** torch.arange(12, device=q.device, dtype=torch.float64) * math.pi
    a = q[:, 0:3, None] * f
    enc = torch.stack([torch.sin(a), torch.cos(a)], 3).reshape(q.shape[0], 72)
    x = torch.cat([enc, q[:, 3:12], torch.zeros(q.shape[0], 15, device=q.device, dtype=torch.float64)], 1)
    at = 0
    for l, (r, c) in enumerate([(64, 96)] + [(64, 64)] * 4 + [(16, 64)]):
        w, b = p[at:at + r * c].reshape(r, c), p[at + r * c:at + r * c + r]
        at += r * c + r
        x = x @ w.T + b
        if l < 5:
            x = torch.relu(x)
    return x[:, :3]
