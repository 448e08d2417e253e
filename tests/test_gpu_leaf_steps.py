"""The traversal's leaf steps, where a wave's lanes test each other's triangles: stacks of parallel triangles give leaf
groups of one to eight triangles, whole waves with a leaf group in every lane (more owners than one step takes) and
waves with one, under the extreme thresholds and the largest LDS stack.  The planes lie at multiples of 1/4 and the rays
run along the axis, so every distance is exact in FP32 and the nearest triangle is known: results are compared for
equality."""
import numpy as np
import pytest

from pyrtx import scenes as S

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

CONFIGS = [{}, {"leaf_lanes": 1, "refill_interval": 1}, {"leaf_lanes": 33}, {"leaf_lanes": 64, "refill_interval": 64},
           {"block_size": 192, "blocks_per_cu": 2}, {"lds_stack_depth": 29}, {"lds_stack_depth": 1}]


@pytest.fixture(scope="module")
def ctx():
    import pyrtx
    c = pyrtx.Context(0)
    yield c
    c.sync()
    c.close()


def _stack(planes, instances, seed, scale):
    rng = np.random.default_rng(seed)
    z = -0.25 * rng.permutation(planes)
    v = np.empty((planes, 3, 3), np.float32)
    v[:, 0, :2], v[:, 1, :2], v[:, 2, :2] = (-4, -4), (4, -4), (0, 4)
    v[:, :, 2] = z[:, None]
    v *= scale
    geom = S.Geometry(v.reshape(-1, 3), np.arange(3 * planes, dtype=np.uint32).reshape(-1, 3))
    xf = np.zeros((instances, 3, 4), np.float32)
    xf[:, :, :3] = np.eye(3)
    xf[:, 0, 3] = 16.0 * scale * np.arange(instances)
    zero = np.zeros(instances, np.uint32)
    return z * scale, S.Scene([[geom]], xf, np.zeros(instances, np.int64), zero, zero + 255, zero, zero)


@pytest.mark.parametrize("rays", [1, 64, 4097])
@pytest.mark.parametrize("planes", [1, 2, 3, 5, 8, 9, 40])
def test_stacked_triangles(ctx, planes, rays):
    _check(ctx, planes, rays, 1.0)


# the triangle test's FP32 products are cubic in the lengths: they vanish at 2^-60 and overflow at 2^45
_range = pytest.mark.xfail(strict=True, reason="cubic products leave the FP32 range")


@pytest.mark.parametrize("log2", [pytest.param(-60, marks=_range), -20, 20, 30, pytest.param(45, marks=_range)])
def test_stacked_triangles_at_other_scales(ctx, log2):
    """Powers of two, exact again; rays along an axis in a large scene overflow the node test's scaled slopes."""
    _check(ctx, 9, 513, 2.0 ** log2)


def _check(ctx, planes, rays, scale):
    import pyrtx
    instances = 3
    z, scene = _stack(planes, instances, planes, scale)
    blases, tlas = ctx.upload_scene(scene)
    rng = np.random.default_rng(rays)
    inst = rng.integers(0, instances, rays)
    up = rng.random(rays) < 0.3
    r = np.zeros((rays, 8), np.float32)
    r[:, 0] = 16.0 * inst + rng.integers(-8, 9, rays) / 16.0
    r[:, 1] = rng.integers(-8, 9, rays) / 16.0
    r[:, 2] = np.where(up, -16.0, 5.0)
    r[:, :3] *= scale
    r[:, 6] = np.where(up, 1.0, -1.0)
    near = np.where(up, 16.0 * scale + z.min(), 5.0 * scale - z.max())
    # tmax: unbounded, exactly at the nearest plane (a hit), and one step below it (a miss)
    kind = rng.integers(0, 3, rays)
    r[:, 7] = np.choose(kind, [np.full(rays, 1e30), near, np.nextafter(near.astype(np.float32), np.float32(0))])
    hit = kind < 2
    prim = np.where(up, z.argmin(), z.argmax())
    d = torch.from_numpy(r).cuda()
    base = ctx.config()
    try:
        for cfg in CONFIGS:
            ctx.set_config(**cfg)
            for flags in (0, pyrtx.RTX_RAY_FLAG_CULL_NO_OPAQUE):  # the default and the ray-flag traversal
                got = ctx.trace_ray_buffer(tlas, d, pyrtx.RTX_QUERY_CLOSEST_HIT, ray_flags=flags)
                occ = ctx.trace_ray_buffer(tlas, d, pyrtx.RTX_QUERY_ANY_HIT, ray_flags=flags)
                first = ctx.trace_ray_buffer(tlas, d, pyrtx.RTX_QUERY_CLOSEST_HIT,
                                             ray_flags=flags | pyrtx.RTX_RAY_FLAG_TERMINATE_ON_FIRST_HIT)
                ctx.sync()
                g, f = got.cpu().numpy(), first.cpu().numpy()
                assert np.array_equal(g[:, 5] != -1, hit), cfg
                assert np.array_equal(g[hit, 0].view(np.float32), near[hit].astype(np.float32)), cfg
                assert np.array_equal(g[hit, 3], prim[hit]) and np.array_equal(g[hit, 5], inst[hit]), cfg
                assert np.array_equal(occ.cpu().numpy() != 0, hit), cfg
                assert np.array_equal(f[:, 5] != -1, hit), cfg
                zf = np.where(up, f[:, 0].view(np.float32) - 16.0 * scale, 5.0 * scale - f[:, 0].view(np.float32))
                assert np.array_equal(zf[hit], z[f[hit, 3]]), cfg
            ctx.set_config(**base)
    finally:
        ctx.set_config(**base)
    del blases
