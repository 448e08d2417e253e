"""Scenes beyond the lengths that the FP32 triangle test can tell apart (its products are cubic in them: they vanish
below about 2^-34 and overflow above 2^41).  Which plane of a stack is nearest, and whether it lies before tmax, is not
decided reliably there; the edge functions and the FP64 refinement still are, so that calls succeed, a ray that meets no
triangle misses, and a hit names a triangle that the ray meets, with its exact distance."""
import numpy as np
import pytest

from test_gpu_leaf_steps import _stack

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("config", [{}, {"leaf_lanes": 1, "refill_interval": 1},
                                    {"block_size": 64, "blocks_per_cu": 20}], ids=["default", "at_once", "lean"])
@pytest.mark.parametrize("log2", [-60, 45])
def test_what_holds_beyond_the_range(log2, config):
    import pyrtx
    planes, instances, rays, scale = 9, 3, 1026, 2.0 ** log2
    ctx = pyrtx.Context(0)
    z, scene = _stack(planes, instances, planes, scale)
    blases, tlas = ctx.upload_scene(scene)
    rng = np.random.default_rng(log2 & 255)
    inst = rng.integers(0, instances, rays)
    up = rng.random(rays) < 0.3
    beside = np.arange(rays) % 2 == 1  # half way between two instances
    r = np.zeros((rays, 8), np.float32)
    r[:, 0] = 16.0 * inst + rng.integers(-8, 9, rays) / 16.0 + 8.0 * beside
    r[:, 1] = rng.integers(-8, 9, rays) / 16.0
    r[:, 2] = np.where(up, -16.0, 5.0)
    r[:, :3] *= scale
    r[:, 6] = np.where(up, 1.0, -1.0)
    r[:, 7] = 1e30
    d = torch.from_numpy(r).cuda()
    ctx.set_config(**config)
    for flags in (0, pyrtx.RTX_RAY_FLAG_CULL_NO_OPAQUE):  # the default and the ray-flag traversal
        got = ctx.trace_ray_buffer(tlas, d, pyrtx.RTX_QUERY_CLOSEST_HIT, ray_flags=flags)
        occ = ctx.trace_ray_buffer(tlas, d, pyrtx.RTX_QUERY_ANY_HIT, ray_flags=flags)
        ctx.sync()
        g, o = got.cpu().numpy(), occ.cpu().numpy()
        hit = g[:, 5] != -1
        assert not hit[beside].any() and not o[beside].any()
        assert np.array_equal(g[hit, 5], inst[hit]) and bool(((g[hit, 3] >= 0) & (g[hit, 3] < planes)).all())
        plane = z[g[hit, 3]]
        want = np.where(up[hit], 16.0 * scale + plane, 5.0 * scale - plane).astype(np.float32)
        assert np.array_equal(g[hit, 0].view(np.float32), want)
    ctx.close()
    del blases
