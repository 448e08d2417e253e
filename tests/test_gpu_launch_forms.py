"""The traversal kernels' forms by launch shape - with the octant table and the triangle tasks in LDS, lean with four
and with five waves per SIMD - find the same: stacks of triangles at known distances, and films of whole paths."""
import pytest

import test_gpu_leaf_steps as leaf
from pyrtx import scenes as S

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SHAPES = [dict(block_size=b, blocks_per_cu=n, lds_stack_depth=d)
          for b, n, d in ((64, 12, 12), (64, 16, 12), (64, 16, 16), (128, 8, 16), (64, 20, 12), (256, 5, 12), (256, 32, 4))]


@pytest.fixture(scope="module")
def ctx():
    import pyrtx
    c = pyrtx.Context(0)
    yield c
    c.sync()
    c.close()


@pytest.mark.parametrize("planes,rays", [(1, 1), (2, 63), (3, 4097), (8, 65), (40, 20011)])
def test_stacked_triangles(ctx, monkeypatch, planes, rays):
    """One to eight triangles a leaf group; every lane of a wave with one, and a single lane."""
    monkeypatch.setattr(leaf, "CONFIGS", SHAPES + [dict(s, leaf_lanes=1, refill_interval=1) for s in SHAPES] +
                        [dict(s, leaf_lanes=64) for s in SHAPES])
    leaf._check(ctx, planes, rays, 1.0)


def test_whole_paths(ctx):
    sc, lights = S.cornell_scene(sphere_level=2)
    blases, tlas = ctx.upload_scene(sc)
    base = ctx.config()
    want = ctx.render(tlas, sc.records, sc.camera, lights, 161, 127, spp=2).clone()
    for shape in SHAPES:
        ctx.set_config(**shape)
        got = ctx.render(tlas, sc.records, sc.camera, lights, 161, 127, spp=2)
        ctx.sync()
        assert torch.equal(got, want), shape
        ctx.set_config(**base)
    del blases
