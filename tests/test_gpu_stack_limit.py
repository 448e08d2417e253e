"""A BLAS emptied by an update under a TLAS that was not rebuilt: rays enter it, find no nodes and pop in the same step.
With a stack limit that the entry's pushes exceed, the ray ends there and the overflow is reported."""
import numpy as np
import pytest

import oracle as O
from pyrtx import scenes as S

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("flags", [0, 0x80], ids=["default", "cull_no_opaque"])  # both traversal variants
@pytest.mark.parametrize("limit,lds", [(1, 12), (1, 1), (2, 1), (3, 1), (0, 12), (0, 1)])
def test_empty_blas_under_a_stack_limit(limit, lds, flags):
    import pyrtx
    ctx = pyrtx.Context(0)
    mesh = S.icosphere(2)
    dev = lambda v: [{"vertices": torch.from_numpy(np.ascontiguousarray(v, np.float32)).cuda(),
                      "indices": torch.from_numpy(mesh.indices.astype(np.int32)).cuda()}]
    blas = ctx.build_blas(dev(mesh.vertices),
                          flags=pyrtx.RTX_BUILD_PREFER_FAST_TRACE_BIT | pyrtx.RTX_BUILD_ALLOW_UPDATE_BIT)
    n = 64  # overlapping copies on a line: every ray along it passes through all of them
    xf = np.zeros((n, 3, 4), np.float32)
    xf[:, :, :3] = np.eye(3)
    xf[:, 0, 3] = 0.25 * np.arange(n)
    zero = np.zeros(n, np.uint32)
    tlas = ctx.build_tlas(O.instance_records(xf, [blas.address] * n, zero, zero + 255, zero, zero))
    rays = np.zeros((5000, 8), np.float32)
    rng = np.random.default_rng(7)
    rays[:, 0] = np.where(rng.random(5000) < 0.5, -4.0, 24.0)
    rays[:, 1:3] = rng.uniform(-0.2, 0.2, (5000, 2))
    rays[:, 4] = np.where(rays[:, 0] < 0, 1.0, -1.0)
    rays[:, 7] = 1e30
    rays = torch.from_numpy(rays).cuda()
    hit = ctx.trace_ray_buffer(tlas, rays, pyrtx.RTX_QUERY_CLOSEST_HIT, ray_flags=flags)
    ctx.sync()
    assert bool((hit[:, 5] != -1).all())
    ctx.update_blas(blas, dev(np.full_like(mesh.vertices, np.nan)))
    ctx.sync()
    ctx.set_config(lds_stack_depth=lds, leaf_lanes=1,
                   stack_limit=limit or pyrtx.RTX_TRACE_STACK_LIMIT_DERIVED)
    for mode in (pyrtx.RTX_QUERY_CLOSEST_HIT, pyrtx.RTX_QUERY_ANY_HIT):
        out = ctx.trace_ray_buffer(tlas, rays, mode, ray_flags=flags)
        code = 0
        try:
            ctx.sync()
        except pyrtx.RtxError as e:
            code = e.code
        # 64 instances take two levels at least: one entry is too few for the groups left on both
        allowed = {0: (0,), 1: (-1001,)}.get(limit, (0, -1001))
        assert code in allowed, code
        got = out[:, 5] if mode == pyrtx.RTX_QUERY_CLOSEST_HIT else out - 1
        assert bool((got == -1).all())
    ctx.close()
