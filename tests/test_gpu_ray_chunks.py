"""How the traversal hands rays to waves: every ray of a launch is traced exactly once, whatever its count (one ray per
wave, partial waves, the first chunks alone, the queues' last chunks) and launch shape, and its result does not depend
on either: bit-identical to the same ray in a launch of another shape."""
import pytest

from helpers import small_mixed_scene
from pyrtx import scenes as S

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SENTINEL = -123456789


@pytest.fixture(scope="module")
def setup():
    import pyrtx
    ctx = pyrtx.Context(0)
    sc = small_mixed_scene(seed=3, instances=10, freq=10, cells=12)
    blases, tlas = ctx.upload_scene(sc)
    lanes = torch.cuda.get_device_properties(0).multi_processor_count * 64  # one 64-thread block per CU
    rays = torch.from_numpy(S.incoherent_rays(sc, 40 * lanes + 64, seed=4)).cuda()
    ctx.set_config(block_size=256, blocks_per_cu=4, ray_chunk=64)
    ref = {m: ctx.trace_ray_buffer(tlas, rays, m).clone() for m in (0, 1)}
    ctx.sync()
    yield ctx, tlas, rays, ref, lanes, blases
    ctx.sync()
    ctx.close()


# counts in units of the lanes of a launch of one 64-thread block per CU: (whole units, offset)
COUNTS = [(0, 1), (0, 63), (0, 65), (0, 255), (0, 257), (1, -1), (1, 0), (1, 1), (2, 31), (8, -1), (8, 0), (8, 1), (33, -7)]


@pytest.mark.parametrize("shape", [(64, 1, 1), (64, 1, 128), (128, 2, 1), (192, 3, 1), (256, 4, 1)])
@pytest.mark.parametrize("mode", [0, 1])
def test_every_ray_once(setup, shape, mode):
    ctx, tlas, rays, ref, lanes, _ = setup
    block, per_cu, chunk = shape
    ctx.set_config(block_size=block, blocks_per_cu=per_cu, ray_chunk=chunk)
    for units, off in COUNTS:
        n = units * lanes + off
        out = torch.full((n + 64, 6) if mode == 0 else (n + 64,), SENTINEL, dtype=torch.int32, device="cuda")
        for _ in range(2):  # the second launch finds the queues as the first one left them
            out[:n] = SENTINEL
            ctx.trace_ray_buffer(tlas, rays[:n], mode, out=out)
        ctx.sync()
        assert torch.equal(out[:n], ref[mode][:n]), (shape, n)
        assert bool((out[n:] == SENTINEL).all()), (shape, n)


def test_small_renders_do_not_depend_on_the_shape():
    import pyrtx
    ctx = pyrtx.Context(0)
    sc, lights = S.cornell_scene(sphere_level=2)
    blases, tlas = ctx.upload_scene(sc)
    films = []
    for block, per_cu, chunk in ((256, 4, 64), (256, 4, 1), (64, 1, 1), (192, 2, 128)):
        ctx.set_config(block_size=block, blocks_per_cu=per_cu, ray_chunk=chunk)
        for w, h, spp in ((5, 3, 1), (63, 33, 3), (161, 127, 2)):
            films.append(((w, h), ctx.render(tlas, sc.records, sc.camera, lights, w, h, spp=spp).clone()))
    ctx.sync()
    for (size, film), (_, first) in zip(films, films[:3] * 4):
        assert torch.equal(film, first), size
    ctx.close()
    del blases
