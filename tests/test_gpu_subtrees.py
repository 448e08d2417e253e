"""The build's bottom-up passes over subtrees in LDS and the nodes above them, against the oracle's postorder pass, at the
sizes where the split between the two can go wrong: around the largest subtree that a wave takes, a few of them, and
skewed trees whose upper nodes have single primitives as children.  Costs are FP32 sums in the same order: exact."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    import pyrtx
    c = pyrtx.Context(0)
    yield c
    c.sync()
    c.close()


def _boxes(n, shape, seed):
    rng = np.random.default_rng(seed)
    if shape == "skewed":  # halving distances: the radix tree is a chain of single primitives
        lo = np.zeros((n, 3))
        lo[:, 0] = 2.0 ** -(np.arange(n) % 20 + 1.0) + np.arange(n) // 20 * 1e-7
        lo[:, 1] = rng.uniform(0, 1e-6, n)
    else:
        lo = rng.uniform(-5, 5, (n, 3))
    ext = rng.uniform(0, 0.2, (n, 3)) ** 2
    b = np.concatenate([lo, lo + ext], 1).astype(np.float32)
    if shape == "invalid":  # inactive primitives have empty boxes
        b[::5, :3], b[::5, 3:] = np.inf, -np.inf
    return b


@pytest.mark.parametrize("shape", ["uniform", "skewed", "invalid"])
@pytest.mark.parametrize("n", [2, 6, 7, 8, 14, 63, 111, 112, 113, 224, 225, 700, 4099])
def test_refined_tree_bit_exact(ctx, n, shape):
    boxes = _boxes(n, shape, n)
    db = torch.from_numpy(boxes).cuda()
    for bits in (30, 63):
        _, order, kl, kr = ctx.debug_lbvh(db, bits)
        for rounds in (0, 1, 3):
            _, left, right, cost, height = ctx.debug_treelet(db, rounds, bits)
            el, er, ec, eh, _ = O.treelet_refine(kl, kr, boxes[order], rounds)
            assert np.array_equal(left, el) and np.array_equal(right, er), (n, shape, bits, rounds)
            assert np.array_equal(height, eh)
            assert np.array_equal(cost, ec)


def _check_structure(ctx, blas, n, width=8):
    """Walks a built BLAS: every slot below slot_count reached once, every triangle once, the header's counts and depth,
    and every child's decoded box around what lies below it."""
    info = ctx.as_info(blas)
    raw = blas.storage.cpu().numpy()
    head = raw[:256]
    lo, qs = head[48:60].view(np.float32), head[80:92].view(np.float32)
    slots = raw[256:256 + 64 * info.slot_count].reshape(-1, 64)
    seen = np.zeros(info.slot_count, bool)
    prims, nodes, deepest = [], 0, 0
    stack = [(0, 1, None)]
    seen[0] = True
    while stack:
        at, depth, outer = stack.pop()
        w = slots[at]
        nodes += 1
        deepest = max(deepest, depth)
        pq, e, imask, vmask, base = w[:6].view(np.uint16), w[6:9], int(w[9]), int(w[10]), int(w[12:16].view(np.uint32)[0])
        assert bin(vmask).count("1") <= width and imask & ~vmask == 0
        p = np.float32(np.float64(pq) * np.float64(qs) + np.float64(lo))
        scale = np.ldexp(np.float64(1.0), e.astype(int) - 127)
        k = 0
        for c in range(8):
            if not vmask >> c & 1:
                assert not w[16:64].reshape(6, 8)[:, c].any()
                continue
            slot = base + k
            k += 1
            assert slot < info.slot_count and not seen[slot]
            seen[slot] = True
            clo = p + scale * w[16:40].reshape(3, 8)[:, c]
            chi = p + scale * w[40:64].reshape(3, 8)[:, c]
            tol = 1e-5 * (np.abs(clo) + np.abs(chi) + scale)
            if imask >> c & 1:
                stack.append((slot, depth + 1, (clo - tol, chi + tol)))
            else:
                v = slots[slot][:36].view(np.float32).reshape(3, 3)
                prims.append(int(slots[slot][36:40].view(np.uint32)[0]))
                assert (v >= clo - tol).all() and (v <= chi + tol).all()
    assert seen.all() and sorted(prims) == list(range(n))
    assert (info.node_count, info.max_depth) == (nodes, deepest)


def _mesh(n, seed):
    g = torch.Generator().manual_seed(seed)
    v = torch.rand(n, 1, 3, generator=g) * 10 + 0.3 * torch.rand(n, 3, 3, generator=g)
    return {"vertices": v.reshape(-1, 3).contiguous().cuda(),
            "indices": torch.arange(3 * n, dtype=torch.int32).reshape(-1, 3).cuda()}


@pytest.mark.parametrize("width", [2, 5, 8])
@pytest.mark.parametrize("n", [1, 2, 8, 9, 111, 112, 113, 900, 20011])
def test_wide_structure(ctx, n, width):
    import pyrtx
    flags = pyrtx.RTX_BUILD_PREFER_FAST_TRACE_BIT | pyrtx.RTX_BUILD_MAX_WIDTH(width if width < 8 else 0)
    for f in (flags, flags | pyrtx.RTX_BUILD_MORTON63_BIT | pyrtx.RTX_BUILD_NO_TREELET_BIT):
        blas = ctx.build_blas([_mesh(n, n)], f)
        ctx.sync()
        _check_structure(ctx, blas, n, width)


def test_wide_structure_batched_and_updated(ctx):
    import pyrtx
    sizes = [1, 2, 1, 5000, 3, 112, 113, 7, 1, 40, 1500]
    meshes = [_mesh(n, 100 + k) for k, n in enumerate(sizes)]
    for blas, n in zip(ctx.build_blas_batch([[m] for m in meshes]), sizes):
        ctx.sync()
        _check_structure(ctx, blas, n)
    many = [[_mesh(1, k)] for k in range(70)]  # more structures than half their primitives
    for blas in ctx.build_blas_batch(many):
        ctx.sync()
        _check_structure(ctx, blas, 1)
    for n in (1, 112, 113, 3000):
        blas = ctx.build_blas([_mesh(n, n)], pyrtx.RTX_BUILD_ALLOW_UPDATE_BIT)
        moved = _mesh(n, n)
        moved["vertices"] = (moved["vertices"] * 1.5 + torch.sin(moved["vertices"])).contiguous()
        ctx.update_blas(blas, [moved])
        ctx.sync()
        _check_structure(ctx, blas, n)


@pytest.mark.parametrize("n", [3, 255, 256, 257, 1023, 1024, 1025, 4095, 4096, 4097, 5121, (1 << 17) - 1, 1 << 17, (1 << 17) + 4097, 1500001])
@pytest.mark.parametrize("kb", [4, 8])
def test_sort_tiles(ctx, n, kb):
    """The sort at the edges of its tiles and of its forms (one block, small tiles, large tiles), many equal keys."""
    rng = np.random.default_rng(n + kb)
    keys = rng.integers(0, 2 ** (8 * kb - 1), n, dtype=np.uint64)
    keys[: n // 3] &= np.uint64(0xFF00FF)
    keys[n // 2:] >>= np.uint64(8 * kb - 12)
    keys = keys.astype(np.uint32 if kb == 4 else np.uint64)
    got, order = ctx.debug_sort(keys)
    want = np.argsort(keys, kind="stable")
    assert np.array_equal(order, want.astype(np.uint32))
    assert np.array_equal(got, keys[want])
