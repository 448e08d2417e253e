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
