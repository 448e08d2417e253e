"""The cache's kernels at the edges of their tiles: predictions of n queries equal those queries' in a larger call bit
for bit and touch nothing past them; a training call of several batches takes the steps that its batches take one by
one; gradients of partial and single blocks, and of more blocks than an Adam thread has slices, match the oracle."""
import numpy as np
import pytest

import oracle as O
from test_gpu_nrc import HI, LO, random_samples

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    import pyrtx
    c = pyrtx.Context(0)
    yield c
    c.sync()
    c.close()


def test_predictions_do_not_depend_on_the_call(ctx):
    import pyrtx
    nrc = pyrtx.Nrc(ctx, LO, HI, seed=5, batch_size=64)
    per_pass = torch.cuda.get_device_properties(0).multi_processor_count * 3 * 8 * 32  # queries of one grid pass
    q = torch.from_numpy(np.ascontiguousarray(random_samples(2 * per_pass + 64, 7)[:, :12])).cuda()
    full = nrc.infer(q).clone()
    for n in (1, 15, 16, 17, 31, 32, 33, 255, 257, 511, 513, per_pass - 1, per_pass, per_pass + 1, 2 * per_pass + 33):
        out = torch.full((n + 64, 3), -7.0, device="cuda")
        ctx._check(ctx.lib.rtx_nrc_cmd_infer(nrc.handle, q.data_ptr(), n, out.data_ptr()))
        ctx.sync()
        assert torch.equal(out[:n], full[:n]), n
        assert bool((out[n:] == -7.0).all()), n
    nrc.close()


@pytest.mark.parametrize("n", [1, 15, 63, 64, 65, 129, 1023, 1088])
def test_gradients_of_partial_blocks(ctx, n):
    """The bound of the larger gradient test (1e-3 of the norm): partial blocks add zeros."""
    import pyrtx
    nrc = pyrtx.Nrc(ctx, LO, HI, seed=3, batch_size=1088)
    smp = random_samples(n, n)
    g, loss = nrc.gradient(torch.from_numpy(smp).cuda())
    _, og, oloss = O.nrc(nrc.params(), smp, np.array(LO, np.float32), np.array(HI, np.float32), bf16=True)
    assert np.linalg.norm(g - og) <= 1e-3 * np.linalg.norm(og)
    assert abs(loss - oloss) <= 1e-3 * oloss
    assert nrc.status()[0] == 0  # a gradient is no step
    nrc.close()


def test_batches_of_a_call_are_steps(ctx):
    import pyrtx
    smp = torch.from_numpy(random_samples(5 * 192 + 70, 3)).cuda()
    whole, parts = (pyrtx.Nrc(ctx, LO, HI, seed=9, batch_size=192) for _ in range(2))
    whole.train(smp)
    for k in range(0, smp.shape[0], 192):
        parts.train(smp[k:k + 192].clone())
        assert parts.status()[0] == k // 192 + 1
    assert whole.status()[0] == 6 and whole.status()[1] == parts.status()[1]
    assert np.array_equal(whole.params(), parts.params())
    # the last step with its own bias corrections
    p0, m, v = pyrtx.Nrc(ctx, LO, HI, seed=9, batch_size=192), None, None
    pe = p0.params().copy()
    m, v = np.zeros_like(pe), np.zeros_like(pe)
    for k in range(0, smp.shape[0], 192):
        g, _ = p0.gradient(smp[k:k + 192].clone())
        O.adam(pe, m, v, g.astype(np.float64), 1e-3, 0.9, 0.99, 1e-8, k // 192 + 1)
        p0.train(smp[k:k + 192].clone())
    assert np.abs(p0.params() - pe).max() < 6e-6  # 1e-6 a step, as the single step's test
    for x in (whole, parts, p0):
        x.close()
