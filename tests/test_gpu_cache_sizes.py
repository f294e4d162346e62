"""The radiance cache's kernels at the edges of their tiles (16 queries per matrix tile, two tiles per wave
and step; 64 training rows per block), against the PyTorch reference of the network."""
import numpy as np
import pytest

import cupbr_amd as cb

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from test_gpu_nrc import _hash32, encode, mlp, random_inputs  # noqa: E402


@pytest.mark.parametrize("n", [1, 15, 17, 31, 33, 65537])
def test_inference_sizes(n):
    """Within the accumulation's rounding of the reference that rounds to BF16 where the kernel does
    (1e-3 of the norm, as at other sizes: room for the few features whose
    rounding the two sine routines decide differently)."""
    rng = np.random.default_rng(n)
    cache = cb.RadianceCache((-1, 0, 2), (2, 5, 3), seed=6)
    x = torch.from_numpy(random_inputs(n, rng, (-1, 0, 2), (2, 5, 3))).cuda()
    got = cache.infer(x)
    want = mlp(torch.from_numpy(cache.get_weights()).cuda(), encode(x, (-1, 0, 2), (2, 5, 3)))
    assert got.shape == (n, 3)
    assert float(torch.linalg.norm(got - want)) <= 1e-3 * float(torch.linalg.norm(want))


@pytest.mark.parametrize("batch,rows", [(512, 1), (1024, 700), (16384, 3000), (24576, 40001)])
def test_training_batch_sizes(batch, rows):
    """Loss and first Adam step of batches of fewer, as many and more 64-row tiles than there are blocks
    (256 CUs), against the BF16-emulating reference: the loss to the rounding of the network (1e-2, as
    at other sizes), each weight with a gradient above 1% of the largest by lr against its sign."""
    rng = np.random.default_rng(batch)
    cache = cb.RadianceCache((0, 0, 0), (1, 1, 1), seed=9)
    w0 = cache.get_weights()
    x = np.zeros((rows, 20), np.float32)
    x[:, :16] = random_inputs(rows, rng)
    x[:, 16:19] = 0.5 + 0.3 * np.sin(3 * x[:, 0:3])
    loss = cache.train(torch.from_numpy(x).cuda(), batch=batch, steps=1, lr=1e-3, return_loss=True)
    step = cache.get_weights() - w0
    pick = (_hash32((1 * 0x9E3779B9 + 0x51ED270B) + np.arange(batch, dtype=np.uint64)) % rows).astype(np.int64)
    xb = torch.from_numpy(x[pick]).cuda()
    w = torch.from_numpy(w0).cuda().requires_grad_(True)
    o = mlp(w, encode(xb[:, :16], (0, 0, 0), (1, 1, 1)))
    want = ((o - xb[:, 16:19]) ** 2 / (o.detach() ** 2 + 0.01)).sum()
    (want / batch).backward()
    grad = w.grad.cpu().numpy()
    big = np.abs(grad) > 1e-2 * np.abs(grad).max()
    assert abs(float(loss[0]) - float(want.detach())) <= 1e-2 * float(want.detach())
    assert np.mean(np.sign(step[big]) == -np.sign(grad[big])) >= 0.98
    assert np.mean(np.abs(np.abs(step[big]) - 1e-3) <= 5e-5) >= 0.98


def test_training_steps_count_across_calls():
    """The step number seeds the batches and corrects the moments' bias: 3 + 2 steps are the 5 steps of
    one call, and setting the weights starts over."""
    rng = np.random.default_rng(1)
    x = np.zeros((500, 20), np.float32)
    x[:, :16] = random_inputs(500, rng)
    x[:, 16:19] = 0.5
    rows = torch.from_numpy(x).cuda()
    cache = cb.RadianceCache((0, 0, 0), (1, 1, 1), seed=2)
    w0 = cache.get_weights()
    cache.train(rows, batch=512, steps=5)
    one = cache.get_weights()
    cache.set_weights(w0)
    cache.train(rows, batch=512, steps=3)
    cache.train(rows, batch=512, steps=2)
    np.testing.assert_array_equal(cache.get_weights(), one)
