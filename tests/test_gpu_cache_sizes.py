"""The radiance cache's kernels at the edges of their tiles (16 queries per matrix tile, two tiles per wave
and step; 64 training rows per block), against the PyTorch reference of the network."""
import numpy as np
import pytest

import cupbr_amd as cb

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from test_gpu_nrc import encode, mlp, random_inputs  # noqa: E402


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
