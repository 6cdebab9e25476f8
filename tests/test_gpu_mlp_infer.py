"""GPU test of the network's one-launch inference: batches around its 16 rows, layer widths around the 16-wide
tiles and the four waves, and layers too wide for LDS (the layer-by-layer path). Small whole numbers: sums are
exact in FP32, and the BF16 rounding of the activations is done the same way here, so results are equal."""
import numpy as np
import pytest

from fastload_amd import DeviceArray
from fastload_amd import selector as sel

pytestmark = pytest.mark.gpu


def bf16(x):
    u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000
    return u.astype(np.uint32).view(np.float32).astype(np.float64)


@pytest.mark.parametrize("dims", [(40, 64, 64, 13), (1, 1, 1, 1), (17, 15, 65, 16), (5, 130, 16, 33), (1024, 64, 8, 4),
                                  (1025, 64, 8, 4)])
@pytest.mark.parametrize("batch", [1, 15, 16, 17, 50])
def test_infer(gpu, dims, batch):
    rng = np.random.default_rng(sum(dims) + batch)
    net = sel.MLP(dims)
    W = [rng.integers(-2, 3, (dims[i], dims[i + 1])).astype(np.float32) for i in range(3)]
    b = [rng.integers(-9, 10, dims[i + 1]).astype(np.float32) for i in range(3)]
    net.set_params(np.concatenate([a.ravel() for p in zip(W, b) for a in p]))
    X = rng.integers(-3, 4, (batch, dims[0])).astype(np.float32)
    h = X.astype(np.float64)
    for i in range(3):
        z = h @ W[i] + b[i]
        h = bf16(np.maximum(z, 0))
    assert np.array_equal(net.forward(X), z.astype(np.float32))
    cls, prob = net.predict(X)
    assert np.array_equal(cls, z.argmax(1))
    p = 1 / np.exp(z - z.max(1, keepdims=True)).sum(1)
    assert np.allclose(prob, p, rtol=1e-6, atol=0)
