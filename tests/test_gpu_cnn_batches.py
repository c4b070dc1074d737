"""A sample's results do not depend on the samples beside it, though the tiles
of the network's launches do: the dilated layers take 32 x 32, 64 x 64 or
128 x 128 GEMM tiles and the others 16 to 64 channels per block by the number of
blocks, and so does the data gradient with its masked epilogue."""
import numpy as np
import pytest

from chemsim_amd.cnn import Net
from oracle import cnn_oracle as K

pytestmark = pytest.mark.gpu

H, W, C = 128, 512, 32


@pytest.fixture(scope="module")
def data():
    rng = np.random.default_rng(21)
    n = 16
    return (K.init_params(C, 13).astype(np.float32), rng.standard_normal((n, H, W, 8)).astype(np.float32),
            rng.standard_normal((n, H, W, 3)).astype(np.float32), (rng.random((n, H, W)) < 0.8).astype(np.float32))


def test_prediction_alone_and_in_a_batch(ctx, data):
    """An output's sums run over its inputs in the same order in every tile:
    one image alone (32 x 32 tiles), among 4 and 8 (64 x 64) and 16 (128 x 128
    at the quarter-size layers) bit for bit."""
    p, x, _, _ = data
    with Net(ctx, H, W, base=C, batch=1) as net:
        net.set_params(p)
        alone = net.forward(x)
    for n in (2, 4, 8, 16):
        with Net(ctx, H, W, base=C, batch=n) as net:
            net.set_params(p)
            np.testing.assert_array_equal(net.forward(x), alone)


@pytest.mark.parametrize("n", [2, 4, 8])
def test_gradient_alone_and_in_a_batch(ctx, data, n):
    """A batch in which one sample has weights: its loss and gradient are the
    sample's own over n, an exact factor.  The other samples add zeros, but the
    weight gradient's K dimension is split differently, so its FP32 sums over up
    to 65536 pixels are grouped differently: eps sqrt(65536 / 2) = 1.1e-5 of a
    sum of random terms, with a factor of nine to spare."""
    p, x, t, w = data
    with Net(ctx, H, W, base=C, batch=1) as net:
        net.set_params(p)
        loss = net.loss_grad(x[:1], t[:1], w[:1])
        ref = net.get_grads().astype(np.float64)
    for at in (0, n - 1):
        order = [k for k in range(1, n)]
        order.insert(at, 0)
        wt = np.zeros((n, H, W), np.float32)
        wt[at] = w[0]
        with Net(ctx, H, W, base=C, batch=n) as net:
            net.set_params(p)
            got_loss = net.loss_grad(x[order], t[order], wt)
            got = net.get_grads().astype(np.float64)
        assert abs(got_loss * n - loss) <= 1e-5 * loss
        assert np.linalg.norm(got * n - ref) <= 1e-4 * np.linalg.norm(ref)
