"""The network's forward pass over the tile shapes that its launches choose by
image size and sample count, against the float64 oracle."""
import numpy as np
import pytest

from chemsim_amd.cnn import Net
from oracle import cnn_oracle as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(16, 64, 1), (64, 128, 2), (128, 512, 1), (128, 512, 4)],
                         ids=lambda s: "x".join(map(str, s)))
def test_forward_over_the_tiles(ctx, shape):
    """Sizes that take the 32 x 32, 64 x 64 and larger tiles of the dilated
    layers and every channel block of the others.  Same points of rounding as
    the oracle, so its tolerance is that of the other forward tests."""
    h, w, n = shape
    c = 32
    p = K.init_params(c, 11).astype(np.float32)
    x = np.random.default_rng(12).standard_normal((n, h, w, 8)).astype(np.float32)
    with Net(ctx, h, w, base=c, batch=n) as net:
        net.set_params(p)
        y = net.forward(x)
    for i in {0, n - 1}:
        ref = K.Net(p, c, bf16_points=True).forward(x[i:i + 1])[0, ..., :3]
        err = np.linalg.norm(y[i] - ref) / np.linalg.norm(ref)
        assert err < 1e-2, (i, err)
