"""The network's kernels at the image sizes where they can go wrong: levels of
one to 72 pixels (below and above the whole-image convolution's 64), sides that
are no multiple of the tiles', batches whose pixels end inside a chunk, a round
of 128 pixels or a wave, with one and several chunks.  Integer activations make
the forward pass exact; the gradients then differ from the emulated reference
only by the order of their FP32 sums and the BF16 rounding of gradients that
this may flip (bounded by 1e-3 of a layer's gradient, as for the larger frames)."""
import numpy as np
import pytest
import torch

from tests import unet_ref as R
from tests.test_learned import _cmp, _gpu_ctx, _inputs, _sparse_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,nb", [(8, 8, 1), (8, 8, 3), (8, 24, 2), (24, 8, 1), (16, 72, 1),
                                    (72, 16, 2), (24, 56, 3), (32, 128, 1)])
def test_forward_is_exact_and_gradients_tight(H, W, nb):
    print("test: network", H, W, nb, flush=True)
    from stroemung_amd.learned import PressureNet
    ctx = _gpu_ctx()
    net = PressureNet(ctx, H, W, nb + 1, seed=1)
    p = _sparse_params(13)
    net.set_params(p)
    rng = np.random.default_rng(14)
    x, _ = _inputs(nb, H, W, 15)
    x[..., 0] = rng.integers(-4, 5, (nb, H, W)) * x[..., 1]
    y = net.forward(x)
    with torch.no_grad():
        want = R.forward(R.unpack(p), torch.tensor(x)).numpy()
    np.testing.assert_array_equal(y, want)
    t = (rng.integers(-3, 4, (nb, H, W)) * x[..., 1]).astype(np.float32)
    loss, g = net.gradients(x, t)
    L16, g16 = R.gradients(p, x, t, bf16_acts=True)
    assert abs(loss - L16) <= 1e-5 * abs(L16)
    for name, off, shape in R.layout()[0]:
        size = int(np.prod(shape))
        _, rel = _cmp(g[off:off + size], g16[off:off + size])
        if np.any(g16[off:off + size]):
            assert rel < 1e-3, (name, rel)
        else:
            assert not np.any(g[off:off + size]), name
    net.close()
    ctx.close()
