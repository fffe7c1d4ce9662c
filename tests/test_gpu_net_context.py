"""A network whose context has been closed still computes (on the default
stream), and gives what it gave before."""
import numpy as np
import pytest

from stroemung_amd.learned import PressureNet
from tests.test_learned import _gpu_ctx, _inputs

pytestmark = pytest.mark.gpu


def test_forward_and_gradients_after_the_context_is_closed():
    print("test: network without its context", flush=True)
    ctx = _gpu_ctx()
    net, late = PressureNet(ctx, 16, 24, 3, seed=1), PressureNet(ctx, 16, 24, 3, seed=1)
    x, t = _inputs(3, 16, 24, 5)
    y, (loss, g) = net.forward(x), net.gradients(x, t)
    ctx.close()
    for n in (net, late):   # with and without gradients before
        np.testing.assert_array_equal(n.forward(x), y)
        l2, g2 = n.gradients(x, t)
        assert l2 == loss
        np.testing.assert_array_equal(g2, g)
        n.close()
