"""What a network keeps on the device: the partial sums of its gradients come with
the first call that needs them, whichever it is, and not with a network that
only infers."""
import numpy as np
import pytest
import torch

from stroemung_amd.learned import PressureNet
from tests.test_learned import _gpu_ctx, _inputs

pytestmark = pytest.mark.gpu

# 32 frames of 64 x 64: dw_partials over the layers come to 87 MB
H, W, NB = 64, 64, 32
MOST = 64 << 20


def _free():
    return torch.cuda.mem_get_info(0)[0]


@pytest.mark.parametrize("first", ["gradients", "reserve", "benchmark"])
def test_gradient_partials_come_with_the_first_call_that_needs_them(first):
    print("test: network memory", first, flush=True)
    ctx = _gpu_ctx()
    net = PressureNet(ctx, H, W, NB, seed=1)
    x, t = _inputs(NB, H, W, 3)
    net.forward(x)
    net.forward(x)
    before = _free()
    net.forward(x)
    assert before - _free() < MOST // 4
    if first == "gradients":
        net.gradients(x, t)
    elif first == "reserve":
        net.reserve(1)
    else:
        net.benchmark(NB, 1)
    after = _free()
    assert before - after > MOST
    want = net.gradients(x, t)
    got = net.gradients(x, t)
    assert after - _free() < MOST // 4
    assert want[0] == got[0] and np.array_equal(want[1], got[1])
    net.close()
    ctx.close()
