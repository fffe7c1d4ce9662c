"""Fields carried to the device and back, exactly: the smallest grids,
sizes on both sides of the staged upload's and the threaded download's limits,
downloads of several chunks with a short last one, rows that do not fit the
staging buffer, some of the fields only, and a channel between two others."""
import numpy as np
import pytest

from stroemung_amd import io as sio
from stroemung_amd import presets
from stroemung_amd.simulation import Context, make_params
from tests.refdata import assert_bits_equal

pytestmark = pytest.mark.gpu

ALL = ("u", "v", "p", "f", "g", "rhs")
PRM = (0.1, 0.1, 0.01, 0.9, 100.0, 1e-9, 10, 1.7, 0.0)


def _round_trip(nx, ny, names):
    rng = np.random.default_rng(nx * 1000 + ny)
    ctx = Context(0)
    other, vel = presets.square_obstacle(40, 30)
    ct = np.full((nx, ny), sio.NOSLIP, dtype=np.uint8)
    ct[1:-1, 1:-1] = sio.FLUID
    chans = [(other, vel), (ct, np.zeros((nx, ny, 2))), (other, vel)]
    for c, w in chans:
        ctx.add_grid(make_params(*PRM), c, w)
    want = []
    for ch, (c, _) in enumerate(chans):
        want.append({k: rng.standard_normal(c.shape) for k in ALL})
        ctx.upload(ch, **want[ch])
    new = {k: rng.standard_normal((nx, ny)) for k in names}
    ctx.upload(1, **new)
    want[1].update(new)
    for ch in (1, 0, 2):
        for fields in (ALL, names):
            got = ctx.download(ch, fields)
            for k in fields:
                assert_bits_equal(got[k], want[ch][k], "%s of channel %d" % (k, ch))
    ctx.close()


@pytest.mark.parametrize("nx,ny,names", [
    (3, 3, ALL), (3, 7, ("p",)), (9, 3, ("u", "rhs")), (33, 31, ("v", "p", "g")),
    (104, 105, ("u", "v", "p")), (105, 105, ("u", "v", "p")),        # 256 KB in three fields
    (511, 256, ("p",)), (513, 256, ("p",)), (149, 147, ALL),         # 1 MB
    (511, 512, ("p",)), (513, 512, ("p",)), (211, 207, ALL),         # 2 MB
    (1031, 1027, ("p",)), (701, 1499, ("u", "v", "p")), (13, 60001, ALL),
    (3, 87000, ALL), (3, 88000, ALL), (3, 530000, ("f",)),           # rows of over 4 MB
])
def test_fields_come_back_as_they_went(nx, ny, names):
    print("test: transfer", nx, ny, names, flush=True)
    _round_trip(nx, ny, names)
