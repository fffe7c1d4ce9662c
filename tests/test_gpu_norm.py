"""The initial norm, bit for bit the oracle's sequential sum: one term, the
sizes around a block (16 terms), two blocks and a segment (512), several
segments with and without a remainder, and channels of different sizes at once,
one of which carries its norm already."""
import numpy as np
import pytest

from oracle import pyoracle as O
from stroemung_amd.simulation import Context, make_params
from tests.gridgen import random_fields
from stroemung_amd import presets

pytestmark = pytest.mark.gpu

# interior sizes: their products are 1, 15 .. 17, 31 .. 33, 511 .. 513, ...
INNER = [(1, 1), (1, 15), (4, 4), (17, 1), (1, 31), (2, 16), (3, 11), (7, 73), (16, 32), (27, 19),
         (32, 32), (25, 41), (31, 33), (60, 60), (97, 101)]


def _norm(ct, vel, fields, **kw):
    s = O.Sim(ct, vel, delx=0.1, dely=0.07, delt=0.0, gamma=0.9, reynolds=100.0,
              sor_absolute_epsilon=1e-3, max_iterations=10, omega=1.7, **kw)
    for n, a in zip(("u", "v", "p"), fields):
        getattr(s, n)[...] = a
    s.construct()
    return s.s.initial_norm_squared


def test_initial_norm_of_channels_at_the_block_edges():
    ctx = Context(0)
    want = []
    for i, (a, b) in enumerate(INNER):
        ct, vel = presets.lid_cavity(a, b)
        given = 3.5 if i == 4 else None
        ctx.add_grid(make_params(0.1, 0.07, 0.0, 0.9, 100.0, 1e-3, 10, 1.7, given), ct, vel)
        f = random_fields(i, ct.shape)
        want.append((f, _norm(ct, vel, f) if given is None else given))
    for c, (f, _) in enumerate(want):
        ctx.upload(c, u=f[0], v=f[1], p=f[2])
    ctx.construct()
    got = [ctx.state(c)["initial_norm_squared"] for c in range(len(INNER))]
    assert got == [w for _, w in want]
    ctx.close()
