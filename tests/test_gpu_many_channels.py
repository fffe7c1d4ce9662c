"""More channels than a grid has blocks in y (65536): construction and a
lexicographic solve of the first, the last and one in between, bit for bit the
oracle's."""
import pytest

from oracle import pyoracle as O
from stroemung_amd import presets
from stroemung_amd.simulation import Context, make_params
from tests.gridgen import random_fields
from tests.refdata import assert_bits_equal

pytestmark = pytest.mark.gpu

KW = dict(delx=0.1, dely=0.07, delt=0.005, gamma=0.9, reynolds=100.0, sor_absolute_epsilon=1e-9,
          max_iterations=3, omega=1.7)
CHANNELS = 65536 + 70


def test_channels_beyond_the_blocks_of_a_grid_in_y():
    print("test: many channels", flush=True)
    ct, vel = presets.lid_cavity(3, 2)
    prm = make_params(*KW.values(), None, solver="lex")
    ctx = Context(0)
    for _ in range(CHANNELS):
        ctx.add_grid(prm, ct, vel)
    some = (0, 65535, 65536, CHANNELS - 1)
    fields = {c: random_fields(i, ct.shape) for i, c in enumerate(some)}
    for c in some:
        u, v, p, _, _, _ = fields[c]
        ctx.upload(c, u=u, v=v, p=p)
    ctx.construct()
    oracles = {}
    for c in some:
        s = oracles[c] = O.Sim(ct, vel, **KW)
        for n, a in zip(("u", "v", "p"), fields[c]):
            getattr(s, n)[...] = a
        s.construct()
        assert ctx.state(c)["initial_norm_squared"] == s.s.initial_norm_squared, c
        rhs = fields[c][5]
        s.rhs[...] = rhs
        ctx.upload(c, rhs=rhs)
    ctx.stage("solve_pressure")
    for c in some:
        it, n2 = oracles[c].solve()
        st = ctx.state(c)
        assert (st["sor_iterations"], st["norm_squared"]) == (it, n2), c
        assert_bits_equal(ctx.download(c)["p"], oracles[c].p, "p of channel %d" % c)
    ctx.close()
