"""Solves that are begun one sweep at a time because the channel's last one was
short (or its limit is): in the fields for channels with four and eight rows to a
lane, on both sides of the sizes where that ends.  They end there, at a sweep or at
the limit, or go on in the pipelined form; alone and beside another channel, and in long channels whose pressure falls off to
nothing."""
import numpy as np
import pytest

from stroemung_amd import presets
from stroemung_amd.simulation import Context
from tests.gridgen import mixed_grid, random_fields
from tests.refdata import assert_bits_equal
from tests.test_gpu_lex import KW, _params, _sim

pytestmark = pytest.mark.gpu

NAMES = ("u", "v", "p", "f", "g", "rhs")


def _compare(ctx, ch, ct, vel, f, kw):
    s = _sim(ct, vel, f, **kw)
    it, n2 = s.solve()
    st = ctx.state(ch)
    assert (st["sor_iterations"], st["norm_squared"]) == (it, n2), (ct.shape, kw)
    assert_bits_equal(ctx.download(ch)["p"], s.p, "p of %s" % (ct.shape,))


@pytest.mark.parametrize("nx,ny", [(77, 60), (216, 64), (217, 64), (97, 48), (60, 112), (48, 97),
                                   (60, 176), (50, 96), (30, 193), (54, 256), (55, 256), (18, 257),
                                   (9, 512), (30, 300)])
def test_solves_expected_to_be_short(nx, ny):
    print("lex begin", nx, ny, flush=True)
    ct, vel = mixed_grid(5, nx, ny) if min(nx, ny) > 10 else presets.lid_cavity(nx - 2, ny - 2)
    f = random_fields(11, ct.shape)
    norms = [_sim(ct, vel, f, **dict(KW, max_iterations=j)).solve()[1] for j in range(1, 6)]
    ends = [dict(KW, initial_norm_squared=float(np.nextafter(n, np.inf))) for n in norms]
    limits = [dict(KW, max_iterations=m) for m in (1, 2, 3, 20)]
    other = mixed_grid(6, 50, 60)
    of = random_fields(12, other[0].shape)
    for first in ends[:2]:                 # the last solve took one sweep, or two
        for kw in [ends[0], ends[1], ends[2], ends[4]] + limits:
            ctx = Context(0)
            ctx.add_grid(_params(first), ct, vel)
            ctx.add_grid(_params(KW), *other)
            for rep in range(2):
                ctx.upload(0, **dict(zip(NAMES, f)))
                ctx.upload(1, **dict(zip(NAMES, of)))
                ctx.stage("solve_pressure")
                if rep == 0:
                    _compare(ctx, 0, ct, vel, f, first)
                    ctx.set_params(0, _params(kw))
            _compare(ctx, 0, ct, vel, f, kw)
            _compare(ctx, 1, *other, of, KW)
            ctx.close()


@pytest.mark.parametrize("nx,ny", [(77, 60), (10, 512), (40, 30), (60, 80)])
def test_solves_of_a_short_limit_one_after_the_other(nx, ny):
    print("lex short limits", nx, ny, flush=True)
    ct, vel = mixed_grid(8, nx, ny) if min(nx, ny) > 10 else presets.lid_cavity(nx - 2, ny - 2)
    f = random_fields(14, ct.shape)
    for m in (1, 2):
        kw = dict(KW, max_iterations=m)
        ctx = Context(0)
        ctx.add_grid(_params(kw), ct, vel)
        ctx.upload(0, **dict(zip(NAMES, f)))
        s = _sim(ct, vel, f, **kw)
        for _ in range(3):
            ctx.stage("solve_pressure")
            it, n2 = s.solve()
            st = ctx.state(0)
            assert (st["sor_iterations"], st["norm_squared"]) == (it, n2), m
            assert_bits_equal(ctx.download(0)["p"], s.p, "p of %s" % (ct.shape,))
        ctx.close()


@pytest.mark.parametrize("nx,ny", [(700, 12), (768, 40), (600, 64)])
def test_short_solves_where_the_pressure_falls_off_to_nothing(nx, ny):
    """Solve after solve of one sweep from p = 0 with a source at one end (the
    values far from it are below the bounds of the pipelined form's quotient), and
    then without any: each of them the oracle's."""
    print("lex decay", nx, ny, flush=True)
    ct, vel = presets.lid_cavity(nx - 2, ny - 2)
    p, rhs = np.zeros(ct.shape), np.zeros(ct.shape)
    rhs[2, 3] = -40.0
    kw = dict(KW, initial_norm_squared=1e300, omega=0.6)
    ctx = Context(0)
    ctx.add_grid(_params(kw), ct, vel)
    f = [np.zeros(ct.shape) for _ in range(6)]
    f[5][...] = rhs
    for source in (rhs, np.ones(ct.shape)):
        ctx.upload(0, p=p, rhs=source)
        f[2][...] = 0.0
        f[5][...] = source
        s = _sim(ct, vel, f, **kw)
        for k in range(20):
            ctx.stage("solve_pressure")
            it, n2 = s.solve()
            st = ctx.state(0)
            assert (st["sor_iterations"], st["norm_squared"]) == (it, n2), k
            assert_bits_equal(ctx.download(0)["p"], s.p, "p after solve %d" % k)
    ctx.close()
