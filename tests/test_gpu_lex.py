"""The lexicographic solve with several sweeps in flight, bit for bit against
the oracle's one-by-one sweeps: the sizes on either side of each of its
instances, solves that end inside a batch of sweeps, values outside the fixed
quotient's bounds, and batches of channels of different instances."""
import numpy as np
import pytest

from oracle import pyoracle as O
from stroemung_amd import presets
from stroemung_amd.simulation import Context, make_params
from tests.gridgen import mixed_grid, random_fields
from tests.refdata import assert_bits_equal

pytestmark = pytest.mark.gpu

KW = dict(delx=0.1, dely=0.07, delt=0.005, gamma=0.9, reynolds=100.0, sor_absolute_epsilon=1e-9,
          max_iterations=40, omega=1.7, initial_norm_squared=0.0)


def _sim(ct, vel, fields, **kw):
    s = O.Sim(ct, vel, **kw)
    for n, a in zip(("u", "v", "p", "f", "g", "rhs"), fields):
        getattr(s, n)[...] = a
    O.lib()
    s.call("rebuild_boundary_list")
    return s


def _params(kw):
    return make_params(kw["delx"], kw["dely"], kw["delt"], kw["gamma"], kw["reynolds"],
                       kw["sor_absolute_epsilon"], kw["max_iterations"], kw["omega"],
                       kw["initial_norm_squared"])


def _solve_both(grids):
    """One stm_solve_pressure of all grids on the GPU, each alone on the oracle."""
    ctx = Context(0)
    for ct, vel, _, kw in grids:
        ctx.add_grid(_params(kw), ct, vel)
    for c, (_, _, f, _) in enumerate(grids):
        ctx.upload(c, **dict(zip(("u", "v", "p", "f", "g", "rhs"), f)))
    ctx.stage("solve_pressure")
    out = []
    for c, (ct, vel, f, kw) in enumerate(grids):
        s = _sim(ct, vel, f, **kw)
        it, n2 = s.solve()
        st = ctx.state(c)
        got = ctx.download(c)["p"]
        assert (st["sor_iterations"], st["norm_squared"]) == (it, n2), (ct.shape, kw)
        met = it > 0 and (n2 < kw["initial_norm_squared"] or n2 < kw["sor_absolute_epsilon"] ** 2)
        assert bool(st["exhausted"]) == (not met)
        assert_bits_equal(got, s.p, "p of %s" % (ct.shape,))
        out.append(it)
    ctx.close()
    return out


@pytest.mark.parametrize("nx,ny", [(3, 3), (4, 3), (3, 9), (9, 4), (50, 24), (31, 25), (40, 31),
                                   (33, 32), (20, 33), (90, 48), (22, 49), (17, 63), (12, 64),
                                   (130, 65), (60, 96), (31, 97), (70, 128), (40, 129), (25, 192),
                                   (13, 193), (14, 256), (24, 257), (11, 512), (12, 513), (8, 560)])
def test_sizes_at_the_edges_of_the_instances(nx, ny):
    print("lex size", nx, ny, flush=True)
    ct, vel = mixed_grid(nx * 1000 + ny, nx, ny) if min(nx, ny) > 10 else presets.simple_inflow((nx, ny))
    _solve_both([(ct, vel, random_fields(nx + ny, ct.shape), KW)])


@pytest.mark.parametrize("itermax", [0, 1, 2, 3, 15, 16, 17, 33, 100])
def test_iteration_limits(itermax):
    print("lex itermax", itermax, flush=True)
    ct, vel = mixed_grid(5, 44, 27)
    _solve_both([(ct, vel, random_fields(3, ct.shape), dict(KW, max_iterations=itermax))])


def test_a_solve_may_end_at_any_sweep_of_a_batch():
    """Ticks of one context: each solve's first batch has the length of the
    solve before, and the bound is moved so that a solve ends at sweep 1, 2,
    ... of its batches (the oracle's norms say where)."""
    print("lex stop positions", flush=True)
    ct, vel = mixed_grid(11, 50, 30)
    f = random_fields(8, ct.shape)
    norms = []
    for k in range(1, 41):
        s = _sim(ct, vel, f, **dict(KW, max_iterations=k))
        norms.append(s.solve()[1])
    assert all(a > b for a, b in zip(norms, norms[1:]))
    ends = []
    for k in range(0, 40, 3):
        # ends at sweep k + 1; two grids, the second ending one sweep later
        grids = [(ct, vel, f, dict(KW, initial_norm_squared=np.nextafter(norms[j], np.inf)))
                 for j in (k, min(k + 1, 39))]
        ends += _solve_both(grids)[:1]
    assert ends == list(range(1, 41, 3))


@pytest.mark.parametrize("nx,ny", [(4, 3), (30, 20), (26, 47), (24, 100), (14, 150), (12, 300)])
def test_solves_that_come_to_end_early(nx, ny):
    """Solve after solve of one equation: the first run to their limit, the
    later ones meet the rule sooner and sooner, down to the first sweep."""
    print("lex converging", nx, ny, flush=True)
    ct, vel = mixed_grid(31, nx, ny) if min(nx, ny) > 10 else presets.simple_inflow((nx, ny))
    f = random_fields(9, ct.shape)
    s = _sim(ct, vel, f, **dict(KW, max_iterations=4000))
    s.solve()                            # a right-hand side the equation can meet:
    p = s.p.copy()                       # that of a pressure the sweeps can reach
    inner = ct[1:-1, 1:-1] == 0
    f[5][...] = 0.0
    s.call("copy_pressure_to_boundaries")
    p = s.p
    f[5][1:-1, 1:-1] = np.where(inner, (p[2:, 1:-1] - 2 * p[1:-1, 1:-1] + p[:-2, 1:-1]) / KW["delx"] ** 2
                                + (p[1:-1, 2:] - 2 * p[1:-1, 1:-1] + p[1:-1, :-2]) / KW["dely"] ** 2, 0.0)
    # the unmasked norm keeps the boundary cells' share; the bound is set
    # between the norms of a long solve and of its end
    s = _sim(ct, vel, f, **dict(KW, max_iterations=100))
    norms = [s.solve()[1] for _ in range(60)]
    bound = norms[40]
    kw = dict(KW, max_iterations=100, initial_norm_squared=float(bound))
    s = _sim(ct, vel, f, **kw)
    ctx = Context(0)
    ctx.add_grid(_params(kw), ct, vel)
    ctx.upload(0, p=f[2], rhs=f[5])
    seen = []
    for k in range(46):
        ctx.stage("solve_pressure")
        it, n2 = s.solve()
        st = ctx.state(0)
        assert (st["sor_iterations"], st["norm_squared"]) == (it, n2), k
        assert_bits_equal(ctx.download(0)["p"], s.p, "p after solve %d" % k)
        seen.append(it)
    ctx.close()
    print(seen, flush=True)


@pytest.mark.parametrize("last", [1, 5, 16, 40])
def test_the_length_of_the_last_solve_changes_nothing(last):
    print("lex last length", last, flush=True)
    ct, vel = mixed_grid(12, 39, 22)
    f, g = random_fields(1, ct.shape), random_fields(2, ct.shape)
    ctx = Context(0)
    ctx.add_grid(_params(dict(KW, max_iterations=last)), ct, vel)
    ctx.upload(0, p=f[2], rhs=f[5])
    ctx.stage("solve_pressure")
    assert ctx.state(0)["sor_iterations"] == last
    ctx.set_params(0, _params(dict(KW, max_iterations=23)))
    ctx.upload(0, p=g[2], rhs=g[5])
    ctx.stage("solve_pressure")
    s = _sim(ct, vel, g, **dict(KW, max_iterations=23))
    it, n2 = s.solve()
    st = ctx.state(0)
    assert (st["sor_iterations"], st["norm_squared"]) == (it, n2)
    assert_bits_equal(ctx.download(0)["p"], s.p, "p")
    ctx.close()


@pytest.mark.parametrize("what", ["zero", "minus_zero", "tiny", "denormal", "huge", "mixed",
                                  "decay", "wide_cells", "inf", "nan"])
def test_values_outside_the_bounds_of_the_fixed_quotient(what):
    print("lex values", what, flush=True)
    ct, vel = mixed_grid(21, 42, 26)
    f = random_fields(4, ct.shape)
    kw = dict(KW, max_iterations=21)
    p, rhs = f[2], f[5]
    if what in ("zero", "minus_zero"):
        p[...] = -0.0 if what == "minus_zero" else 0.0
        rhs[...] = p
    elif what == "tiny":
        p *= 1e-300
        rhs *= 1e-300
    elif what == "denormal":
        p *= 1e-312
        rhs *= 1e-312
    elif what == "huge":
        p *= 1e290
        rhs *= 1e290
    elif what == "mixed":
        p[::3] *= 1e-280
        p[1::3] *= 1e270
    elif what == "decay":   # one source: values fall off by orders per cell and sweep
        p[...] = 0.0
        rhs[...] = 0.0
        rhs[5, 5] = 1e-250
    elif what == "wide_cells":
        kw.update(delx=1e-12, dely=3e9)
    elif what == "inf":
        p[20, 13] = np.inf
    else:
        p[20, 13] = np.nan
    if what in ("inf", "nan"):   # the norms are NaN: compared as such
        ctx = Context(0)
        ctx.add_grid(_params(kw), ct, vel)
        ctx.upload(0, p=p, rhs=rhs)
        ctx.stage("solve_pressure")
        s = _sim(ct, vel, f, **kw)
        it, n2 = s.solve()
        got = ctx.download(0)["p"]
        assert ctx.state(0)["sor_iterations"] == it
        assert np.array_equal(np.isnan(got), np.isnan(s.p))
        assert np.array_equal(got[~np.isnan(got)], s.p[~np.isnan(s.p)])
        ctx.close()
        return
    _solve_both([(ct, vel, f, kw)])


def test_fluid_on_the_frame_is_not_swept():
    print("lex frame", flush=True)
    ct, vel = presets.empty((23, 19))
    ct[8:12, 7:11] = 1
    _solve_both([(ct, vel, random_fields(6, ct.shape), KW)])


def test_a_batch_of_every_instance():
    print("lex batch", flush=True)
    grids = []
    for k, (nx, ny) in enumerate([(30, 20), (25, 50), (64, 100), (16, 200), (13, 400), (12, 600),
                                  (90, 24), (18, 31)]):
        ct, vel = mixed_grid(70 + k, nx, ny)
        grids.append((ct, vel, random_fields(k, ct.shape), dict(KW, max_iterations=10 + 3 * k)))
    _solve_both(grids)


@pytest.mark.parametrize("nx,ny", [(3, 3), (102, 22), (96, 48), (97, 48), (15, 300), (9, 512)])
def test_a_solve_after_one_of_a_single_sweep(nx, ny):
    """The kernel that begins the solve of a channel in LDS after a solve of one
    sweep: the next one ends in it (one or two sweeps, or itermax), or goes on
    elsewhere (three and more), at 4608 cells and just beyond, alone and beside a
    channel whose last solve was long."""
    ct, vel = mixed_grid(5, nx, ny) if min(nx, ny) > 8 else presets.lid_cavity(nx - 2, ny - 2)
    f = random_fields(11, ct.shape)
    fields = dict(zip(("u", "v", "p", "f", "g", "rhs"), f))
    always = dict(KW, initial_norm_squared=1e300)
    norms = [_sim(ct, vel, f, **dict(KW, max_iterations=j)).solve()[1] for j in range(1, 8)]
    cases = [dict(KW, initial_norm_squared=float(np.nextafter(norms[j], np.inf)))
             for j in (0, 1, 2, 6)]
    cases += [dict(KW, max_iterations=m) for m in (1, 2, 3, 37)]
    other = mixed_grid(6, 50, 40)
    of = random_fields(12, other[0].shape)
    for kw in cases:
        ctx = Context(0)
        ctx.add_grid(_params(always), ct, vel)
        ctx.add_grid(_params(KW), *other)
        for rep in range(2):
            ctx.upload(0, **fields)
            ctx.upload(1, **dict(zip(("u", "v", "p", "f", "g", "rhs"), of)))
            ctx.stage("solve_pressure")
            if rep == 0:
                assert ctx.state(0)["sor_iterations"] == 1
                ctx.set_params(0, _params(kw))
        s = _sim(ct, vel, f, **kw)
        it, n2 = s.solve()
        st = ctx.state(0)
        assert (st["sor_iterations"], st["norm_squared"]) == (it, n2), kw
        assert_bits_equal(ctx.download(0)["p"], s.p, "p of %s" % (ct.shape,))
        o = _sim(*other, of, **KW)
        assert (ctx.state(1)["sor_iterations"], ctx.state(1)["norm_squared"]) == o.solve()
        assert_bits_equal(ctx.download(1)["p"], o.p, "the other channel's p")
        ctx.close()
