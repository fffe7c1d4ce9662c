"""The blocked red-black sweeps, bit for bit against the oracle, at the grid
sides where a variant's tiling changes: the largest single tile, the smallest
pair of tiles, the largest pair, the smallest three; with walls at odd and even
sides, obstacles across the tiles, ghosts that are stale at the start, and a
last launch of fewer sweeps than the others."""
import numpy as np
import pytest

from oracle import pyoracle as O
from stroemung_amd import presets
from stroemung_amd.simulation import Context, make_params
from tests.gridgen import mixed_grid, random_fields
from tests.refdata import assert_bits_equal

pytestmark = pytest.mark.gpu

# variant: (sweeps per launch, region's rows, region's pairs * 2)
REGIONS = [(1, 32, 128), (2, 32, 128), (4, 48, 128), (4, 32, 128), (4, 80, 128), (6, 80, 128),
           (8, 80, 128), (6, 72, 128), (8, 96, 128), (6, 96, 96)]


def _sides(region, halo):
    """The largest and smallest sides with 1 | 2 and 2 | 3 parts."""
    one, two = region - 3, 2 * region - 3 - 2 * halo
    return [one, one + 1, two, two + 1]


def _check(variant, ct, vel, seed):
    k = REGIONS[variant][0]
    n = 2 * k + 1
    fields = random_fields(seed, ct.shape)
    kw = dict(delx=0.3, dely=0.2, delt=0.01, gamma=0.9, reynolds=100.0,
              sor_absolute_epsilon=1e-6, max_iterations=50, omega=1.7)
    ctx = Context(0)
    ch = ctx.add_grid(make_params(*[kw[x] for x in ("delx", "dely", "delt", "gamma", "reynolds",
                                                    "sor_absolute_epsilon", "max_iterations",
                                                    "omega")], solver="rb", check_every=0),
                      ct, vel)
    ctx.upload(ch, **dict(zip(("u", "v", "p", "f", "g", "rhs"), fields)))
    assert ctx.solver_variant(variant)[:2] == (variant, k)
    ctx.stage("rb_sweeps", n)
    o = O.Sim(ct, vel, solver=O.SOLVER_RB, **kw)
    for name, a in zip(("u", "v", "p", "f", "g", "rhs"), fields):
        getattr(o, name)[...] = a
    assert o.call("rebuild_boundary_list") == 0
    o.set(rhs_mean=ctx.state(ch)["rhs_mean"])
    o.call("rb_sweeps", n)
    assert_bits_equal(ctx.download(ch, ("p",))["p"], o.p, "variant %d, %s" % (variant, ct.shape))
    ctx.close()


@pytest.mark.parametrize("variant", range(len(REGIONS)))
def test_sweeps_at_the_sides_where_the_tiling_changes(variant):
    k, ex, ey = REGIONS[variant]
    halo = 2 * k + 2
    for i, (nx, ny) in enumerate(zip(_sides(ex, halo), _sides(ey, halo))):
        print("test: sweeps", variant, nx, ny, flush=True)
        _check(variant, *mixed_grid(40 + i, nx, ny), seed=i)
        _check(variant, *presets.lid_cavity(nx - 2, ny - 2), seed=i)


@pytest.mark.parametrize("variant", range(len(REGIONS)))
def test_sweeps_on_narrow_grids(variant):
    for i, (nx, ny) in enumerate([(3, 200), (4, 131), (200, 3), (133, 4), (5, 5)]):
        print("test: sweeps", variant, nx, ny, flush=True)
        _check(variant, *presets.lid_cavity(nx - 2, ny - 2), seed=i)
