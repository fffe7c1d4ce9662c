"""The solve's statistics of small channels (one workgroup for all of a channel)
against the kernels of the general path, bit for bit: the same channel alone and
beside one of more than 256 tiles, which sends both the general way; one tile,
one row of tiles, 255, 256 and 257 tiles, sides that are no multiple of a tile."""
import numpy as np
import pytest

from stroemung_amd import presets
from stroemung_amd.simulation import Context, make_params
from tests.gridgen import mixed_grid, random_fields

pytestmark = pytest.mark.gpu


def _params(solver):
    return make_params(0.1, 0.07, 0.005, 0.9, 100.0, 1e-3, 4, 1.7, 0.0, solver=solver,
                       check_every=1 if solver == "lex" else 0)


@pytest.mark.parametrize("solver", ["rb", "lex"])
@pytest.mark.parametrize("nx,ny", [(3, 3), (4, 64), (5, 65), (9, 200), (130, 17), (64, 1020),
                                   (1020, 64), (340, 190), (1028, 40)])
def test_statistics_do_not_depend_on_the_path(nx, ny, solver):
    print("test: statistics", nx, ny, solver, flush=True)
    tiles = -(-nx // 4) * -(-ny // 64)
    grids = [mixed_grid(7, nx, ny) if min(nx, ny) > 8 else presets.lid_cavity(nx - 2, ny - 2)]
    got = []
    for extra in ([], [presets.lid_cavity(1100, 10)]):   # 276 tiles
        ctx = Context(0)
        for ct, vel in grids + extra:
            ctx.add_grid(_params(solver), ct, vel)
        f = random_fields(3, (nx, ny))
        ctx.upload(0, **dict(zip(("u", "v", "p", "f", "g", "rhs"), f)))
        ctx.stage("solve_pressure")
        s = ctx.state(0)
        got.append((s["rhs_mean"], s["tolerance_squared"], s["sor_iterations"], s["exhausted"],
                    ctx.download(0, ("p",))["p"].tobytes()))
        ctx.close()
    assert got[0] == got[1], tiles
