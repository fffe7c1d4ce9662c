"""A lexicographic solve with a limit of no sweeps leaves the pressure as it is,
ghosts included, in a channel of each instance, alone and after other solves."""
import numpy as np
import pytest

from stroemung_amd import presets
from stroemung_amd.simulation import Context
from tests.gridgen import random_fields
from tests.refdata import assert_bits_equal
from tests.test_gpu_lex import KW, _params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny", [9, 40, 60, 90, 120, 180, 240, 400, 600])
def test_a_solve_without_sweeps(ny):
    print("lex no sweeps", ny, flush=True)
    ct, vel = presets.lid_cavity(18, ny - 2)
    p = random_fields(ny, ct.shape)[2]
    p[3, 3] = np.nan
    ctx = Context(0)
    ctx.add_grid(_params(dict(KW, max_iterations=0)), ct, vel)
    for last in (0, 1, 9):
        if last:
            ctx.set_params(0, _params(dict(KW, max_iterations=last)))
            ctx.stage("solve_pressure")
            ctx.set_params(0, _params(dict(KW, max_iterations=0)))
        ctx.upload(0, p=p)
        ctx.stage("solve_pressure")
        st = ctx.state(0)
        assert (st["sor_iterations"], st["norm_squared"], bool(st["exhausted"])) == (0, 0.0, True)
        assert_bits_equal(ctx.download(0)["p"], p, "p")
    ctx.close()
