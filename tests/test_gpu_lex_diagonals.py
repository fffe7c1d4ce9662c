"""Lexicographic solves on the grids whose longest diagonals are about a wave
long (64 cells), begun in LDS by the kernel for solves that end early: square
interiors of 64 and 65 cells a side and what lies around them."""
import numpy as np
import pytest

from stroemung_amd.simulation import Context
from tests.gridgen import mixed_grid, random_fields
from tests.refdata import assert_bits_equal
from tests.test_gpu_lex import KW, _params, _sim

pytestmark = pytest.mark.gpu

NAMES = ("u", "v", "p", "f", "g", "rhs")


@pytest.mark.parametrize("nx,ny", [(66, 66), (66, 69), (69, 66), (67, 67), (67, 68), (68, 67)])
def test_diagonals_of_64_and_65_cells_after_a_solve_of_one_sweep(nx, ny):
    print("lex diagonal", nx, ny, flush=True)
    ct, vel = mixed_grid(9, nx, ny, n_rect=2)
    f = random_fields(13, ct.shape)
    always = dict(KW, initial_norm_squared=1e300)
    norms = [_sim(ct, vel, f, **dict(KW, max_iterations=j)).solve()[1] for j in (1, 2)]
    cases = [dict(KW, initial_norm_squared=float(np.nextafter(n, np.inf))) for n in norms]
    cases += [dict(KW, max_iterations=m) for m in (1, 2, 3, 20)]
    for kw in cases:
        ctx = Context(0)
        ctx.add_grid(_params(always), ct, vel)
        for rep in range(2):
            ctx.upload(0, **dict(zip(NAMES, f)))
            ctx.stage("solve_pressure")
            if rep == 0:
                assert ctx.state(0)["sor_iterations"] == 1
                ctx.set_params(0, _params(kw))
        s = _sim(ct, vel, f, **kw)
        it, n2 = s.solve()
        st = ctx.state(0)
        assert (st["sor_iterations"], st["norm_squared"]) == (it, n2), kw
        assert_bits_equal(ctx.download(0)["p"], s.p, "p of %s" % (ct.shape,))
        ctx.close()
