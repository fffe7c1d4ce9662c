"""The scratch of the pipelined lexicographic solve: none for red-black channels,
one made when such a channel becomes lexicographic, and at most half of the free
memory -- beyond that the channels are solved in their fields, with the same bits,
also where a diagonal has more cells than a wave lanes."""
import pytest
import torch

from stroemung_amd import presets
from stroemung_amd.simulation import Context, make_params
from tests.gridgen import mixed_grid, random_fields
from tests.refdata import assert_bits_equal
from tests.test_gpu_lex import KW, _params, _sim

pytestmark = pytest.mark.gpu

NAMES = ("u", "v", "p", "f", "g", "rhs")
GB = 1 << 30


def _free():
    return torch.cuda.mem_get_info(0)[0]


def _rb_params():
    return make_params(0.1, 0.07, 0.005, 0.9, 100.0, 1e-9, 4, 1.7, 0.0, solver="rb")


def _check(ctx, ch, ct, vel, f, kw):
    s = _sim(ct, vel, f, **kw)
    it, n2 = s.solve()
    st = ctx.state(ch)
    assert (st["sor_iterations"], st["norm_squared"]) == (it, n2), (ct.shape, kw)
    assert_bits_equal(ctx.download(ch)["p"], s.p, "p of %s" % (ct.shape,))


def test_red_black_channels_take_none_until_they_become_lexicographic():
    print("lex scratch: red-black channels", flush=True)
    ct, vel = mixed_grid(3, 30, 20)
    wide = presets.empty((3, 512))     # 18 MB of scratch if it were lexicographic
    ctx = Context(0)
    ctx.add_grid(_params(KW), ct, vel)
    for _ in range(200):
        ctx.add_grid(_rb_params(), *wide)
    f, fw = random_fields(4, ct.shape), random_fields(5, wide[0].shape)
    ctx.upload(0, **dict(zip(NAMES, f)))
    before = _free()
    ctx.stage("solve_pressure")
    assert before - _free() < GB // 2
    _check(ctx, 0, ct, vel, f, KW)
    for ch in (200, 77):               # one after the other; the first keeps its part
        ctx.set_params(ch, _params(KW))
        for c in (0, 77, 200):
            ctx.upload(c, **dict(zip(NAMES, fw if c else f)))
        ctx.stage("solve_pressure")
        _check(ctx, 0, ct, vel, f, KW)
        _check(ctx, ch, *wide, fw, KW)
    ctx.set_params(200, _rb_params())  # and back, and once more
    ctx.stage("solve_pressure")
    ctx.set_params(200, _params(KW))
    ctx.upload(200, **dict(zip(NAMES, fw)))
    ctx.stage("solve_pressure")
    _check(ctx, 200, *wide, fw, KW)
    ctx.close()


def test_channels_whose_scratch_is_more_than_half_the_memory():
    print("lex scratch: more than half", flush=True)
    torch.cuda.mem_get_info(0)
    wide = presets.empty((3, 512))
    n = torch.cuda.mem_get_info(0)[1] // 2 // (17 * 1024 * 1024) + 1
    ctx = Context(0)
    grids = [mixed_grid(9, nx, ny, n_rect=2) for nx, ny in
             ((66, 66), (67, 67), (67, 68), (68, 67), (90, 40), (100, 80))]
    kws = [dict(KW, max_iterations=m) for m in (5, 1, 2, 3, 7, 4)]
    for (ct, vel), kw in zip(grids, kws):
        ctx.add_grid(_params(kw), ct, vel)
    for _ in range(n):
        ctx.add_grid(_params(dict(KW, max_iterations=1)), *wide)
    fields = [random_fields(20 + c, ct.shape) for c, (ct, _) in enumerate(grids)]
    for c, f in enumerate(fields):
        ctx.upload(c, **dict(zip(NAMES, f)))
    before = _free()
    ctx.stage("solve_pressure")
    assert before - _free() < GB // 2
    for c, ((ct, vel), f, kw) in enumerate(zip(grids, fields, kws)):
        _check(ctx, c, ct, vel, f, kw)
    ctx.close()
