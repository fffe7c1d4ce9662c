"""What a user of this framework has it do, as cases that can be timed.

Every case goes through the public Python layer (Context, PressureNet), which
is a thin binding of the C ABI, and takes its grids and scalars from the
repository's own presets and workloads.  Kinds:

frame     one simulation in the reference's lexicographic mode, advanced and
          drawn: the GUI's loop (a tick, the image, the fields the user looks at)
lex       lexicographic ticks of one channel or of many together
rb        red-black ticks: the lid cavity, or channels of uneven size
sweeps    a fixed number of red-black sweeps on a large grid
load      a saved state put into a running simulation (scalars, u, v, p) and
          constructed: F, G, the right-hand side and the initial norm
learned   ticks whose solve runs two-grid cycles with the pressure network
forward   the network on a host batch
gradients loss and parameter gradients of a host batch
train     Adam steps on the device-resident training set

Fields are host arrays by the nature of the interface: the library owns the
device memory, and a program uploads a state and reads fields back.
"""
import math

import numpy as np
import torch

from stroemung_amd import presets, workloads
from stroemung_amd.learned import PressureNet
from stroemung_amd.simulation import Context, make_params

FIELDS = ("u", "v", "p")


def listed():
    return [
        # the reference's own case, drawn every tick: the smallest call there is
        {"name": "frame_100x20", "kind": "frame", "imax": 100, "jmax": 20, "iters": 100},
        # an ensemble of small channels (one workgroup each), read back every 8 ticks
        {"name": "lex_256x_100x20", "kind": "lex", "count": 256, "imax": 100, "jmax": 20,
         "iters": 100, "ticks": 8},
        # the reference's solver on a longer, finer channel
        {"name": "lex_400x80", "kind": "lex", "count": 1, "imax": 400, "jmax": 80, "iters": 100,
         "ticks": 1},
        # one ragged channel solved to its residual: a tick is mostly short launches
        {"name": "rb_131x67", "kind": "rb", "count": 1, "imax": 131, "jmax": 67, "eps": 1e-4,
         "iters": 6000, "check": 4, "ticks": 1},
        # the benchmark's cavity with a sweep limit per tick
        {"name": "rb_cavity_1024", "kind": "rb", "count": 0, "imax": 1024, "jmax": 1024,
         "eps": 1e-6, "iters": 12000, "check": 6, "ticks": 1},
        # uneven channels that converge one after another
        {"name": "rb_32_channels", "kind": "rb", "count": 32, "imax": 512, "jmax": 256,
         "eps": 1e-4, "iters": 6000, "check": 8, "ticks": 1},
        # smoothing a grid larger than the last-level cache
        {"name": "sweeps_4000x3000", "kind": "sweeps", "imax": 4000, "jmax": 3000, "n": 2000},
        # restarting a simulation from a stored state
        {"name": "load_1000x501", "kind": "load", "imax": 1000, "jmax": 501},
        # the learned solve on a batch of cavities: 8 cycles of 16 sweeps
        {"name": "learned_32x_256", "kind": "learned", "count": 32, "n": 256, "coarsen": 4,
         "cycles": 8, "sweeps": 16, "step": "momentum", "ticks": 4},
        # the network on the cavities' frame
        {"name": "forward_64x64x32", "kind": "forward", "h": 64, "w": 64, "batch": 32},
        {"name": "gradients_64x64x32", "kind": "gradients", "h": 64, "w": 64, "batch": 32},
        # training on the uneven channels' frame (its deepest level is 8 x 4 pixels)
        {"name": "train_64x32x32", "kind": "train", "h": 64, "w": 32, "batch": 32, "steps": 16},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("frame", "lex", "lex", "rb", "rb", "cavity", "sweeps", "load", "learned",
                       "forward", "gradients", "train"))
    if kind == "frame":
        return {"kind": "frame", "imax": _log(rng, 40, 200), "jmax": _log(rng, 12, 60),
                "iters": rng.choice((60, 100, 150))}
    if kind == "lex":
        jmax = _log(rng, 12, 120)
        imax = min(_log(rng, 2 * jmax, 6 * jmax), 32000 // jmax)
        count = 1 if imax * jmax > 4400 or rng.random() < 0.4 else _log(rng, 2, 256)
        return {"kind": "lex", "count": count, "imax": imax, "jmax": jmax,
                "iters": rng.choice((50, 100)), "ticks": 8 if imax * jmax < 4400 else 1}
    if kind == "rb":
        count = rng.choice((1, 1, 4, 12, 32))
        return {"kind": "rb", "count": count, "imax": _log(rng, 80, 512), "jmax": _log(rng, 40, 256),
                "eps": 1e-4, "iters": rng.choice((3000, 6000)), "check": rng.choice((2, 4, 6, 8)),
                "ticks": 1}
    if kind == "cavity":
        n = _log(rng, 100, 1024)
        return {"kind": "rb", "count": 0, "imax": n, "jmax": max(64, n - rng.randint(0, n // 3)),
                "eps": 1e-6, "iters": rng.choice((4000, 8000)), "check": rng.choice((4, 6, 8)),
                "ticks": 1}
    if kind == "sweeps":
        return {"kind": "sweeps", "imax": _log(rng, 500, 4000), "jmax": _log(rng, 400, 3000),
                "n": rng.randint(500, 1900)}
    if kind == "load":
        return {"kind": "load", "imax": _log(rng, 100, 1000), "jmax": _log(rng, 40, 500)}
    if kind == "learned":
        n = rng.choice((128, 192, 250, 256))
        return {"kind": "learned", "count": rng.randint(4, 32), "n": n,
                "coarsen": rng.choice((2, 4, 4, 8)), "cycles": rng.randint(3, 8),
                "sweeps": rng.choice((8, 16, 16)), "step": rng.choice(("momentum", "energy")),
                "ticks": 4}
    h, w = 8 * rng.randint(2, 12), 8 * rng.randint(2, 12)
    batch = max(1, min(rng.randint(1, 64), 32 * 64 * 64 // (h * w)))
    if kind == "train":
        return {"kind": "train", "h": h, "w": w, "batch": min(batch, 32), "steps": rng.randint(4, 14)}
    return {"kind": kind, "h": h, "w": w, "batch": batch}


# ------------------------------------------------------------------- inputs

def _stream_velocity(g, t, dx, dy, base, amp):
    """A divergence-free swirl (a few modes of a stream function, one scale of
    which is small) over a mean flow `base`, zero where there is no fluid."""
    nx, ny = t.shape
    x = (np.arange(nx + 1) / nx)[:, None]
    y = (np.arange(ny + 1) / ny)[None, :]
    psi = np.zeros((nx + 1, ny + 1))
    for k in range(5):
        a, b = int(g.integers(1, 4 + 3 * k)), int(g.integers(1, 3 + 2 * k))
        psi += (g.normal() / (1 + k) / math.hypot(a, b)) * np.sin(
            math.pi * a * x + g.uniform(0, 6.28)) * np.sin(math.pi * b * y)
    psi *= min(nx * dx, ny * dy)
    u = (psi[1:, 1:] - psi[1:, :-1]) / dy
    v = -(psi[1:, 1:] - psi[:-1, 1:]) / dx
    s = amp / max(1e-12, float(np.abs(u).max()), float(np.abs(v).max()))
    fluid = t == 0
    return np.where(fluid, base + s * u, 0.0), np.where(fluid, s * v, 0.0)


def _pressure(g, t, amp):
    nx, ny = t.shape
    x = ((np.arange(nx) + 0.5) / nx)[:, None]
    y = ((np.arange(ny) + 0.5) / ny)[None, :]
    p = amp * (1.0 - x) + np.zeros((nx, ny))
    for k in range(4):
        p += amp * 0.3 * g.normal() / (k + 1) * np.cos(math.pi * (k + 1) * x + k) * np.cos(
            math.pi * int(g.integers(0, 4)) * y)
    return np.where(t == 0, p, 0.0)


def _fields(g, t, prm, base, amp, pamp):
    u, v = _stream_velocity(g, t, prm.delx, prm.dely, base, amp)
    return {"u": u, "v": v, "p": _pressure(g, t, pamp)}


def _grids(case, seed):
    """[(cell types, wall velocities, params, fields)] of a solver case."""
    g = np.random.default_rng([seed, 17])
    kind = case["kind"]
    out = []
    if kind in ("frame", "lex"):
        count = case.get("count", 1)
        rng = presets.SplitMix64(seed + 1000)
        for k in range(count):
            if count == 1:   # the square obstacle, scaled with the channel
                side = max(4, 2 * (case["jmax"] // 10))
                ct, vel = presets.square_obstacle(case["imax"], case["jmax"], side=side,
                                                  centre=case["imax"] // 5)
            else:
                ct, vel = presets.random_channel(rng, case["imax"], case["jmax"])
            # as a run that started from rest: its initial norm is zero, so
            # a solve ends at eps or after `iters`
            prm = make_params(0.1, 0.1, 0.005, 0.9, 100.0, 1e-3, case["iters"], 1.7,
                              initial_norm_squared=0.0)
            out.append((ct, vel, prm, _fields(g, ct, prm, 1.0, 0.2, 0.5)))
        return out
    if kind == "rb":
        if case["count"] == 0:
            ct, vel = presets.lid_cavity(case["imax"], case["jmax"])
            n = max(case["imax"], case["jmax"])
            prm = make_params(1.0 / n, 1.0 / n, 0.0, 0.9, 1000.0, case["eps"], case["iters"], 1.8,
                              tau=0.5, solver="rb", check_every=case["check"])
            return [(ct, vel, prm, _fields(g, ct, prm, 0.0, 0.5, 0.05))]
        # workloads.random_channels, the sizes a part of the case (not of the seed)
        sizes = presets.SplitMix64(case["imax"] * 1000 + case["jmax"])
        rng = presets.SplitMix64(seed)
        grids = []
        for _ in range(case["count"]):
            ni, nj = case["imax"], case["jmax"]
            if case["count"] > 1:
                ni = presets.log_uniform_int(sizes, 64, ni)
                nj = presets.log_uniform_int(sizes, 32, nj)
            ct, vel = presets.random_channel(rng, ni, nj)
            prm = make_params(1.0 / nj, 1.0 / nj, 0.0, 0.9, 50.0 + 950.0 * rng.uniform(),
                              case["eps"], case["iters"], 1.7, tau=0.5, solver="rb",
                              check_every=case["check"])
            grids.append((ct, vel, prm))
        return [gr + (_fields(g, gr[0], gr[2], 1.0, 0.3, 0.5),) for gr in grids]
    if kind == "sweeps":
        ct, vel = presets.lid_cavity(case["imax"], case["jmax"])
        n = max(case["imax"], case["jmax"])
        prm = make_params(1.0 / n, 1.0 / n, 0.0, 0.9, 1000.0, 1e-6, 10_000_000, 1.8, tau=0.5,
                          solver="rb", check_every=0)
        p = _pressure(g, ct, 0.05)
        rhs = np.where(ct == 0, _pressure(g, ct, 1.0) + 0.1 * g.standard_normal(ct.shape), 0.0)
        return [(ct, vel, prm, {"p": p, "rhs": rhs})]
    if kind == "load":
        ct, vel = presets.random_channel(presets.SplitMix64(seed + 5), case["imax"], case["jmax"])
        h = 1.0 / case["jmax"]
        prm = make_params(h, h, 1e-4, 0.9, 500.0, 1e-3, 100, 1.7)
        return [(ct, vel, prm, _fields(g, ct, prm, 1.0, 0.3, 0.5))]
    if kind == "learned":
        grids = workloads.random_cavities(case["count"], case["n"], seed,
                                          itermax=case["cycles"] * case["sweeps"])
        return [gr + (_fields(g, gr[0], gr[2], 0.0, 0.5, 0.05),) for gr in grids]
    raise ValueError(kind)


# (input channels, output channels) of the network's 3x3 convolutions
CONVS = ((32, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128), (128, 256), (256, 256),
         (384, 128), (128, 128), (192, 64), (64, 64), (96, 32), (32, 32))


def _layout():
    """[(offset of the weights, shape, offset of the biases)], head, total."""
    out, off = [], 0
    for cin, cout in CONVS:
        w = off
        off += cout * 9 * cin
        out.append((w, (cout, 9, cin), off))
        off = (off + cout + 7) // 8 * 8
    return out, off, off + 40


def _weights(seed):
    """He-initialised parameters with small random biases."""
    g = np.random.default_rng([seed, 23])
    lay, head, n = _layout()
    p = np.zeros(n, np.float32)
    for k, (w, (cout, taps, cin), b) in enumerate(lay):
        fan = 9 * (2 if k == 0 else cin)
        a = g.standard_normal((cout, taps, cin)) * math.sqrt(2.0 / fan)
        if k == 0:
            a[:, :, 2:] = 0.0
        p[w:w + a.size] = a.ravel()
        p[b:b + cout] = 0.05 * g.standard_normal(cout)
    p[head:head + 32] = 0.1 * math.sqrt(1.0 / 32) * g.standard_normal(32)
    p[head + 32] = 0.01 * g.standard_normal()
    return p


def _batch(case, seed):
    """Normalised residuals with a fluid fraction, and smooth targets."""
    g = np.random.default_rng([seed, 29])
    nb, h, w = case["batch"], case["h"], case["w"]
    x = np.zeros((nb, h, w, 2), np.float32)
    x[..., 0] = g.standard_normal((nb, h, w))
    x[..., 1] = 1.0
    for b in range(nb):
        i, j = int(g.integers(0, h - 4)), int(g.integers(0, w - 4))
        a, c = int(g.integers(2, max(3, h // 3))), int(g.integers(2, max(3, w // 3)))
        x[b, i:i + a, j:j + c] = 0.0
        x[b, i:i + a, min(j + c, w - 1), 1] = 0.5
    yy = np.linspace(0, 3.0, h)[:, None]
    xx = np.linspace(0, 3.0, w)[None, :]
    t = np.stack([g.normal() * np.cos(yy * g.uniform(0.5, 2)) * np.cos(xx * g.uniform(0.5, 2))
                  + 0.2 * g.normal() for _ in range(nb)]).astype(np.float32)
    return x, t


# ------------------------------------------------------------------ passes

class _State:
    def __init__(self, case):
        self.case = case
        self.ctx = self.net = None

    def __del__(self):
        if self.net is not None:
            self.net.close()
        if self.ctx is not None:
            self.ctx.close()


def prepare(case, seed):
    s = _State(case)
    kind = case["kind"]
    s.ctx = ctx = Context(0)
    if kind in ("forward", "gradients"):
        s.net = PressureNet(ctx, case["h"], case["w"], case["batch"], seed=1)
        s.net.set_params(_weights(seed))
        s.x, s.t = _batch(case, seed)
        return s
    if kind == "train":
        # pairs from the solver, as train_net captures them: channels whose
        # interior fills the frame at coarsening 2
        grids = workloads.random_channels(case["batch"], seed, (2 * case["h"],) * 2,
                                          (2 * case["w"],) * 2, eps=1e-3, itermax=400)
        for ct, vel, prm in grids:
            ctx.add_grid(prm, ct, vel)
        g = np.random.default_rng([seed, 17])
        for k, (ct, vel, prm) in enumerate(grids):
            ctx.upload(k, **_fields(g, ct, prm, 1.0, 0.3, 0.5))
        ctx.construct()
        s.net = PressureNet(ctx, case["h"], case["w"], case["batch"], seed=1)
        s.net.set_params(_weights(seed))
        s.net.reserve(2 * case["batch"])
        ctx.set_capture(s.net, points=2, sweeps=16, coarsen=2)
        ctx.tick()
        ctx.set_capture(None)
        return s
    s.grids = _grids(case, seed)
    for ct, vel, prm, _ in s.grids:
        ctx.add_grid(prm, ct, vel)
    for k, (_, _, _, f) in enumerate(s.grids):
        ctx.upload(k, **f)
    if kind == "sweeps":
        ctx.autotune(8)
        return s
    ctx.construct()
    if kind in ("rb", "learned"):
        # as the benchmark does: tuned after a first tick (the adaptive step
        # has no length before it), then back to the stored state
        ctx.tick()
        for k, (_, _, _, f) in enumerate(s.grids):
            ctx.upload(k, **f)
        ctx.construct()
        ctx.autotune(8)
    if kind == "learned":
        f = case["coarsen"]
        n = -(-case["n"] // f)
        n = (n + 7) // 8 * 8
        s.net = PressureNet(ctx, n, n, case["count"], seed=1)
        s.net.set_params(_weights(seed))
        ctx.set_learned(s.net, cycles=case["cycles"], sweeps=case["sweeps"], step=case["step"],
                        coarsen=f)
        ctx.set_graphs(True)
    return s


def _read(ctx, fields):
    got = [ctx.download(k, fields) for k in range(len(ctx.shapes))]
    return {f: np.concatenate([d[f].ravel() for d in got]) for f in fields}


def run(s):
    case, ctx = s.case, s.ctx
    kind = case["kind"]
    if kind == "forward":
        return {"y": s.net.forward(s.x)}
    if kind == "gradients":
        loss, g = s.net.gradients(s.x, s.t)
        return {"loss": np.float32(loss), "g": g}
    if kind == "train":
        loss = s.net.train(case["steps"], case["batch"], lr=1e-3, seed=7)
        return {"loss": np.float32(loss), "params": s.net.get_params()}
    if kind == "frame":
        its, nrm = ctx.tick()
        return {"image": ctx.render(0, "speed"), "its": its[0], "norm": nrm[0],
                **ctx.download(0, FIELDS)}
    if kind == "sweeps":
        ctx.stage("rb_sweeps", case["n"])
        return ctx.download(0, ("p",))
    if kind == "load":
        ct, vel, prm, f = s.grids[0]
        ctx.set_params(0, prm)
        ctx.upload(0, **f)
        ctx.construct()
        st = ctx.state(0)
        return {"norm": st["initial_norm_squared"], "speed": np.array(st["speed_range"]),
                **ctx.download(0, ("f", "g", "rhs"))}
    if kind == "rb":   # from the stored state, so every pass solves the same problem
        for k, (_, _, _, f) in enumerate(s.grids):
            ctx.upload(k, **f)
    its = nrm = None
    for _ in range(case["ticks"]):
        its, nrm = ctx.tick()
    return {"its": np.array(its), "norm": np.array(nrm), **_read(ctx, FIELDS)}


# -------------------------------------------------------------------- work

def work(case):
    """Fields read and written once per tick and pass; per cell update 8
    operations, per term of a norm 11, about 100 for the other stages."""
    kind = case["kind"]
    if kind in ("forward", "gradients", "train"):
        pix = case["batch"] * case["h"] * case["w"]
        level = (0, 0, 1, 1, 2, 2, 3, 3, 2, 2, 1, 1, 0, 0)
        fl = sum(2.0 * 9 * (2 if k == 0 else ci) * co * pix / 4 ** lv
                 for k, ((ci, co), lv) in enumerate(zip(CONVS, level))) + 64.0 * pix
        n = _layout()[2]
        if kind == "forward":
            return {"bytes": 12.0 * pix + 2.0 * n, "flops": fl}
        if kind == "gradients":
            return {"bytes": 12.0 * pix + 6.0 * n, "flops": 3 * fl}
        return {"bytes": case["steps"] * (8.0 * pix + 28.0 * n), "flops": 3 * fl * case["steps"]}
    if kind == "learned":
        cells = float(case["count"] * case["n"] ** 2 * case["ticks"])
        return {"bytes": 50.0 * cells,
                "flops": cells * (100 + case["cycles"] * (8 * case["sweeps"] + 60))}
    cells = float(case["imax"] * case["jmax"])
    if kind == "frame":
        return {"bytes": 53.0 * cells, "flops": cells * (100 + 19 * case["iters"])}
    if kind == "lex":
        cells *= case["count"] * case["ticks"]
        return {"bytes": 50.0 * cells, "flops": cells * (100 + 19 * case["iters"])}
    if kind == "sweeps":
        return {"bytes": 25.0 * cells, "flops": 8.0 * cells * case["n"]}
    if kind == "load":
        return {"bytes": 65.0 * cells, "flops": 100.0 * cells}
    if case["count"] > 1:   # log-uniform sizes, and channels that converge early
        cells *= 0.3 * case["count"]
    done = case["iters"] * (1.0 if case["count"] == 0 else 0.3)
    return {"bytes": 50.0 * cells, "flops": cells * (100 + 8 * done)}


# ------------------------------------------------ the same values in 64 bits

class _Plain:
    """One tick's stages in NumPy on a stack of equal grids (B, nx, ny)."""

    def __init__(self, grids, device):
        ct = np.stack([g[0] for g in grids])
        self.t, self.vel = ct, np.stack([g[1] for g in grids])
        self.prm = grids[0][2]
        self.re = np.array([g[2].reynolds for g in grids])[:, None, None]
        self.dx = np.array([g[2].delx for g in grids])[:, None, None]
        self.dy = np.array([g[2].dely for g in grids])[:, None, None]
        self.delt = np.array([g[2].delt for g in grids])[:, None, None]
        self.B, self.nx, self.ny = ct.shape
        self.u, self.v, self.p = (np.stack([g[3].get(k, np.zeros(ct.shape[1:])) for g in grids])
                                  for k in FIELDS)
        self.f, self.g, self.rhs = (np.zeros_like(self.p) for _ in range(3))
        self.fl = fl = ct == 0
        pad = np.zeros((self.B, self.nx + 2, self.ny + 2), bool)
        pad[:, 1:-1, 1:-1] = fl
        self.nb = {"n": pad[:, 1:-1, :-2] & ~fl, "s": pad[:, 1:-1, 2:] & ~fl,
                   "w": pad[:, :-2, 1:-1] & ~fl, "e": pad[:, 2:, 1:-1] & ~fl}
        self.device = device
        inner = np.zeros_like(fl)
        inner[:, 1:-1, 1:-1] = True
        self.inner = inner & fl

    def walls(self):
        """The boundary velocities, cell after cell in (x, y) order."""
        self.restore = []
        u, v = self.u, self.v
        for b, x, y in zip(*np.nonzero(~self.fl)):
            n, s, w, e = (self.nb[k][b, x, y] for k in "nswe")
            N, S, W, E, I = (b, x, y - 1), (b, x, y + 1), (b, x - 1, y), (b, x + 1, y), (b, x, y)
            ty = self.t[I]
            if not (n or s or w or e):
                pass
            elif ty == 3:   # outflow
                nu = u[N] if n else u[E] if e and not s else u[E] if e else u[W] if w else u[S]
                nv = v[E] if e and not s else v[S] if s else v[W] if w else v[N]
                u[I], v[I] = nu, nv
            else:
                bu, bv = self.vel[I] if ty in (2, 4) else (0.0, 0.0)
                ku, kv = (2 * bu, 2 * bv) if ty == 4 else (0.0, 0.0)
                if w:
                    u[W] = bu
                if n:
                    if not e or w:
                        u[I] = ku - u[N]
                    v[N] = bv
                if s:
                    if not e:
                        u[I] = ku - u[S]
                    v[I] = bv
                if e:
                    u[I] = bu
                    if not s:
                        v[I] = kv - v[E]
                if w and not s:
                    v[I] = kv - v[W]
            self.restore.append((I, u[W] if w else u[I], v[N] if n else v[I]))

    def fgr(self):
        u, v, dx, dy, re, gm = self.u, self.v, self.dx, self.dy, self.re, self.prm.gamma
        c = (slice(None), slice(1, -1), slice(1, -1))

        def at(a, i, j):
            return a[:, 1 + i:self.nx - 1 + i, 1 + j:self.ny - 1 + j]

        def donor(a, b, p, q, h):   # ((a+b)(p+q)) upwinded differences over 4h
            return ((a[0] * p[0] - b[0] * q[0]) + gm * (abs(a[0]) * p[1] - abs(b[0]) * q[1])) / (4 * h)

        uc, vc = at(u, 0, 0), at(v, 0, 0)
        ue, uw, un, us, usw = at(u, 1, 0), at(u, -1, 0), at(u, 0, -1), at(u, 0, 1), at(u, -1, 1)
        ve, vw, vn, vs, vne = at(v, 1, 0), at(v, -1, 0), at(v, 0, -1), at(v, 0, 1), at(v, 1, -1)
        du2 = donor((uc + ue,), (uw + uc,), (uc + ue, uc - ue), (uw + uc, uw - uc), dx)
        duvy = donor((vc + ve,), (vn + vne,), (uc + us, uc - us), (un + uc, un - uc), dy)
        duvx = donor((uc + us,), (uw + usw,), (vc + ve, vc - ve), (vw + vc, vw - vc), dx)
        dv2 = donor((vc + vs,), (vn + vc,), (vc + vs, vc - vs), (vn + vc, vn - vc), dy)
        lu = (ue - 2 * uc + uw) / dx ** 2 + (us - 2 * uc + un) / dy ** 2
        lv = (ve - 2 * vc + vw) / dx ** 2 + (vs - 2 * vc + vn) / dy ** 2
        self.f[c] = uc + self.delt * (lu / re - du2 - duvy)
        self.g[c] = vc + self.delt * (lv / re - duvx - dv2)
        bnd = ~self.fl
        fw, gn = np.zeros_like(bnd), np.zeros_like(bnd)
        fw[:, :-1] = self.nb["w"][:, 1:]
        gn[:, :, :-1] = self.nb["n"][:, :, 1:]
        self.f = np.where(bnd | fw, u, self.f)
        self.g = np.where(bnd | gn, v, self.g)
        self.rhs[:, 1:, 1:] = ((self.f[:, 1:, 1:] - self.f[:, :-1, 1:]) / dx
                               + (self.g[:, 1:, 1:] - self.g[:, 1:, :-1]) / dy) / self.delt

    def ghost_plan(self):
        """Flat indices of the ghosts and of the two cells each one averages."""
        i = np.arange(self.B * self.nx * self.ny).reshape(self.p.shape)
        n, s, w, e = (self.nb[k] for k in "nswe")
        vert = np.where(n, i - 1, i + 1)
        horz = np.where(e, i + self.ny, i - self.ny)
        any_v, any_h = n | s, e | w
        a, b = np.where(any_v, vert, horz), np.where(any_h, horz, vert)
        k = any_v | any_h
        return i[k], a[k], b[k]

    def norm(self):
        p, r = self.p, np.zeros_like(self.p)
        c = p[:, 1:-1, 1:-1]
        r = ((p[:, 2:, 1:-1] - c) - (c - p[:, :-2, 1:-1])) / self.dx ** 2 + (
            (p[:, 1:-1, 2:] - c) - (c - p[:, 1:-1, :-2])) / self.dy ** 2 - self.rhs[:, 1:-1, 1:-1]
        return (r * r).sum((1, 2)) / self.fl.sum((1, 2))

    def lex(self, iters, eps):
        """Gauss-Seidel in (x, y) order, an anti-diagonal at a time."""
        gi, ga, gb = self.ghost_plan()
        dx2, dy2 = float(self.prm.delx) ** 2, float(self.prm.dely) ** 2
        om = self.prm.omega
        mid = om / (2 / dx2 + 2 / dy2)
        n = self.nx * self.ny
        p, rhs, fl = self.p.reshape(self.B, n), self.rhs.reshape(self.B, n), self.fl.reshape(self.B, n)
        st, ny = self.ny - 1, self.ny
        cuts = []
        for d in range(2, self.nx + self.ny - 3):
            lo, hi = max(1, d - (self.ny - 2)), min(self.nx - 2, d - 1)
            a, m = lo * ny + d - lo, hi - lo + 1
            cuts.append([slice(a + o, a + o + (m - 1) * st + 1, st) for o in (0, ny, -ny, 1, -1)])
        for k in range(iters):
            flat = self.p.reshape(-1)
            flat[gi] = (flat[ga] + flat[gb]) * 0.5
            for c, e, w, s, no in cuts:
                x = (1 - om) * p[:, c] + mid * ((p[:, e] + p[:, w]) / dx2
                                                + (p[:, s] + p[:, no]) / dy2 - rhs[:, c])
                p[:, c] = np.where(fl[:, c], x, p[:, c])
            nrm = self.norm()
            assert (nrm >= eps * eps).all(), "ends early: not a case of this file"
        return nrm

    def torch_rb(self, n, check, eps):
        """Red-black sweeps (at most n) to the masked residual bound, tested
        every `check` sweeps (0: never)."""
        dev = self.device
        T = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
        p, fl = T(self.p), T(self.inner)
        rx, ry = T(1 / self.dx ** 2), T(1 / self.dy ** 2)
        om = self.prm.omega
        mid = om / (2 * rx + 2 * ry)
        rhs = T(self.rhs)
        num = fl.sum((1, 2), keepdim=True).clamp(min=1)
        rhs = torch.where(fl, rhs - (rhs * fl).sum((1, 2), keepdim=True) / num, 0.0)
        tol = eps * eps * (rhs * rhs).sum((1, 2))
        gi, ga, gb = (T(a) for a in self.ghost_plan())
        xy = (torch.arange(self.nx, device=dev)[:, None] + torch.arange(self.ny, device=dev)) % 2
        half = [fl & (xy == k) for k in (0, 1)]
        live = torch.ones(self.B, 1, 1, dtype=torch.bool, device=dev)
        c = (slice(None), slice(1, -1), slice(1, -1))
        masks = [h[c] for h in half]
        mr = mid * rhs[c]
        mx, my = mid * rx, mid * ry
        res = torch.zeros(self.B, dtype=torch.float64, device=dev)

        def ghosts():
            q = p.view(-1)
            q[gi] = (q[ga] + q[gb]) * 0.5

        k = 0
        while k < n:
            m = min(check, n - k) if check else n
            for _ in range(m):
                ghosts()
                for h in (0, 1):
                    x = (1 - om) * p[c] + (mx * (p[:, 2:, 1:-1] + p[:, :-2, 1:-1]) + my * (
                        p[:, 1:-1, 2:] + p[:, 1:-1, :-2]) - mr)
                    p[c] = torch.where(masks[h], x, p[c])
            k += m
            ghosts()
            if check:
                q = p[c]
                r = rx * ((p[:, 2:, 1:-1] - q) - (q - p[:, :-2, 1:-1])) + ry * (
                    (p[:, 1:-1, 2:] - q) - (q - p[:, 1:-1, :-2])) - rhs[c]
                r2 = torch.where(fl[c], r * r, 0.0).sum((1, 2))
                res = torch.where(live[:, 0, 0], r2, res)
                live = live & (r2 > tol)[:, None, None]
                masks = [h[c] & live for h in half]
                if not bool(live.any()):
                    break
        self.p = p.cpu().numpy()
        return res.cpu().numpy() / self.fl.sum((1, 2))

    def adapt(self):
        """The adaptive step from the fields a tick starts with."""
        um = np.abs(np.where(self.fl, self.u, 0.0))
        vm = np.abs(np.where(self.fl, self.v, 0.0))
        um[:, :-1] = np.maximum(um[:, :-1], np.where(self.fl[:, 1:], abs(self.u[:, :-1]), 0.0))
        vm[:, :, :-1] = np.maximum(vm[:, :, :-1], np.where(self.fl[:, :, 1:], abs(self.v[:, :, :-1]), 0.0))
        um, vm = um.max((1, 2), keepdims=True), vm.max((1, 2), keepdims=True)
        self.delt = self.prm.tau * np.minimum(
            self.re / 2 / (1 / self.dx ** 2 + 1 / self.dy ** 2),
            np.minimum(self.dx / np.maximum(um, 1e-300), self.dy / np.maximum(vm, 1e-300)))

    def project(self):
        u, v, p = self.u, self.v, self.p
        u[:, :-1, :-1] = self.f[:, :-1, :-1] - (self.delt / self.dx) * (p[:, 1:, :-1] - p[:, :-1, :-1])
        v[:, :-1, :-1] = self.g[:, :-1, :-1] - (self.delt / self.dy) * (p[:, :-1, 1:] - p[:, :-1, :-1])
        for i, a, b in self.restore:
            u[i], v[i] = a, b


def _network(params, x):
    """The U-Net on x (nb, H, W, 2) in the dtype of the parameters."""
    lay, head, _ = _layout()

    def conv(k, a):
        w0, (cout, _, cin), b0 = lay[k]
        w = params[w0:w0 + cout * 9 * cin].reshape(cout, 9, cin)[:, :, :a.shape[-1]]
        nb, h, wd, ci = a.shape
        q = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1))
        out = params[b0:b0 + cout]
        for tap in range(9):
            i, j = divmod(tap, 3)
            out = out + q[:, i:i + h, j:j + wd].reshape(-1, ci) @ w[:, tap].t().contiguous()
        return torch.relu(out).reshape(nb, h, wd, cout)

    def pool(a):
        nb, h, w, c = a.shape
        return a.reshape(nb, h // 2, 2, w // 2, 2, c).amax((2, 4))

    def join(low, skip):
        return torch.cat([low.repeat_interleave(2, 1).repeat_interleave(2, 2), skip], -1)

    e0 = conv(1, conv(0, x))
    e1 = conv(3, conv(2, pool(e0)))
    e2 = conv(5, conv(4, pool(e1)))
    e3 = conv(7, conv(6, pool(e2)))
    d2 = conv(9, conv(8, join(e3, e2)))
    d1 = conv(11, conv(10, join(d2, e1)))
    d0 = conv(13, conv(12, join(d1, e0)))
    return d0 @ params[head:head + 32] + params[head + 32]


def _padded(grids):
    """The grids at one size: solid cells, which nothing reads, beyond their ends."""
    nx, ny = (max(g[0].shape[k] for g in grids) for k in (0, 1))

    def pad(a, fill):
        return np.pad(a, [(0, nx - a.shape[0]), (0, ny - a.shape[1])] + [(0, 0)] * (a.ndim - 2),
                      constant_values=fill)

    return [(pad(ct, 1), pad(vel, 0.0), prm, {k: pad(f[k], 0.0) for k in f})
            for ct, vel, prm, f in grids]


def exact(case, seed):
    kind = case["kind"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if kind in ("train", "learned"):   # inputs or corrections of 16-bit networks on the way
        return None
    if kind in ("forward", "gradients"):
        params = torch.tensor(_weights(seed), dtype=torch.float64, device=dev)
        x, t = (torch.tensor(a, dtype=torch.float64, device=dev) for a in _batch(case, seed))
        if kind == "forward":
            return {"y": _network(params, x).cpu().numpy()}
        params.requires_grad_(True)
        y = _network(params, x)
        m = (x[..., 1] > 0).double()
        loss = ((m * (y - t) ** 2).sum((1, 2)) / (m * t * t).sum((1, 2))).mean()
        loss.backward()
        g = params.grad.clone()
        w = g[:CONVS[0][1] * 9 * 32].reshape(32, 9, 32)
        w[:, :, 2:] = 0.0
        return {"loss": float(loss.detach()), "g": g.cpu().numpy()}
    grids = _grids(case, seed)
    if kind == "sweeps":
        s = _Plain(grids, dev)
        s.rhs = grids[0][3]["rhs"][None].copy()
        s.torch_rb(case["n"], 0, 0.0)
        return {"p": s.p[0]}
    if kind == "load":
        s = _Plain(grids, dev)
        s.fgr()
        sp = np.sqrt(np.where(s.fl, s.u ** 2 + s.v ** 2, np.nan))
        return {"norm": float(s.norm()[0]), "speed": np.array([np.nanmin(sp), np.nanmax(sp)]),
                "f": s.f[0], "g": s.g[0], "rhs": s.rhs[0]}
    shapes = [g[0].shape for g in grids]
    s = _Plain(_padded(grids), dev)
    for _ in range(case.get("ticks", 1)):
        if kind == "rb":
            s.adapt()
        s.walls()
        s.fgr()
        if kind == "rb":
            nrm = s.torch_rb(case["iters"], case["check"], case["eps"])
        else:
            nrm = s.lex(case["iters"], 1e-3)
        s.project()
    out = {k: [getattr(s, k)[b, :nx, :ny] for b, (nx, ny) in enumerate(shapes)] for k in FIELDS}
    if kind == "frame":
        return {"image": None, "its": None, "norm": float(nrm[0]),
                **{k: out[k][0] for k in FIELDS}}
    return {"its": None, "norm": np.array(nrm),
            **{k: np.concatenate([a.ravel() for a in out[k]]) for k in FIELDS}}
