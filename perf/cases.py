"""Timing cases of the framework: what a user's program has it compute, through
its public entry points, over the sizes, precisions and options it serves.

A case is a dict of plain values.  ``prepare`` makes what the program holds
before the call (inputs from a seed, the plan or network it keeps), ``run``
is one pass, ``exact`` the same result in plain 64-bit torch, ``work`` the
bytes and operations the pass cannot do without.

The inputs are a slice of a plasma wake: coarse particles displaced and
pushed along a radial wave around the beam axis with smooth disturbances on
top, and the densities and fields that belong to them (the deposition of
those particles and the Poisson solves of that density), so that every
kernel meets the displacements, gradients and cancellations of a real run.
"""

import math
import random
import types

import numpy as np
import torch
import torch.nn.functional as nnf

import lcode3d_amd as lc
from lcode3d_amd.unet import LAYERS, UNetPredictor

FIELDS = ("Ex", "Ey", "Ez", "Bx", "By", "Bz")
DENSITIES = ("ro", "jx", "jy", "jz")
COARSE = ("x_offt", "y_offt", "px", "py", "pz")

#: grid_steps the FFT solvers take: N - 1 even with the prime factors 2, 3, 5
GRIDS = tuple(n + 1 for n in range(64, 1281, 2)
              if n // math.gcd(n, 2 ** 11 * 3 ** 7 * 5 ** 5) == 1)


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def _step(name, n, **kw):
    return dict({"name": name, "kind": "step", "n": n, "precision": "fp64",
                 "coarseness": 3, "fineness": 2, "variant_a": True, "beam": "array",
                 "cells": 1.2, "box": 16.0}, **kw)


def listed():
    return [
        # the smallest grid runs are set up and tried out with: a slice is a
        # dozen short launches
        _step("step_129", 129, coarseness=2, cells=.6, box=6.4),
        # a size without a compile-time transform plan, behind the bunch (the
        # beam is the scalar 0 there), the fields without Variant A
        _step("step_361_scalar_beam", 361, variant_a=False, beam="scalar", cells=1.0),
        # the production slice
        _step("step_641", 641),
        # the large case: fine plasma, a strong wake off the axis
        _step("step_1281_fine", 1281, fineness=3, cells=4.2),
        # the production slice with float32 grids
        _step("step_641_mixed", 641, precision="mixed"),
        # the same slice with the predictor pass replaced by an extrapolation
        # of earlier slices' fields
        _step("guided_641_mixed", 641, kind="guided", precision="mixed", box=10.),
        # a short run from the start, as main() does it: set-up and slices
        {"name": "run_257", "kind": "run", "n": 257, "coarseness": 2, "fineness": 2,
         "slices": 16, "box": 12.8},
        # the operators on their own, as diagnostics and training data
        # (predictor_fields) call them: a deposition, a push and the field
        # solves at a ragged size
        _step("deposit_641", 641, kind="deposit"),
        _step("push_1081", 1081, kind="push", cells=3.0),
        _step("fields_451", 451, kind="fields"),
        # the learned predictor: a guess for the next slice, and one training
        # step (forward, backward, Adam)
        _step("unet_guess_641", 641, kind="guess", precision="mixed"),
        {"name": "unet_train_641", "kind": "train", "n": 641},
    ]


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(("step", "step", "step", "guided", "run", "deposit", "push",
                       "fields", "guess", "train"))
    top = {"run": 321, "step": 1281, "guided": 901}.get(kind, 1281)
    want = math.exp(rng.uniform(math.log(65), math.log(top)))
    n = min((g for g in GRIDS if g <= top), key=lambda g: abs(g - want))
    if kind == "train":
        return {"kind": kind, "n": int(n) + rng.choice((0, 2, 4))}
    if kind == "run":
        return {"kind": kind, "n": n, "coarseness": rng.choice((2, 3)), "fineness": 2,
                "slices": rng.randint(4, 16), "box": round(n * .05, 3)}
    # float32 grids are for the production sizes and a wake that is under way
    # (a momentum that a slice only begins to build up has few digits there)
    mixed = n > 320 and kind in ("step", "guided", "guess") and rng.random() < .5
    c = _step("", n, kind=kind, coarseness=rng.choice((2, 3)), fineness=rng.choice((2, 2, 3)),
              variant_a=rng.random() < .75, beam=rng.choice(("array", "array", "scalar")),
              cells=round(rng.uniform(1.2 if mixed else .1, 4.2), 2),
              box=round(rng.uniform(6., 16.), 2), precision="mixed" if mixed else "fp64")
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# Plain torch statements of the path, in 64 bits
# ---------------------------------------------------------------------------

def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _config(case):
    n = case["n"]
    h = case["box"] / (n - 1)
    return types.SimpleNamespace(
        grid_steps=n, grid_step_size=h, xi_step_size=h / 5 if n > 300 else h,
        field_solver_subtraction_trick=1, field_solver_variant_A=case.get("variant_a", True),
        field_solver_precision=case.get("precision", "fp64"),
        reflect_padding_steps=5, plasma_padding_steps=10,
        plasma_coarseness=case["coarseness"], plasma_fineness=case["fineness"],
        reflect_boundary=h * (n / 2 - 5))


def _plasma(cfg):
    """Coarse particles and the coarse -> fine interpolation of one axis."""
    steps, h = cfg.grid_steps - 2 * cfg.plasma_padding_steps, cfg.grid_step_size
    c, f = cfg.plasma_coarseness, cfg.plasma_fineness
    half = np.arange(steps // (2 * c)) * (h * c)
    coarse = np.concatenate([-half[:0:-1], half])
    if f % 2:
        half = np.arange(steps // 2 * f) * (h / f)
        fine = np.concatenate([-half[:0:-1], half])
    else:
        half = (.5 + np.arange(steps // 2 * f)) * (h / f)
        fine = np.concatenate([-half[::-1], half])
    nc = len(coarse)
    at = np.searchsorted(coarse, fine)
    nxt, prv = np.clip(at, 0, nc - 1), np.clip(at - 1, 0, nc - 1)
    wp, wn = (coarse[nxt] - fine) / (h * c), (fine - coarse[prv]) / (h * c)
    wp[nxt == 0], wn[nxt == 0] = 0, 1
    wn[prv == nc - 1], wp[prv == nc - 1] = 0, 1
    up = lambda a: torch.as_tensor(a, device=_dev())  # noqa: E731
    x = up(coarse)
    ones = torch.ones((nc, nc), dtype=torch.float64, device=_dev())
    return types.SimpleNamespace(
        x=x[:, None].expand(nc, nc).contiguous(), y=x[None, :].expand(nc, nc).contiguous(),
        m=ones * c ** 2, q=-ones * c ** 2, fine=up(fine), prv=up(prv), nxt=up(nxt),
        wp=up(wp), wn=up(wn))


def _tsc(cfg, x, y):
    """Centre cells and the weights of the 3 x 3 cells around them."""
    n, h = cfg.grid_steps, cfg.grid_step_size
    xh, yh = x / h + .5, y / h + .5
    fx, fy = xh.floor(), yh.floor()
    i = (fx.long() + n // 2).clamp(1, n - 2)
    j = (fy.long() + n // 2).clamp(1, n - 2)
    a, b = xh - fx - .5, yh - fy - .5
    wx = ((.5 - a) ** 2 / 2, .75 - a ** 2, (.5 + a) ** 2 / 2)
    wy = ((.5 - b) ** 2 / 2, .75 - b ** 2, (.5 + b) ** 2 / 2)
    return i, j, [(di, dj, wx[di + 1] * wy[dj + 1]) for di in (-1, 0, 1) for dj in (-1, 0, 1)]


def _deposit(cfg, pl, xo, yo, px, py, pz, ro_initial=None):
    n = cfg.grid_steps
    small = 1 / (cfg.plasma_coarseness * cfg.plasma_fineness) ** 2

    def mix(a):
        rows = pl.wp[:, None] * a[pl.prv] + pl.wn[:, None] * a[pl.nxt]
        return rows[:, pl.prv] * pl.wp[None, :] + rows[:, pl.nxt] * pl.wn[None, :]

    m, q = small * mix(pl.m), small * mix(pl.q)
    px, py, pz = small * mix(px), small * mix(py), small * mix(pz)
    gamma = torch.sqrt(m ** 2 + px ** 2 + py ** 2 + pz ** 2)
    ro = q / (1 - pz / gamma)
    vals = (ro, px * (ro / gamma), py * (ro / gamma), pz * (ro / gamma))
    i, j, w = _tsc(cfg, pl.fine[:, None] + mix(xo), pl.fine[None, :] + mix(yo))
    out = [torch.zeros(n * n, dtype=torch.float64, device=xo.device) for _ in range(4)]
    for di, dj, wk in w:
        at = ((i + di) * n + j + dj).reshape(-1)
        for o, v in zip(out, vals):
            o.index_add_(0, at, (v * wk).reshape(-1))
    out = [o.view(n, n) for o in out]
    if ro_initial is not None:
        out[0] = out[0] + ro_initial
    return out


def _estimate(cfg, pl, s):
    g = torch.sqrt(pl.m ** 2 + s.px ** 2 + s.py ** 2 + s.pz ** 2)
    r = cfg.reflect_boundary
    out = []
    for x0, off, p in ((pl.x, s.x_offt, s.px), (pl.y, s.y_offt, s.py)):
        x = x0 + off + p / (g - s.pz) * cfg.xi_step_size
        x = torch.where(x >= r, 2 * r - x, x)
        out.append(torch.where(x <= -r, -2 * r - x, x) - x0)
    return out


def _push(cfg, pl, s, ex, ey, fields):
    dxi, n, r = cfg.xi_step_size, cfg.grid_steps, cfg.reflect_boundary
    i, j, w = _tsc(cfg, pl.x + (s.x_offt + ex) / 2, pl.y + (s.y_offt + ey) / 2)
    Ex, Ey, Ez, Bx, By, Bz = (sum(f.reshape(-1)[(i + di) * n + j + dj] * wk for di, dj, wk in w)
                              for f in fields)
    px, py, pz = s.px, s.py, s.pz
    for _ in range(2):
        g = torch.sqrt(pl.m ** 2 + pz ** 2 + px ** 2 + py ** 2)
        vx, vy, vz = px / g, py / g, pz / g
        k = pl.q * dxi / (1 - pz / g)
        dx, dy, dz = (k * (Ex + vy * Bz - vz * By), k * (Ey - vx * Bz + vz * Bx),
                      k * (Ez + vx * By - vy * Bx))
        px, py, pz = s.px + dx / 2, s.py + dy / 2, s.pz + dz / 2
    g = torch.sqrt(pl.m ** 2 + pz ** 2 + px ** 2 + py ** 2)
    out = []
    for x0, off, p, new in ((pl.x, s.x_offt, px, s.px + dx), (pl.y, s.y_offt, py, s.py + dy)):
        off = off + p / (g - pz) * dxi
        x = x0 + off
        for sign in (1, -1):
            hit = x * sign > r
            x = torch.where(hit, sign * 2 * r - x, x)
            off, new = torch.where(hit, x - x0, off), torch.where(hit, -new, new)
        out.append((off, new))
    return out[0][0], out[1][0], out[0][1], out[1][1], s.pz + dz


def _sine(a, dim):
    """Type-1 sine transform along dim: 2 sum sin(pi (k + 1)(m + 1) / (M + 1)) a[m]."""
    z = torch.zeros_like(a.narrow(dim, 0, 1))
    return -torch.fft.rfft(torch.cat([z, a, z, -a.flip(dim)], dim), dim=dim).imag.narrow(
        dim, 1, a.shape[dim])


def _cosine(a, dim):
    """Type-1 cosine transform along dim."""
    inner = a.narrow(dim, 1, a.shape[dim] - 2).flip(dim)
    return torch.fft.rfft(torch.cat([a, inner], dim), dim=dim).real


def _solve(cfg, rhs, tx, ty, add):
    """(lam_x + lam_y + add) u = rhs under the transforms tx along i, ty along j."""
    n, h = cfg.grid_steps, cfg.grid_step_size
    lam = 4 / h ** 2 * torch.sin(torch.arange(n, dtype=torch.float64, device=rhs.device)
                                 * math.pi / (2 * (n - 1))) ** 2
    lx = lam[1:-1] if tx is _sine else lam
    ly = lam[1:-1] if ty is _sine else lam
    den = (lx[:, None] + ly[None, :] + add) * (2. * (n - 1)) ** 2
    zero = den == 0
    f = torch.where(zero, 0., ty(tx(rhs, 0), 1) / torch.where(zero, 1., den))
    return ty(tx(f, 0), 1)


def _diff(cfg, a, dim):
    out = torch.zeros_like(a)
    d = (a[2:, 1:-1] - a[:-2, 1:-1]) if dim == 0 else (a[1:-1, 2:] - a[1:-1, :-2])
    out[1:-1, 1:-1] = d / (2 * cfg.grid_step_size)
    return out


def _transverse(cfg, trick, beam, ro, jx, jy, jz, jx_prev, jy_prev, add=1):
    """Ex, Ey, Bx, By; trick None: the Poisson equations without that term."""
    djx, djy = (jx_prev - jx) / cfg.xi_step_size, (jy_prev - jy) / cfg.xi_step_size
    t = trick if trick is not None else (0., 0., 0., 0.)
    r, z = ro + beam, jz + beam
    rhs = (-((_diff(cfg, r, 0) - djx) - t[0]), -((_diff(cfg, r, 1) - djy) - t[1]),
           (_diff(cfg, z, 1) - djy) + t[2], -((_diff(cfg, z, 0) - djx) - t[3]))
    out = []
    for k, f in enumerate(rhs):
        if k in (1, 2):
            out.append(nnf.pad(_solve(cfg, f[1:-1, :], _sine, _cosine, add), (0, 0, 1, 1)))
        else:
            out.append(nnf.pad(_solve(cfg, f[:, 1:-1], _cosine, _sine, add), (1, 1)))
    return out


def _longitudinal(cfg, jx, jy):
    ez = _solve(cfg, -(_diff(cfg, jx, 0) + _diff(cfg, jy, 1))[1:-1, 1:-1], _sine, _sine, 0)
    bz = _solve(cfg, -(_diff(cfg, jx, 1) - _diff(cfg, jy, 0)), _cosine, _cosine, 0)
    return nnf.pad(ez, (1, 1, 1, 1)), bz - bz.mean()


def _field_pass(cfg, prev, trick, beam, dens):
    ro, jx, jy, jz = dens
    a = cfg.field_solver_variant_A
    Ex, Ey, Bx, By = _transverse(cfg, (trick[0], trick[1], trick[3], trick[4]), beam,
                                 (ro + prev.ro) / 2 if a else ro, jx, jy,
                                 (jz + prev.jz) / 2 if a else jz, prev.jx, prev.jy)
    if a:
        Ex, Ey, Bx, By = 2 * Ex - prev.Ex, 2 * Ey - prev.Ey, 2 * Bx - prev.Bx, 2 * By - prev.By
    Ez, Bz = _longitudinal(cfg, jx, jy)
    return (Ex, Ey, Ez, Bx, By, Bz)


def _slice(cfg, pl, ro0, prev, beam, guess=None, first_fields=False):
    """One slice; guess: these fields for the predictor pass's;
    first_fields: only the predictor pass's fields."""
    old = [getattr(prev, k) for k in FIELDS]
    at = _push(cfg, pl, prev, *_estimate(cfg, pl, prev), old)
    fields = guess
    if fields is None:
        fields = _field_pass(cfg, prev, old, beam, _deposit(cfg, pl, *at, ro0))
    if first_fields:
        return fields
    avg = [(f + o) / 2 for f, o in zip(fields, old)]
    at = _push(cfg, pl, prev, at[0], at[1], avg)
    fields = _field_pass(cfg, prev, avg, beam, _deposit(cfg, pl, *at, ro0))
    avg = [(f + o) / 2 for f, o in zip(fields, old)]
    at = _push(cfg, pl, prev, at[0], at[1], avg)
    dens = _deposit(cfg, pl, *at, ro0)
    return types.SimpleNamespace(**dict(zip(COARSE + FIELDS + DENSITIES,
                                            (*at, *fields, *dens))))


def _ro_initial(cfg, pl):
    z = torch.zeros_like(pl.m)
    return -_deposit(cfg, pl, z, z, z, z, z)[0]


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _smooth(rnd, x, y, half):
    """A smooth disturbance of order one that fades out towards the edge."""
    out = 0
    for _ in range(4):
        a, b = rnd.uniform(.5, 3.) * math.pi / half, rnd.uniform(.5, 3.) * math.pi / half
        out = out + rnd.uniform(-.5, .5) * torch.sin(a * x + rnd.uniform(0, 6.28)) \
            * torch.cos(b * y + rnd.uniform(0, 6.28))
    return out * (1 - (x / half) ** 2).clamp(0) * (1 - (y / half) ** 2).clamp(0)


def _wake(case, seed):
    """Config, plasma, a slice of the wake and the next slice's beam."""
    rnd = random.Random(seed)
    cfg, h = _config(case), case["box"] / (case["n"] - 1)
    pl = _plasma(cfg)
    half = case["box"] / 2
    sigma = rnd.uniform(.08, .14) * half
    cx = rnd.uniform(-.1, .1) * half if case["cells"] > 2 else 0.
    wave = rnd.uniform(.5, 1.)
    x, y = pl.x - cx, pl.y
    env = torch.exp(.5 - (x * x + y * y) / (2 * sigma * sigma))
    d = case["cells"] * h
    # momenta of the order of the displacement (both in plasma units: the
    # wave turns the one into the other over a radian of xi), in units of
    # the macroparticles' mass
    p = d * float(pl.m[0, 0])
    s = types.SimpleNamespace(
        x_offt=-d * wave * x / sigma * env + .1 * d * _smooth(rnd, pl.x, pl.y, half),
        y_offt=-d * wave * y / sigma * env + .1 * d * _smooth(rnd, pl.x, pl.y, half),
        px=.6 * p * x / sigma * env + .1 * p * _smooth(rnd, pl.x, pl.y, half),
        py=.6 * p * y / sigma * env + .1 * p * _smooth(rnd, pl.x, pl.y, half),
        pz=.4 * p * env + .1 * p * _smooth(rnd, pl.x, pl.y, half))
    ro0 = _ro_initial(cfg, pl)
    s.ro, s.jx, s.jy, s.jz = _deposit(cfg, pl, s.x_offt, s.y_offt, s.px, s.py, s.pz, ro0)
    g = (torch.arange(cfg.grid_steps, device=_dev(), dtype=torch.float64)
         - cfg.grid_steps // 2) * h
    beam = 0.
    if case["beam"] == "array":
        beam = rnd.uniform(.02, .1) * torch.exp(
            -((g[:, None] - cx) ** 2 + g[None, :] ** 2) / (2 * sigma * sigma))
    s.Ex, s.Ey, s.Bx, s.By = _transverse(cfg, None, beam, s.ro, s.jx, s.jy, s.jz, s.jx, s.jy,
                                         add=0)
    s.Ez, s.Bz = _longitudinal(cfg, s.jx, s.jy)
    # the slice after it, its fields in step with its change of current (the
    # fields push the plasma, whose currents make the fields)
    fields = [getattr(s, k) for k in FIELDS]
    for _ in range(3):
        at = _push(cfg, pl, s, *_estimate(cfg, pl, s), fields)
        dens = _deposit(cfg, pl, *at, ro0)
        Ex, Ey, Bx, By = _transverse(cfg, (fields[0], fields[1], fields[3], fields[4]), beam,
                                     *dens, s.jx, s.jy)
        Ez, Bz = _longitudinal(cfg, dens[1], dens[2])
        fields = [Ex, Ey, Ez, Bx, By, Bz]
    s = types.SimpleNamespace(**dict(zip(COARSE + FIELDS + DENSITIES, (*at, *fields, *dens))))
    if case["precision"] == "mixed":   # grids are float32 there
        for k in FIELDS + DENSITIES:
            setattr(s, k, getattr(s, k).float())
    return cfg, pl, ro0, s, beam


def _wide(s):
    return types.SimpleNamespace(**{k: v.double() for k, v in vars(s).items()})


def _terms(cfg, pl, ro0, s, beam):
    """Three earlier slices' fields whose extrapolation 2 F1 - 2 F3 + F4 is
    the predictor pass's fields (what a good guess comes to)."""
    f1 = _slice(cfg, pl, ro0, _wide(s), beam, first_fields=True)
    old = [getattr(s, k).double() for k in FIELDS]
    f3, f4 = [.98 * o for o in old], [.96 * o for o in old]
    first = [(f + 2 * b - c) / 2 for f, b, c in zip(f1, f3, f4)]
    t = getattr(s, "Ex").dtype
    return [(w, tuple(v.to(t) for v in vs)) for w, vs in ((2., first), (-2., f3), (1., f4))]


def _beams(case, cfg, seed):
    """The beam of each slice of a run: a bunch that grows from nothing."""
    rnd = random.Random(seed)
    sigma, amp = rnd.uniform(.5, 1.), rnd.uniform(.02, .1)
    g = (torch.arange(cfg.grid_steps, device=_dev(), dtype=torch.float64)
         - cfg.grid_steps // 2) * cfg.grid_step_size
    shape = torch.exp(-(g[:, None] ** 2 + g[None, :] ** 2) / (2 * sigma * sigma))
    return [amp * (1 - math.cos(k * cfg.xi_step_size * math.sqrt(math.pi / 2))) * shape
            for k in range(case["slices"])]


def _layers(seed):
    rng = np.random.default_rng(seed)
    return [(rng.standard_normal((co, ci, 3, 3)) * math.sqrt(2. / (9 * ci))
             * (.1 if k == len(LAYERS) - 1 else 1.), .05 * rng.standard_normal(co))
            for k, (ci, co) in enumerate(LAYERS)]


def _planes(case, seed):
    """Input planes (14 channels of order one) and targets of the network."""
    rnd = random.Random(seed)
    s = (case["n"] + 3) // 4
    g = torch.linspace(-.95, .95, s, device=_dev(), dtype=torch.float64)
    x, y = g[:, None].expand(s, s), g[None, :].expand(s, s)
    make = lambda k: torch.stack([2 * _smooth(rnd, x, y, 1.) for _ in range(k)], -1)  # noqa: E731
    planes = torch.zeros((s, s, 32), dtype=torch.float64, device=_dev())
    planes[..., :14] = make(14)
    return planes.to(torch.bfloat16), make(6).float().contiguous()


def _scales(s, beam):
    """Per-channel scales as training fits them: the planes' RMS."""
    rms = lambda a: max(float(a.double().square().mean().sqrt()), 1e-9)  # noqa: E731
    f = [rms(getattr(s, k)) for k in FIELDS]
    b = rms(beam) if isinstance(beam, torch.Tensor) else 1.
    return np.array(f + [.02 * v for v in f] + [b, rms(s.ro)], dtype=np.float32), \
        np.array([1e-3 * v for v in f], dtype=np.float32)


# ---------------------------------------------------------------------------
# prepare, run, exact, work
# ---------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        net = UNetPredictor(case["n"])
        net.set_params(_layers(seed))
        x, t = _planes(case, seed)
        return types.SimpleNamespace(kind=kind, net=net, x=x.view(torch.int16), t=t)
    if kind == "run":
        cfg = _config(case)
        return types.SimpleNamespace(kind=kind, cfg=cfg, beams=_beams(case, cfg, seed))
    cfg, pl, ro0, s, beam = _wake(case, seed)
    _, _, const, vp, _ = lc.init(cfg)
    st = types.SimpleNamespace(kind=kind, cfg=cfg, const=const, vp=vp, beam=beam,
                               prev=lc.GPUArrays(**vars(s)))
    if kind == "guided":
        st.guess = _terms(cfg, pl, ro0, s, beam)
    elif kind == "fields":
        st.j_prev = (.98 * s.jx, .98 * s.jy)
    elif kind == "push":
        st.est = [e.contiguous() for e in _estimate(cfg, pl, s)]
    elif kind == "guess":
        st.net = UNetPredictor(case["n"])
        st.net.set_params(_layers(seed))
        st.net.scale, st.net.tscale = _scales(s, beam)
        st.older = [lc.GPUArrays(**{k: getattr(s, k) * w for k in FIELDS + DENSITIES})
                    for w in (.98, .96)]
    return st


def run(state):
    s, kind = state, state.kind
    if kind == "train":
        loss = s.net.train_step(s.x, s.t)
        return {"loss": loss, "grad": s.net.grad, "params": s.net.params}
    if kind == "run":
        _, _, const, vp, st = lc.init(s.cfg)
        c = s.cfg.grid_steps // 2
        axis = torch.empty(len(s.beams), dtype=torch.float64, device=st.Ez.device)
        for k, beam in enumerate(s.beams):
            st = lc.step(s.cfg, const, vp, st, beam)
            axis[k] = st.Ez[c, c]
        return {"axis": axis, **{k: getattr(st, k) for k in COARSE + FIELDS + DENSITIES}}
    p, c = s.prev, s.const
    if kind == "step":
        return vars(lc.step(s.cfg, c, s.vp, p, s.beam))
    if kind == "guided":
        return vars(lc.step(s.cfg, c, s.vp, p, s.beam, guess=s.guess))
    if kind == "deposit":
        return lc.deposit(s.cfg, c.ro_initial, p.x_offt, p.y_offt, c.m, c.q, p.px, p.py, p.pz,
                          s.vp)
    if kind == "push":
        return lc.move_smart(s.cfg, c.m, c.q, c.x_init, c.y_init, p.x_offt, p.y_offt, *s.est,
                             p.px, p.py, p.pz, *(getattr(p, k) for k in FIELDS))
    if kind == "fields":
        return (*lc.calculate_Ex_Ey_Bx_By(s.cfg, p.Ex, p.Ey, p.Bx, p.By, s.beam, p.ro, p.jx,
                                          p.jy, p.jz, *s.j_prev),
                lc.calculate_Ez(s.cfg, p.jx, p.jy), lc.calculate_Bz(s.cfg, p.jx, p.jy))
    return s.net.guess(p, *s.older, s.beam)


def _network(layers, x):
    """The network in 64 bits on [14, S, S] planes."""
    conv = lambda k, a: nnf.conv2d(a, *layers[k], padding=1)  # noqa: E731
    relu = nnf.relu

    def pool(a):
        return nnf.avg_pool2d(nnf.pad(a, (0, a.shape[-1] % 2, 0, a.shape[-2] % 2)), 2)

    def up(a, like):
        return a.repeat_interleave(2, -2).repeat_interleave(2, -1)[
            ..., :like.shape[-2], :like.shape[-1]]

    e0 = relu(conv(0, x[None]))
    e1 = relu(conv(1, pool(e0)))
    e2 = relu(conv(2, pool(e1)))
    e3 = relu(conv(3, pool(e2)))
    d2 = relu(conv(4, torch.cat([up(e3, e2), e2], 1)))
    d1 = relu(conv(5, torch.cat([up(d2, e1), e1], 1)))
    d0 = relu(conv(6, torch.cat([up(d1, e0), e0], 1)))
    return conv(7, d0)[0]


def _params(seed, round_weights):
    out = []
    for w, b in _layers(seed):
        w, b = (torch.as_tensor(a.astype(np.float32)) for a in (w, b))
        w = w.bfloat16() if round_weights else w
        out.append([w.double(), b.double()])
    return out


def _mean4(a):
    """4 x 4 means of a grid, zeros beyond the far edge."""
    pad = (-a.shape[-1]) % 4
    return nnf.avg_pool2d(nnf.pad(a, (0, pad, 0, pad))[None], 4)[0]


def _exact_train(case, seed):
    planes, t = _planes(case, seed)
    x = planes.double().cpu().permute(2, 0, 1)[:14]
    layers = _params(seed, True)
    flat = [p.requires_grad_() for wb in layers for p in wb]
    y = _network(layers, x)
    loss = ((y.permute(1, 2, 0) - t.double().cpu()) ** 2).mean()
    loss.backward()
    grad = torch.cat([p.grad.reshape(-1) for p in flat])
    start = torch.cat([p.reshape(-1) for wb in _params(seed, False) for p in wb])
    return {"loss": loss.detach().reshape(1), "grad": grad,
            "params": start - 1e-3 * grad / (grad.abs() + 1e-8)}


def _exact_guess(case, seed):
    _, _, _, s, beam = _wake(case, seed)
    scale, tscale = (torch.as_tensor(a).double() for a in _scales(s, beam))
    w = _wide(s)
    f = [getattr(w, k).cpu() for k in FIELDS]
    second, third = ([(getattr(s, k) * c).double().cpu() for k in FIELDS] for c in (.98, .96))
    n = case["n"]
    b = beam.cpu() if isinstance(beam, torch.Tensor) else torch.full((n, n), float(beam)).double()
    planes = f + [a - c for a, c in zip(f, second)] + [b, w.ro.cpu()]
    x = torch.stack([_mean4(a[None])[0] / k for a, k in zip(planes, scale)])
    y = _network(_params(seed, True), x.bfloat16().double()) * tscale[:, None, None]
    y = y.repeat_interleave(4, -2).repeat_interleave(4, -1)[:, :n, :n]
    return tuple(3 * a - 3 * c + d + v for a, c, d, v in zip(f, second, third, y))


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "guess":
        return _exact_guess(case, seed)
    if kind == "run":
        cfg = _config(case)
        pl = _plasma(cfg)
        ro0, z, n = _ro_initial(cfg, pl), torch.zeros_like(pl.m), cfg.grid_steps
        zero = torch.zeros((n, n), dtype=torch.float64, device=_dev())
        s = types.SimpleNamespace(**{k: z for k in COARSE},
                                  **{k: zero for k in FIELDS + DENSITIES})
        axis = []
        for beam in _beams(case, cfg, seed):
            s = _slice(cfg, pl, ro0, s, beam)
            axis.append(s.Ez[n // 2, n // 2])
        return {"axis": torch.stack(axis), **vars(s)}
    cfg, pl, ro0, s, beam = _wake(case, seed)
    w = _wide(s)
    if kind == "step":
        return vars(_slice(cfg, pl, ro0, w, beam))
    if kind == "guided":
        terms = _terms(cfg, pl, ro0, s, beam)
        guess = [sum(c * vs[k].double() for c, vs in terms) for k in range(6)]
        return vars(_slice(cfg, pl, ro0, w, beam, guess=guess))
    if kind == "deposit":
        return _deposit(cfg, pl, w.x_offt, w.y_offt, w.px, w.py, w.pz, ro0)
    if kind == "push":
        return _push(cfg, pl, w, *_estimate(cfg, pl, w), [getattr(w, k) for k in FIELDS])
    return (*_transverse(cfg, (w.Ex, w.Ey, w.Bx, w.By), beam, w.ro, w.jx, w.jy, w.jz,
                         .98 * w.jx, .98 * w.jy), *_longitudinal(cfg, w.jx, w.jy))


def work(case):
    """Every input read once, every output written once; operations of the
    transforms at 2.5 log2(2 N) a point and line, of a fine particle's
    interpolation and 36 products at 220, of a push at 700."""
    kind, n = case["kind"], case["n"]
    if kind in ("guess", "train"):
        s, cells = (n + 3) // 4, 0
        for k, (ci, co) in enumerate(LAYERS):
            side = s
            for _ in range((0, 1, 2, 3, 2, 1, 0, 0)[k]):
                side = (side + 1) // 2
            cells += 18 * ci * co * side * side
        params = sum(co * (9 * ci + 1) for ci, co in LAYERS)
        if kind == "train":
            return {"bytes": s * s * (2 * 14 + 4 * 6) + 28 * params, "flops": 3 * cells}
        size = 4 if case["precision"] == "mixed" else 8
        return {"bytes": n * n * (size * 25 + 8) + 2 * params, "flops": cells}
    c, f = case["coarseness"], case["fineness"]
    steps = n - 20
    nc2 = (2 * (steps // (2 * c)) - 1) ** 2
    nf2 = (steps // 2 * f * 2 - f % 2) ** 2
    grid = (4 if case.get("precision") == "mixed" else 8) * n * n
    solve = 4 * 2.5 * math.log2(2 * n) * n * n     # one field, there and back
    if kind == "deposit":
        return {"bytes": 8 * 7 * nc2 + 5 * grid, "flops": 220 * nf2}
    if kind == "push":
        return {"bytes": 8 * 16 * nc2 + 6 * grid, "flops": 700 * nc2}
    if kind == "fields":
        return {"bytes": 17 * grid, "flops": 6 * solve}
    flops = 3 * (700 * nc2 + 220 * nf2) + (6 if kind == "guided" else 12) * solve
    if kind == "guided":
        flops -= 220 * nf2
    if kind == "run":
        return {"bytes": 8 * (case["slices"] * n * n + 10 * n * n + 5 * nc2),
                "flops": case["slices"] * flops}
    beams = 8 * n * n if case["beam"] == "array" else 0
    terms = 18 * grid if kind == "guided" else 0
    return {"bytes": 20 * grid + 8 * n * n + beams + terms + 8 * 14 * nc2, "flops": flops}
