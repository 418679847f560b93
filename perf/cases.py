"""What a user of this framework has it do, as cases that can be timed and checked.

A case is one call (or the few calls) that a program makes once its chunk is set up:

* ``steps``: the driver's loop (``diffuse``) over a few timesteps from an energy field that the
  program holds on the host, with the field summary of every step and the energy read back;
* ``solve``: the solver plug-in alone (``settings.solver.solve(chunk, settings, rx, ry)``) on
  device-resident fields, with the solution read back;
* ``predict``: the warm-start network's prediction of the next solution;
* ``train``: optimiser steps of that network on crops recorded from the chunk's own solves.

The decks are the repository's two families with values drawn from the seed: the three-state
reference deck (background, a hot and a cold rectangle of low density) and the random rectangles
(densities over four decades).  Domain 10 x 10 and a timestep of 0.004, as in the decks, unless the
case says otherwise.
"""
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "tealeaf.jl_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "tealeaf.jl_amd"))

import tealeaf_hip as T  # noqa: E402
from tealeaf_hip import unet  # noqa: E402

WEIGHTS = os.path.join(ROOT, "tealeaf.jl_amd", "weights", "unet_warmstart.npy")
HALO = 2
DOMAIN = 10.0


def listed():
    return [
        # the smallest runs (tests, unit problems): CG by its own stop rule, latency of every launch and copy counts
        dict(name="cg_steps_64", do="steps", deck="reference", solver="cg", precision="fp64", nx=64, ny=64, steps=3),
        # the 512^2 deck that ships with the framework, the size of its QA line
        dict(name="cg_steps_512", do="steps", deck="reference", solver="cg", precision="fp64", nx=512, ny=512, steps=2),
        # plain FP64 CG as plug-in on a ragged grid, with the reciprocal coefficient
        dict(name="cg_1501x1103", do="solve", deck="rectangles", solver="cg", precision="fp64", nx=1501, ny=1103, coefficient=2),
        # the largest plain FP64 CG solve: the baseline method of the benchmark
        dict(name="cg_3072", do="solve", deck="rectangles", solver="cg", precision="fp64", nx=3072, ny=3072),
        # the other FP64 solvers at ordinary sizes, with the deck's CG pre-steps and inner steps
        dict(name="cheby_2048", do="solve", deck="reference", solver="cheby", precision="fp64", nx=2048, ny=2048, presteps=30),
        dict(name="ppcg_1300x1700", do="solve", deck="reference", solver="ppcg", precision="fp64", nx=1300, ny=1700, presteps=8, inner=10),
        dict(name="jacobi_steps_200x300", do="steps", deck="reference", solver="jacobi", precision="fp64", nx=200, ny=300, steps=1),
        # the mixed-precision solver, the framework's fast path: ordinary, ragged and the benchmark's size
        # (there with a tenth of the timestep, to keep one solve near a second)
        dict(name="ir_1024", do="solve", deck="rectangles", solver="cg", precision="fp32_ir", nx=1024, ny=1024),
        dict(name="ir_2047x1533", do="solve", deck="rectangles", solver="cg", precision="fp32_ir", nx=2047, ny=1533),
        dict(name="ir_8192", do="solve", deck="rectangles", solver="cg", precision="fp32_ir", nx=8192, ny=8192, dt=0.0004),
        # the learned warm start: inference over a whole grid, and fine-tuning on recorded crops
        dict(name="unet_predict_2048", do="predict", deck="rectangles", nx=2048, ny=2048),
        dict(name="unet_train_16", do="train", deck="rectangles", nx=256, ny=256, batch=16, steps=4, loss="energy"),
    ]


def _size(rng, lo, hi):
    """Two edges between lo and hi, spread over their logarithm, at most a factor of two apart."""
    a = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    b = min(max(a * math.exp(rng.uniform(-math.log(2), math.log(2))), lo), hi)
    return int(round(a)), int(round(b))


def draw(rng):
    what = rng.choice(["cg_steps", "cg_steps", "cg", "cg", "cheby", "ppcg", "jacobi", "ir", "ir", "ir", "predict", "train"])
    if what == "cg_steps":
        nx, ny = _size(rng, 40, 640)
        return dict(do="steps", deck="reference", solver="cg", precision="fp64", nx=nx, ny=ny, steps=rng.randint(1, 3), launch=rng.randint(0, 1))
    if what == "cg":
        nx, ny = _size(rng, 100, 3000)
        return dict(do="solve", deck="rectangles", solver="cg", precision="fp64", nx=nx, ny=ny, coefficient=rng.randint(1, 2))
    if what == "cheby":
        nx, ny = _size(rng, 100, 2048)
        return dict(do="solve", deck="reference", solver="cheby", precision="fp64", nx=nx, ny=ny, presteps=rng.randint(8, 40))
    if what == "ppcg":
        nx, ny = _size(rng, 100, 1800)
        return dict(do="solve", deck="reference", solver="ppcg", precision="fp64", nx=nx, ny=ny, presteps=rng.randint(8, 40),
                    inner=rng.choice([4, 7, 10, 10, 10, 15, 20]))
    if what == "jacobi":
        nx, ny = _size(rng, 40, 320)
        return dict(do="steps", deck="reference", solver="jacobi", precision="fp64", nx=nx, ny=ny, steps=1)
    if what == "ir":
        nx, ny = _size(rng, 120, 4096)
        if rng.random() < 0.5:
            nx = max(120, nx // 4 * 4)
        return dict(do="solve", deck="rectangles", solver="cg", precision="fp32_ir", nx=nx, ny=ny, coefficient=rng.randint(1, 2))
    if what == "predict":
        nx, ny = _size(rng, 200, 4096)
        return dict(do="predict", deck="rectangles", nx=nx // 4 * 4, ny=ny // 4 * 4)
    return dict(do="train", deck="rectangles", nx=256, ny=256, batch=rng.randint(4, 24), steps=rng.randint(1, 5),
                loss=rng.choice(["energy", "residual", "mse"]))


# ------------------------------------------------------------------ decks

def _states(case, seed):
    """(density, energy, xmin, xmax, ymin, ymax) of every state; the first fills the domain."""
    g = random.Random(1000003 * int(seed) + 17)
    if case["deck"] == "reference":
        x1, x2 = g.uniform(0.8, 1.2), g.uniform(5.0, 7.0)
        y0, y1 = g.uniform(0.8, 1.2), g.uniform(1.8, 2.4)
        return [(100.0, 0.0001, 0, 0, 0, 0), (0.1, g.uniform(20.0, 30.0), 0.0, x1, y0, y1),
                (0.1, g.uniform(0.08, 0.12), x1, x2, y0, y1)]
    out = [(100.0, 0.0001, 0, 0, 0, 0)]
    for _ in range(32):
        w, h = g.uniform(0.2, 3.0), g.uniform(0.2, 3.0)
        x, y = g.uniform(0.0, DOMAIN - w), g.uniform(0.0, DOMAIN - h)
        out.append((10.0 ** g.uniform(-2.0, 2.0), g.uniform(1e-4, 25.0), x, x + w, y, y + h))
    return out


def _deck(case, seed):
    rows = ["*tea"]
    for i, (rho, e, x0, x1, y0, y1) in enumerate(_states(case, seed)):
        rows.append(f"state {i + 1} density={rho:.17g} energy={e:.17g}" + (
            f" geometry=rectangle xmin={x0:.17g} xmax={x1:.17g} ymin={y0:.17g} ymax={y1:.17g}" if i else ""))
    rows += [f"x_cells={case['nx']}", f"y_cells={case['ny']}", "xmin=0.0", "ymin=0.0", f"xmax={DOMAIN}", f"ymax={DOMAIN}",
             f"initial_timestep={case.get('dt', 0.004)!r}", "end_step=10", "summary_frequency=1", f"halo_depth={HALO}",
             f"coefficient={case.get('coefficient', 1)}", f"max_iters={100000 if case['deck'] == 'rectangles' else 10000}", "eps=1e-15", f"presteps={case.get('presteps', 30)}",
             f"ppcg_inner_steps={case.get('inner', 10)}", f"use_{case.get('solver', 'cg')}"]
    if case["deck"] == "rectangles":
        rows += ["stop_rule=relative", "rel_tol=1e-10", f"precision={case.get('precision', 'fp64')}"]
    return "\n".join(rows + ["*endtea", ""])


# ---------------------------------------------------------------- the path

def prepare(case, seed):
    settings = T.Settings.from_text(_deck(case, seed))
    settings.set(launch=case.get("launch", T.TL_LAUNCH_STREAM))
    chunk = T.initialiseapp(settings)
    dt = case.get("dt", 0.004)
    state = dict(case=case, settings=settings, chunk=chunk, rx=dt / settings.dx ** 2, ry=dt / settings.dy ** 2)
    if case["do"] == "steps":
        state["energy"] = chunk.field("energy")
    elif case["do"] == "predict":
        unet.load_weights(chunk, WEIGHTS)
    elif case["do"] == "train":
        unet.load_weights(chunk, WEIGHTS)
        unet.record(chunk, capacity=32, crops_per_step=8)
        T.diffuse(chunk, settings, 4)
        unet.record(chunk, capacity=0, crops_per_step=0)
    return state


def run(state):
    case, chunk, settings = state["case"], state["chunk"], state["settings"]
    if case["do"] == "steps":
        chunk.set_field("energy", state["energy"])
        summaries, _ = T.diffuse(chunk, settings, case["steps"])
        return {"energy": chunk.interior("energy"), "summaries": summaries}
    if case["do"] == "solve":
        settings.solver.solve(chunk, settings, state["rx"], state["ry"])
        return {"u": chunk.interior("u")}
    if case["do"] == "predict":
        return {"guess": unet.predict(chunk, state["rx"], state["ry"], settings.coefficient)[HALO:-HALO, HALO:-HALO]}
    # fine-tuning: a rate below the training's own 1e-3, as for weights that are trained already
    loss = unet.train(chunk, steps=case["steps"], batch=case["batch"], lr=2e-5, seed=1, loss=case["loss"])
    return {"loss": loss, "weights": unet.get_weights(chunk)}


def work(case):
    cells = case["nx"] * case["ny"]
    if case["do"] == "predict":
        # density and energy in, the guess out; the multiply-adds of the network's convolutions
        return {"bytes": 24.0 * cells, "flops": 55000.0 * cells}
    if case["do"] == "train":
        # forward, input and weight gradients of the network over the batch's crops, read once each step
        px = case["steps"] * case["batch"] * 128 * 128
        return {"bytes": 28.0 * px, "flops": 3 * 55000.0 * px}
    # density and energy in, the solution out (for every step).  Arithmetic: about 21 operations a cell and iteration
    # (operator, three updates, two products); iterations estimated from the operator's condition number
    dt, low = case.get("dt", 0.004), 0.01 if case["deck"] == "rectangles" else 0.1
    kappa = 1.0 + 4.0 * dt * ((case["nx"] / DOMAIN) ** 2 + (case["ny"] / DOMAIN) ** 2) / low
    iters = 0.5 * kappa * 40.0 if case["solver"] == "jacobi" else 6.0 * math.sqrt(kappa)
    steps = case.get("steps", 1)
    return {"bytes": 24.0 * cells * steps, "flops": 21.0 * cells * iters * steps}


# ------------------------------------------------------------------- exact

def _fields(case, seed):
    """Interior density and energy: a state covers the cells that its rectangle, moved inwards by a hundredth of a cell as the
    deck format has it, touches; later states over earlier ones."""
    nx, ny = case["nx"], case["ny"]
    dx, dy = DOMAIN / nx, DOMAIN / ny
    k, j = torch.arange(nx, dtype=torch.float64, device="cuda"), torch.arange(ny, dtype=torch.float64, device="cuda")
    rho = torch.empty(ny, nx, dtype=torch.float64, device="cuda")
    e = torch.empty_like(rho)
    for i, (d, en, x0, x1, y0, y1) in enumerate(_states(case, seed)):
        if i == 0:
            rho.fill_(d)
            e.fill_(en)
            continue
        x0, x1, y0, y1 = x0 + dx / 100, x1 - dx / 100, y0 + dy / 100, y1 - dy / 100
        inside = (((j + 1) * dy >= y0) & (j * dy < y1))[:, None] & (((k + 1) * dx >= x0) & (k * dx < x1))[None, :]
        rho[inside] = d
        e[inside] = en
    return rho, e


def _solution(case, rho, e):
    """The solution of one implicit step from energy e: (1 + sum of face coefficients) u - neighbours = rho e, with no flux
    through the domain's faces; conjugate gradients with a diagonal preconditioner, restarted from the true residual."""
    dt, nx, ny = case.get("dt", 0.004), case["nx"], case["ny"]
    w = rho if case.get("coefficient", 1) == 1 else 1.0 / rho
    kx = dt / (DOMAIN / nx) ** 2 * (w[:, 1:] + w[:, :-1]) / (2.0 * w[:, 1:] * w[:, :-1])
    ky = dt / (DOMAIN / ny) ** 2 * (w[1:] + w[:-1]) / (2.0 * w[1:] * w[:-1])

    def apply(v):
        o = v.clone()
        f = kx * (v[:, 1:] - v[:, :-1])
        o[:, :-1] -= f
        o[:, 1:] += f
        f = ky * (v[1:] - v[:-1])
        o[:-1] -= f
        o[1:] += f
        return o

    dinv = torch.ones_like(rho)
    dinv[:, :-1] += kx
    dinv[:, 1:] += kx
    dinv[:-1] += ky
    dinv[1:] += ky
    dinv = 1.0 / dinv
    b = rho * e
    u, goal = b.clone(), 1e-15 * float(b.norm())
    for _ in range(4):
        r = b - apply(u)
        first = float(r.norm())
        if first <= goal:
            break
        stop = max(goal, 1e-7 * first)
        x, z = torch.zeros_like(u), dinv * r
        p, rz = z.clone(), (r * z).sum()
        for it in range(200000):
            q = apply(p)
            a = rz / (p * q).sum()
            x += a * p
            r -= a * q
            if it % 50 == 49 and float(r.norm()) <= stop:
                break
            z = dinv * r
            new = (r * z).sum()
            p = z + (new / rz) * p
            rz = new
        u += x
    return u


def exact(case, seed):
    if case["do"] in ("predict", "train"):
        # the network's 16-bit activations and weights have no counterpart in 64 bits, and the recorded crops stay on the device
        return None
    if case["nx"] * case["ny"] > 10_000_000:
        return None  # too long with plain tensor operations
    rho, e = _fields(case, seed)
    if case["do"] == "solve":
        return {"u": _solution(case, rho, e).cpu()}
    vol = DOMAIN / case["nx"] * DOMAIN / case["ny"]
    rows = []
    for _ in range(case["steps"]):
        u = _solution(case, rho, e)
        e = u / rho
        m = vol * rho
        rows.append([vol * rho.numel(), float(m.sum()), float((m * e).sum()), float((m * u).sum())])
    return {"energy": e.cpu(), "summaries": np.array(rows)}
