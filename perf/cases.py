"""The workloads whose speed is tracked: what a user of this framework runs, through its public entry points.

A case is one of five kinds of work:

* ``step``: one or more substeps of a simulation loop, each ``CollisionPipeline.collide`` followed by
  ``SolverVBD.step``, from given positions and velocities.  ``graph`` replays them as one captured HIP graph (how
  the benchmark runs whole frames); otherwise they are launched one by one, as a plain Python loop does.
* ``solve``: one substep of a batch of worlds, each iterated to its own force-residual tolerance.
* ``warm``: the start of a warm-started substep: forward step, 1-ring features, network, low-passed candidates.
* ``mlp`` / ``train``: inference on a batch of feature rows / one training step (gradient and Adam).

Scenes, sizes and options are those of ``newton_amd.scenes``, the tests and the benchmark.  Models, solvers and
pipelines are kept per scene (a program builds them once); states come from the seed.
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

from newton_amd import CollisionPipeline, scenes
from newton_amd.solvers import SolverVBD
from newton_amd.warmstart import LearnedWarmStart, WarmStartMLP

DEV = "cuda:0"
CONTACT_MARGIN = 0.01


def listed():
    return [
        # the smallest simulation (the 32x32 hanging cloth, 5 iterations) in a plain Python loop: latency and launches
        {"name": "hanging_32_loop", "work": "step", "scene": "hanging", "size": 32, "iterations": 5, "substeps": 1,
         "graph": False},
        # the same cloth as an interactive program runs it: a frame of 10 substeps as one graph
        {"name": "hanging_32_frame", "work": "step", "scene": "hanging", "size": 32, "iterations": 5, "substeps": 10,
         "graph": True},
        # an odd-sized cloth with damped springs on every edge and hinge, draped, launched from Python
        {"name": "springs_97_loop", "work": "step", "scene": "springs", "size": 97, "iterations": 10, "substeps": 1,
         "graph": False},
        # the configured 256x256 cloth draped over the sphere and the ground, 10 iterations
        {"name": "drop_256", "work": "step", "scene": "drop", "size": 256, "iterations": 10, "substeps": 1,
         "graph": True},
        # the same cloth on a body another solver moves, with edge and face contact records
        {"name": "moving_256", "work": "step", "scene": "moving", "size": 256, "iterations": 10, "substeps": 1,
         "graph": True},
        # two stacked sheets in self-contact over the sphere
        {"name": "layers_128", "work": "step", "scene": "layers", "size": 128, "iterations": 10, "substeps": 1,
         "graph": True},
        # many cloth worlds of uneven size at once (940 k vertices), pass shape autotuned as the benchmark does
        {"name": "cloth_512_worlds", "work": "step", "scene": "worlds", "size": 512, "iterations": 5, "substeps": 1,
         "graph": True},
        # many tetrahedral cubes landing on the ground (155 k vertices, 583 k tets), autotuned
        {"name": "cubes_128_worlds", "work": "step", "scene": "cubes", "size": 128, "iterations": 8, "substeps": 1,
         "graph": True},
        # wind-driven cloth worlds, each iterated to a tenth of its initial residual, autotuned
        {"name": "wind_16_solve", "work": "solve", "size": 16, "side": 128, "tolerance": 0.1, "most": 40},
        # the warm start of the headline batch: 1,048,576 particles, 32 low-pass sweeps
        {"name": "warm_64_worlds", "work": "warm", "size": 64, "side": 128, "sweeps": 32},
        # network inference on the headline batch's rows
        {"name": "mlp_1m", "work": "mlp", "rows": 1048576},
        # one training step on a 128x128 cloth's rows
        {"name": "train_16k", "work": "train", "rows": 16384},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["hanging", "springs", "drop", "moving", "layers", "worlds", "cubes", "solve", "warm", "mlp",
                       "train"])
    if kind in ("hanging", "springs", "drop", "moving", "layers"):
        lo, hi = {"hanging": (12, 160), "springs": (24, 200), "drop": (32, 256), "moving": (32, 256),
                  "layers": (24, 128)}[kind]
        return {"work": "step", "scene": kind, "size": _log_int(rng, lo, hi), "iterations": rng.randint(3, 10),
                "substeps": rng.choice([1, 1, 2]) if kind != "moving" else 1, "graph": rng.random() < 0.7}
    if kind == "worlds":
        return {"work": "step", "scene": kind, "size": _log_int(rng, 8, 512), "iterations": 5, "substeps": 1,
                "graph": True}
    if kind == "cubes":
        return {"work": "step", "scene": kind, "size": _log_int(rng, 2, 128), "iterations": 8, "substeps": 1,
                "graph": True}
    if kind == "solve":
        return {"work": "solve", "size": _log_int(rng, 2, 16), "side": rng.randint(40, 128),
                "tolerance": rng.choice([0.3, 0.1]), "most": rng.randint(8, 40)}
    if kind == "warm":
        return {"work": "warm", "size": _log_int(rng, 1, 64), "side": rng.randint(48, 128),
                "sweeps": rng.choice([0, 8, 32])}
    if kind == "mlp":
        return {"work": "mlp", "rows": _log_int(rng, 1000, 1000000)}
    return {"work": "train", "rows": _log_int(rng, 1000, 150000)}


# ---- scenes -------------------------------------------------------------------------------------------------


def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "graph", "substeps")))


@functools.lru_cache(maxsize=16)
def _scene(key):
    """Model, solver, pipeline and step parameters of a case: what a program builds once."""
    case = dict(key)
    kind = case.get("scene", case["work"])
    n = case["size"]
    full, kw = False, {}
    if kind == "hanging":
        model, _, info = scenes.cloth_hanging(DEV, verts_per_side=n)
    elif kind in ("drop", "springs"):
        model, _, info = scenes.cloth_drop_on_sphere(DEV, verts_per_side=n, springs=kind == "springs")
    elif kind == "moving":
        model, _, info = scenes.cloth_on_moving_sphere(DEV, verts_per_side=n)
        full, kw = True, {"integrate_with_external_rigid_solver": True}
    elif kind == "layers":
        model, _, info = scenes.cloth_layers_on_sphere(DEV, verts_per_side=n)
        kw = info["solver_kwargs"]
    elif kind == "worlds":
        model, _, info = scenes.cloth_batched(DEV, worlds=n)
    elif kind == "cubes":
        model, _, info = scenes.soft_cubes_batched(DEV, worlds=n)
    else:
        model, _, info = scenes.cloth_wind_batched(DEV, worlds=n, verts_per_side=case["side"])
    pipe = None
    if model.shape_count:
        pipe = CollisionPipeline(model, soft_contact_margin=CONTACT_MARGIN, enable_rigid_soft_full_surface_contact=full)
    if pipe is not None and full:
        kw = dict(kw, soft_contact_capacity=pipe.soft_contact_max)
    solver = SolverVBD(model, iterations=case.get("iterations", info["iterations"]), **kw)
    out = {"kind": kind, "model": model, "solver": solver, "pipe": pipe, "info": info, "dt": info["dt"],
           "contacts": pipe.contacts() if pipe is not None else None, "tuned": kind not in ("worlds", "cubes", "solve")}
    if kind == "warm":
        out["warm"] = LearnedWarmStart(model, info["dt"], WarmStartMLP(DEV, seed=5), delta_sweeps=case["sweeps"])
    return out


def _waves(g, x, modes=6, shortest=0.3):
    """A smooth random field on the points x, about unit amplitude."""
    k = torch.randn((3, modes), generator=g, device=DEV)
    k = k / k.norm(dim=0) * (2.0 * math.pi / (shortest * (1.0 + 3.0 * torch.rand(modes, generator=g, device=DEV))))
    amp = torch.randn((modes, 3), generator=g, device=DEV) / math.sqrt(modes)
    return torch.sin(x @ k + 6.3 * torch.rand(modes, generator=g, device=DEV)) @ amp


def _drape(x, z, ball, ground, lift):
    """A sheet over a ball and the ground: its cap on the ball, a 35 degree cone from there down, then flat; the
    horizontal coordinates halfway between unstretched radii and unchanged ones."""
    a = math.radians(35.0)
    r = torch.sqrt(x * x + z * z).clamp(min=1e-6)
    r0, h0 = ball * math.sin(a), ball * math.cos(a)
    s0, s1 = ball * a, ball * a + (h0 - ground) / math.sin(a)
    cone = (r - s0).clamp(min=0.0)
    rho = torch.where(r < s0, ball * torch.sin(r / ball),
                      torch.where(r < s1, r0 + cone * math.cos(a), r0 + (s1 - s0) * math.cos(a) + r - s1))
    rho = 0.5 * (rho + r)
    y_ball = torch.sqrt((ball * ball - rho * rho).clamp(min=0.0))
    y = torch.where(rho < r0, y_ball, (h0 - (rho - r0) * math.tan(a)).clamp(min=ground)) + lift
    return rho / r * x, y, rho / r * z


def _start(sc, seed):
    """Positions, velocities and external forces of a state."""
    m, kind = sc["model"], sc["kind"]
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    q = m.particle_q.clone()
    free = ((m.particle_flags & 1) != 0) & (m.particle_inv_mass != 0)
    qd = 0.3 * _waves(g, q)
    if kind in ("drop", "springs", "moving", "layers"):
        # particle radius 0.1: the sheet touches at 0.5 from the ball's centre and 0.1 above the ground
        gap = 0.008
        layer = torch.round((q[:, 1] - q[0, 1]) / gap)
        x, y, z = _drape(q[:, 0], q[:, 2], 0.5, 0.1, -1.0e-3)
        if kind == "layers":  # folds: the upper sheet comes within the contact radius here and there
            y = y + gap * layer * (0.9 - 0.55 * _waves(g, q)[:, 0].clamp(0.0, 1.0))
        q = torch.stack([x, y, z], dim=1)
        q = q + 2.0e-4 * _waves(g, q) + 5.0e-5 * torch.randn(q.shape, generator=g, device=DEV)
        qd = 0.3 * qd - torch.tensor([0.0, 0.1, 0.0], device=DEV)
    elif kind in ("cubes", "worlds"):
        # landing: each world's lowest part just inside the ground's contact range
        w = m.particle_world.long()
        low = torch.full((int(w.max()) + 1,), 1.0e9, device=DEV).scatter_reduce(0, w, q[:, 1], "amin")
        q[:, 1] += (0.009 if kind == "cubes" else 0.098) - low[w]
        q = q + 5.0e-4 * _waves(g, q)
        if kind == "worlds":
            q = q + 1.0e-4 * torch.randn(q.shape, generator=g, device=DEV)
        qd = qd - torch.tensor([0.0, 0.5, 0.0], device=DEV)
    else:
        # the residual-driven solves start from smooth fields: rough ones are gone after two or three sweeps
        rough = 1.0e-4 * (kind == "hanging")
        q = torch.where(free[:, None], q + 4.0e-3 * _waves(g, q) + rough * torch.randn(q.shape, generator=g, device=DEV), q)
    qd = torch.where(free[:, None], qd, torch.zeros_like(qd))
    f = 2.0 * _waves(g, q, shortest=0.5) * m.particle_mass[:, None]
    return q.contiguous(), qd.contiguous(), f.contiguous()


def prepare(case, seed):
    if case["work"] in ("mlp", "train"):
        g = torch.Generator(device=DEV).manual_seed(int(seed))
        n = case["rows"]
        feat = torch.randn((n, 48), generator=g, device=DEV).to(torch.bfloat16).view(torch.int16)
        mlp = WarmStartMLP(DEV, seed=int(seed))
        if case["work"] == "mlp":
            return {"work": "mlp", "mlp": mlp, "feat": feat, "out": torch.empty((n, 3), device=DEV)}
        target = 0.5 * torch.randn((n, 3), generator=g, device=DEV)
        weight = (torch.rand(n, generator=g, device=DEV) > 0.05).float()
        return {"work": "train", "mlp": mlp, "feat": feat, "target": target, "weight": weight}

    sc = _scene(_key(case))
    m = sc["model"]
    q, qd, f = _start(sc, seed)
    a, b = m.state(), m.state()
    a.particle_f = b.particle_f = f
    s = {"work": case["work"], "scene": sc, "a": a, "b": b, "q": q, "qd": qd, "graph": None}
    if case["work"] == "solve":
        s.update(tolerance=case["tolerance"], most=case["most"])
    if case["work"] == "warm":
        g = torch.Generator(device=DEV).manual_seed(int(seed) + 1000003)
        s["corr"] = 1.0e-5 * _waves(g, q)
        s["corr"][m.particle_inv_mass == 0] = 0.0
    if sc["kind"] == "moving":
        t = torch.zeros((), device=DEV)
        a.body_q, b.body_q = sc["info"]["body_pose"](t), sc["info"]["body_pose"](t + sc["dt"])
    if not sc["tuned"]:
        a.particle_q.copy_(q)
        a.particle_qd.copy_(qd)
        if sc["pipe"] is not None:
            sc["pipe"].collide(a, sc["contacts"])
        sc["solver"].autotune(a, sc["contacts"], sc["dt"])
        sc["tuned"] = True
    if case["work"] == "step":
        s["substeps"] = case["substeps"]
        if case["graph"]:
            stream = torch.cuda.Stream()
            stream.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(stream):
                _frame(s)
                torch.cuda.synchronize()
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=stream):
                    _frame(s)
            torch.cuda.current_stream().wait_stream(stream)
            s["graph"] = graph
    return s


def _frame(s):
    sc, a, b = s["scene"], s["a"], s["b"]
    a.particle_q.copy_(s["q"])
    a.particle_qd.copy_(s["qd"])
    for _ in range(s["substeps"]):
        sc["pipe"].collide(a, sc["contacts"])
        sc["solver"].step(a, b, None, sc["contacts"], sc["dt"])
        a, b = b, a
    s["last"] = a


def run(s):
    if s["work"] == "mlp":
        return s["mlp"].forward(s["feat"], s["out"])
    if s["work"] == "train":
        loss = s["mlp"].train_step(s["feat"], s["target"], s["weight"])
        return [loss, s["mlp"].grad, s["mlp"].params]
    if s["work"] == "step":
        if s["graph"] is not None:
            s["graph"].replay()
        else:
            _frame(s)
        return [s["last"].particle_q, s["last"].particle_qd]
    sc, a, b = s["scene"], s["a"], s["b"]
    a.particle_q.copy_(s["q"])
    a.particle_qd.copy_(s["qd"])
    if s["work"] == "solve":
        r = sc["solver"].step_to_residual_worlds(a, b, None, None, sc["dt"], rel_tol=s["tolerance"],
                                                 max_iterations=s["most"])
        return [b.particle_q, b.particle_qd, r["world_iterations"]]
    sc["warm"].corr = s["corr"]
    sc["solver"].begin_step(a, None, sc["dt"])
    return sc["warm"](sc["solver"], a, sc["dt"])


# ---- what a pass cannot do without ----------------------------------------------------------------------------

# FP32 operations of one vertex's share of an element's force and Hessian (a division or square root as one)
FLOPS_TRI, FLOPS_HINGE, FLOPS_TET, FLOPS_SPRING, FLOPS_SOLVE = 210, 330, 420, 90, 70
FLOPS_ROW = 2 * (48 * 128 + 128 * 128 + 128 * 128 + 128 * 3)


def work(case):
    if case["work"] == "mlp":
        n = case["rows"]
        return {"bytes": n * (96 + 12) + 4 * 39683, "flops": n * FLOPS_ROW}
    if case["work"] == "train":
        n = case["rows"]
        return {"bytes": n * (96 + 12 + 4) + 8 * 4 * 39683, "flops": 3 * n * FLOPS_ROW}
    m = _scene(_key(case))["model"]
    n = m.particle_count
    if case["work"] == "warm":
        # positions, velocities, forces, corrections, mass, area, 1-ring in; two candidates and the step's state out
        ring = 6.0 * n
        return {"bytes": n * (4 * 12 + 8) + 4 * ring + n * (24 + 36),
                "flops": n * FLOPS_ROW + 60 * ring + case["sweeps"] * 6 * (ring + n)}
    elements = 44 * m.tri_count + 32 * m.edge_count + 64 * m.tet_count + 20 * m.spring_count
    solid = m.tet_count > 0  # the cubes' surface triangles and edges carry no material
    per_iteration = (FLOPS_TET * 4 * m.tet_count if solid else FLOPS_TRI * 3 * m.tri_count + FLOPS_HINGE * 4 * m.edge_count)
    per_iteration += FLOPS_SPRING * 2 * m.spring_count + FLOPS_SOLVE * n
    if case["work"] == "solve":
        its, subs = case["most"] // 2, 1  # the worlds stop at counts of their own
    else:
        its, subs = case["iterations"], case["substeps"]
    return {"bytes": elements + n * (16 + 36 + 24), "flops": subs * its * per_iteration}


# About four times what the path differs from exact() on an MI355X: the largest is a step's velocities, 6e-5 after
# one substep and 2.5e-4 after ten (positions are rounded to 1e-7 of a metre and divided by a step of 1/600 s);
# 5e-3 for the network's BF16 products and gradients; 4e-8 for the candidates of a warm start
def tolerance(case):
    if case["work"] == "mlp":
        return {"rel": 2.0e-2}
    if case["work"] == "train":
        return {"rel": 2.0e-2}
    if case["work"] == "warm":
        return {"rel": 1.5e-7}
    if case["work"] == "solve":
        # a world near its tolerance may stop one iteration earlier or later
        return {"rel": 1.0e-3, "differ": 0.1}
    return {"rel": 1.0e-3 if case["substeps"] > 2 else 3.0e-4}


# ---- the same in 64 bits, in plain torch ------------------------------------------------------------------------


def exact(case, seed):
    if case["work"] in ("mlp", "train"):
        return _exact_mlp(case, seed)
    sc = _scene(_key(case))
    m = sc["model"]
    if case["work"] == "warm":
        return _exact_warm(case, seed, sc)
    if case["work"] == "solve" or case["scene"] in ("moving", "layers"):
        # no such value: the iteration counts, the contact lists of the self-contact detection and the fixed-count
        # line searches of edge and face contacts follow comparisons of rounded numbers
        return None
    q, qd, f = (t.double() for t in _start(sc, seed))
    return _exact_steps(case, m, q, qd, f, sc["dt"])


def _mlp64(feat, params):
    x, at = feat, 0
    for k, (i, o) in enumerate(((48, 128), (128, 128), (128, 128), (128, 3))):
        w, b = params[at:at + i * o].reshape(i, o), params[at + i * o:at + i * o + o]
        at += i * o + o
        x = x @ w + b
        if k < 3:
            x = x * torch.sigmoid(x)
    return x


def _exact_mlp(case, seed):
    s = prepare(case, seed)
    params = s["mlp"].params.double().requires_grad_(case["work"] == "train")
    feat = s["feat"].view(torch.bfloat16).double()
    if case["work"] == "mlp":
        return torch.cat([_mlp64(x, params) for x in feat.split(131072)])
    total, n = 0.0, case["rows"]
    for x, t, w in zip(feat.split(131072), s["target"].double().split(131072), s["weight"].double().split(131072)):
        part = (w[:, None] * (_mlp64(x, params) - t) ** 2).sum() / (3.0 * n)
        part.backward()
        total = total + part.detach()
    grad = params.grad
    # the first Adam step from zero moments
    return [total.reshape(1), grad, params.detach() - 1e-3 * grad / (grad.abs() + 1e-8)]


def _exact_warm(case, seed, sc):
    ws, m, dt = sc["warm"], sc["model"], sc["dt"]
    x0, qd, f = (t.double() for t in _start(sc, seed))
    s = prepare(case, seed)
    c = s["corr"].double()
    w = m.particle_inv_mass.double()[:, None]
    free = (((m.particle_flags & 1) != 0) & (m.particle_inv_mass != 0))[:, None]
    acc = f * w
    y = torch.where(free, x0 + (qd + (m.gravity[0].double() + acc) * dt) * dt, x0)
    off, nbr = ws.nbr_off.long(), ws.nbr.long()
    deg = off[1:] - off[:-1]
    row = torch.repeat_interleave(torch.arange(len(deg), device=DEV), deg)
    inv = (1.0 / deg.double())[:, None]
    sd, scc, sl, mm, ma = (float(v) for v in ws.scales.double())
    a, cc = (y - x0) / sd, c / scc

    def total(v):
        return torch.zeros((len(deg),) + v.shape[1:], dtype=torch.float64, device=DEV).index_add_(0, row, v)

    def most(v, how):
        i = row[:, None].expand(-1, v.shape[1]) if v.dim() == 2 else row
        return torch.zeros((len(deg),) + v.shape[1:], dtype=torch.float64, device=DEV).scatter_reduce(0, i, v, how, include_self=False)

    dx = x0[nbr] - x0[row]
    ln, ac = dx.norm(dim=1) / sl, cc.norm(dim=1)
    pin = (m.particle_mass[nbr] == 0).double()
    feat = torch.cat([
        a, cc, total(a[nbr]) * inv - a, total(cc[nbr]) * inv - cc, most(a[nbr], "amax") - a, most(a[nbr], "amin") - a,
        most(cc[nbr], "amax") - cc, most(cc[nbr], "amin") - cc, total(dx) * inv / sl, total(ln)[:, None] * inv,
        most(ln, "amax")[:, None], most(ln, "amin")[:, None], acc * dt * dt / sd, a.norm(dim=1)[:, None], ac[:, None],
        total(ac[nbr])[:, None] * inv, most(ac[nbr], "amax")[:, None], m.particle_mass.double()[:, None] / mm,
        ws.area.double()[:, None] / ma, total(pin)[:, None] * inv, deg.double()[:, None] / 6.0,
        total(y[nbr] - y[row]) * inv / sl, total(dx * pin[:, None]) * inv / sl, torch.ones_like(inv)], dim=1)
    params = ws.mlp.params.double()
    delta = torch.cat([_mlp64(x, params) for x in feat.split(131072)]) * (ws.blend * scc)
    active = free.double()
    for _ in range(case["sweeps"]):
        delta = active * (delta + total((active * delta)[nbr])) / (1.0 + deg.double())[:, None]
    return [y + c, y + c + delta]


def _outer(a, b):
    return a[:, :, None] * b[:, None, :]


def _dot(a, b):
    return (a * b).sum(dim=1)


def _membrane(q, x0, i, slot, pose, area, mu, lam, kd, dt):
    def columns(x):
        e1, e2 = x[i[:, 1]] - x[i[:, 0]], x[i[:, 2]] - x[i[:, 0]]
        return (e1 * pose[:, 0, 0, None] + e2 * pose[:, 1, 0, None], e1 * pose[:, 0, 1, None] + e2 * pose[:, 1, 1, None])

    f0, f1 = columns(q)
    a, b, c = _dot(f0, f0), _dot(f1, f1), _dot(f0, f1)
    area_ratio = (a * b - c * c).clamp(min=1e-20).sqrt()
    el = lam + mu
    s = el * (area_ratio - 1.0 - mu / el)
    g0 = (f0 * b[:, None] - f1 * c[:, None]) / area_ratio[:, None]
    g1 = (f1 * a[:, None] - f0 * c[:, None]) / area_ratio[:, None]
    sign = torch.stack([(slot == 1).double() - (slot == 0).double(), (slot == 2).double() - (slot == 0).double()], dim=1)
    d = torch.einsum("nk,nkj->nj", sign, pose)  # dF columns / dx
    d0, d1 = d[:, :1], d[:, 1:]
    force = -((mu[:, None] * f0 + s[:, None] * g0) * d0 + (mu[:, None] * f1 + s[:, None] * g1) * d1)
    r = (s.clamp(min=0.0) / area_ratio)[:, None]
    dj, w = g0 * d0 + g1 * d1, f1 * d0 - f0 * d1
    eye = torch.eye(3, dtype=torch.float64, device=DEV)
    h = (mu[:, None] * (d0 * d0 + d1 * d1) + r * _dot(w, w)[:, None])[:, :, None] * eye
    h = h + (el[:, None] - r)[:, :, None] * _outer(dj, dj) - r[:, :, None] * _outer(w, w)
    p0, p1 = columns(x0)
    r00, r01, r11 = ((u - v) / dt for u, v in ((a, _dot(p0, p0)), (c, _dot(p0, p1)), (b, _dot(p1, p1))))
    k00, k01, k11 = 2.0 * d0 * f0, d0 * f1 + d1 * f0, 2.0 * d1 * f1
    force = force - kd[:, None] * (k00 * r00[:, None] + 2.0 * k01 * r01[:, None] + k11 * r11[:, None])
    h = h + (kd / dt)[:, None, None] * (_outer(k00, k00) + 2.0 * _outer(k01, k01) + _outer(k11, k11))
    return area[:, None] * force, area[:, None, None] * h


def _angle(p):
    x0, x1, x2, x3 = p.unbind(1)
    n1, n2 = torch.linalg.cross(x2 - x0, x3 - x0), torch.linalg.cross(x3 - x1, x2 - x1)
    n1, n2, e = (v / v.norm(dim=1, keepdim=True) for v in (n1, n2, x3 - x2))
    return torch.atan2(_dot(torch.linalg.cross(n1, n2), e), _dot(n1, n2))


def _hinge(q, x0, i, slot, rest, length, ke, kd, dt):
    p = q[i].requires_grad_(True)
    theta = _angle(p)
    d = torch.autograd.grad(theta.sum(), p)[0][torch.arange(len(slot), device=DEV), slot]
    theta, p = theta.detach(), p.detach()
    turn = theta - _angle(x0[i])
    turn = torch.where(turn > math.pi, turn - 2 * math.pi, torch.where(turn < -math.pi, turn + 2 * math.pi, turn))
    k = ke * length
    force = -(k * (theta - rest) + kd * length * turn / dt)[:, None] * d
    return force, (k + kd * length / dt)[:, None, None] * _outer(d, d)


def _tet(q, i, slot, dm, mu, lam):
    vol = 1.0 / (6.0 * torch.linalg.det(dm))
    x = q[i]
    f = (x[:, 1:] - x[:, :1]).transpose(1, 2) @ dm
    j = torch.linalg.det(f)
    cof = torch.stack([torch.linalg.cross(f[:, :, 1], f[:, :, 2]), torch.linalg.cross(f[:, :, 2], f[:, :, 0]),
                       torch.linalg.cross(f[:, :, 0], f[:, :, 1])], dim=2)
    el = lam + mu
    stress = mu[:, None, None] * f + (el * (j - 1.0 - mu / el))[:, None, None] * cof
    w = torch.cat([-dm.sum(dim=1, keepdim=True), dm], dim=1)[torch.arange(len(slot), device=DEV), slot]
    cw = (cof @ w[:, :, None])[:, :, 0]
    eye = torch.eye(3, dtype=torch.float64, device=DEV)
    h = (mu * _dot(w, w))[:, None, None] * eye + el[:, None, None] * _outer(cw, cw)
    return -vol[:, None] * (stress @ w[:, :, None])[:, :, 0], vol[:, None, None] * h


def _spring(q, x0, i, end, rest, ke, kd, dt):
    d, d0 = q[i[:, 0]] - q[i[:, 1]], x0[i[:, 0]] - x0[i[:, 1]]
    ln = d.norm(dim=1).clamp(min=1e-8)
    u = d / ln[:, None]
    pull = ke * (rest - ln) - kd / dt * (ln - d0.norm(dim=1).clamp(min=1e-8))
    eye = torch.eye(3, dtype=torch.float64, device=DEV)
    uu = _outer(u, u)
    h = ke[:, None, None] * (eye - (rest / ln)[:, None, None] * (eye - uu)) + (kd / dt)[:, None, None] * uu
    return (1.0 - 2.0 * end.double())[:, None] * pull[:, None] * u, h


def _turn(quat, v):
    u, w = quat[:3].expand_as(v), quat[3]
    t = 2.0 * torch.linalg.cross(u, v)
    return v + w * t + torch.linalg.cross(u, t)


def _touching(m, x):
    """Soft contacts of the positions x: (particle, point on the shape, normal, shape) per shape."""
    out = []
    for s in range(m.shape_count):
        t = m.shape_transform[s].double()
        up = _turn(t[3:], torch.tensor([[0.0, 0.0, 1.0]], dtype=torch.float64, device=DEV))
        rel = x - t[:3]
        if int(m.shape_type[s]) == 3:
            ln = rel.norm(dim=1, keepdim=True)
            dist, n = ln[:, 0] - float(m.shape_scale[s, 0]), rel / ln
        else:
            dist, n = (rel * up).sum(dim=1), up.expand_as(rel)
        reach = CONTACT_MARGIN + float(m.shape_margin[s]) + m.particle_radius.double()
        p = ((dist < reach) & ((m.particle_flags & 1) != 0)).nonzero()[:, 0]
        out.append((p, (x - n * dist[:, None])[p], n[p], s))
    return out


def _contact(m, q, x0, p, at, n, s, eps, dt):
    ke = 0.5 * (m.soft_contact_ke + float(m.shape_material_ke[s]))
    kd = 0.5 * (m.soft_contact_kd + float(m.shape_material_kd[s]))
    mu = math.sqrt(m.soft_contact_mu * float(m.shape_material_mu[s]))
    depth = m.particle_radius.double()[p] + float(m.shape_margin[s]) - _dot(n, q[p] - at)
    u = q[p] - x0[p]
    un = _dot(n, u)
    nn = _outer(n, n)
    fn = depth * ke
    damp = torch.where(un < 0.0, kd / dt, 0.0)
    force = n * (fn - damp * un)[:, None]
    h = (ke + damp)[:, None, None] * nn
    ut = u - n * un[:, None]
    size, e = ut.norm(dim=1), eps * dt
    scale = mu * fn * torch.where(size > e, 1.0 / size.clamp(min=1e-30), (2.0 - size / e) / e)
    scale = torch.where(size > 0.0, scale, torch.zeros_like(scale))
    force = force - scale[:, None] * ut
    h = h + scale[:, None, None] * (torch.eye(3, dtype=torch.float64, device=DEV) - nn)
    on = (depth > 0.0).double()
    return on[:, None] * force, on[:, None, None] * h


def _exact_steps(case, m, q, qd, f, dt):
    mass, w = m.particle_mass.double(), m.particle_inv_mass.double()[:, None]
    free = (((m.particle_flags & 1) != 0) & (m.particle_inv_mass != 0))
    tri, hinge = m.tri_indices.long().reshape(-1, 3), m.edge_indices.long().reshape(-1, 4)
    tet, spring = m.tet_indices.long().reshape(-1, 4), None
    tm, bend, tetm = m.tri_materials.double(), m.edge_bending_properties.double(), m.tet_materials.double()
    pose, area, dm = m.tri_poses.double(), m.tri_areas.double(), m.tet_poses.double()
    rest, length = m.edge_rest_angle.double(), m.edge_rest_length.double()
    if m.spring_count:
        spring = m.spring_indices.long().reshape(-1, 2)
        srest, ske, skd = m.spring_rest_length.double(), m.spring_stiffness.double(), m.spring_damping.double()
    color = torch.empty(len(q), dtype=torch.long, device=DEV)
    groups = [g.long() for g in m.particle_color_groups]
    for c, g in enumerate(groups):
        color[g] = c
    tri_on = (tm[:, 0] > 0) | (tm[:, 1] > 0)
    hinge_on = (bend[:, 0] > 0) & (hinge[:, 0] >= 0) & (hinge[:, 1] >= 0)

    def of(c, idx, on):
        hit = (color[idx.clamp(min=0)] == c) & free[idx.clamp(min=0)]
        return (hit & on[:, None]).nonzero().unbind(1)

    plans = []
    for c in range(len(groups)):
        plans.append((of(c, tri, tri_on), of(c, hinge, hinge_on),
                      of(c, tet, torch.ones(len(tet), dtype=torch.bool, device=DEV)),
                      of(c, spring, torch.ones(len(spring), dtype=torch.bool, device=DEV)) if spring is not None else None))
    eye = torch.eye(3, dtype=torch.float64, device=DEV)
    for _ in range(case["substeps"]):
        touch = _touching(m, q)
        x0 = q
        y = torch.where(free[:, None], q + (qd + (m.gravity[0].double() + f * w) * dt) * dt, q)
        d = y - x0
        q = y.clone()
        for _ in range(case["iterations"]):
            for c, (ti, hi, ki, si) in enumerate(plans):
                force = (mass / dt ** 2)[:, None] * (y - q)
                h = (mass / dt ** 2)[:, None, None] * eye.repeat(len(q), 1, 1)

                def add(who, fe, he):
                    force.index_add_(0, who, fe)
                    h.index_add_(0, who, he)

                if len(ti[0]):
                    t, k = ti
                    add(tri[t, k], *_membrane(q, x0, tri[t], k, pose[t], area[t], tm[t, 0], tm[t, 1], tm[t, 2], dt))
                if len(hi[0]):
                    t, k = hi
                    add(hinge[t, k], *_hinge(q, x0, hinge[t], k, rest[t], length[t], bend[t, 0], bend[t, 1], dt))
                if len(ki[0]):
                    t, k = ki
                    add(tet[t, k], *_tet(q, tet[t], k, dm[t], tetm[t, 0], tetm[t, 1]))
                if si is not None and len(si[0]):
                    t, k = si
                    add(spring[t, k], *_spring(q, x0, spring[t], k, srest[t], ske[t], skd[t], dt))
                for p, at, n, s in touch:
                    add(p, *_contact(m, q, x0, p, at, n, s, 1e-2, dt))
                g = groups[c][free[groups[c]]]
                d = d.clone()
                d[g] += torch.linalg.solve(h[g], force[g])
                q = torch.where(free[:, None], x0 + d, x0)
        qd = (q - x0) / dt
    return [q, qd]
