"""The hydro step's performance cases: what a user of this framework has it do, through luna_hydro's public entry points.

A pass is a few steps (static: time_step + step; moving: time_step, moving_begin, the new mesh, moving_finish; a line: the
fused step), a derivative of a step, or a batch of the limiter network's training, from the same state each time. Meshes are
jittered-lattice Voronoi meshes of this repository's producer and states are flows in motion (waves with a blast, a shear
layer), both drawn from the seed. exact() restates the scheme in plain torch in 64 bits.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "luna-cpp_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

from luna_hydro import autograd, hydro, learned, mesh as meshlib, problems  # noqa: E402

GAMMA = 5.0 / 3.0


def listed():
    return [
        # the 1D Sod tube at its usual 1024 cells, a run's steps one launch each: the smallest calls, latency alone counts
        {"name": "line_sod", "kind": "line", "cells": 1024, "limiter": "minmod", "riemann": "hllc", "steps": 64},
        # a 3D test-sized blast (the size of a parameter study or a test run): a few thousand cells, launches count
        {"name": "blast_small", "kind": "static", "dim": 3, "n": 19, "precision": "double", "riemann": "hllc", "hll": 0.0, "steps": 8},
        # the drivers' default precision in 2D (grad32) on a shear layer, LUNA's time-step rule, an odd size
        {"name": "shear_grad32", "kind": "static", "dim": 2, "n": 511, "precision": "grad32", "riemann": "hllc", "hll": 0.0, "steps": 4},
        # the drivers' default precision in 3D (grad16), the other Riemann solver
        {"name": "blast_grad16", "kind": "static", "dim": 3, "n": 72, "precision": "grad16", "riemann": "hll", "hll": 0.0, "steps": 4},
        # the static headline: the blast at 128^3 in double
        {"name": "blast_static", "kind": "static", "dim": 3, "n": 128, "precision": "double", "riemann": "hllc", "hll": 0.0, "steps": 4},
        # the moving headline: a whole moving step with the geometry pass of the new mesh, a GPU mesh producer's arrays in place
        {"name": "blast_moving", "kind": "moving", "dim": 3, "n": 104, "precision": "double", "riemann": "hllc", "hll": 0.0, "limiter": "face"},
        # the moving mesh with the HLL fallback at compressions, as the strong-blast runs take it, mid-sized and odd
        {"name": "blast_moving_hll", "kind": "moving", "dim": 3, "n": 47, "precision": "double", "riemann": "hllc", "hll": 1.0, "limiter": "face"},
        # the learned limiter on the moving shear layer it was made for
        {"name": "shear_learned", "kind": "moving", "dim": 2, "n": 384, "precision": "double", "riemann": "hllc", "hll": 0.0, "limiter": "learned"},
        # forward mode: a time step and a step with the tangent of the state
        {"name": "tangent", "kind": "tangent", "dim": 3, "n": 80, "riemann": "hllc"},
        # reverse mode: the gradient of a loss through a checkpointed rollout of steps
        {"name": "rollout_gradient", "kind": "gradient", "dim": 3, "n": 56, "riemann": "hllc", "steps": 4, "every": 2},
        # the reverse of a moving step, on the host mesh producer's geometry derivatives (the acoustic inverse problem's step)
        {"name": "moving_adjoint", "kind": "moving_adjoint", "dim": 3, "n": 20, "riemann": "hllc"},
        # the limiter network: a training batch's loss and gradient, and its fractions
        {"name": "network_batch", "kind": "network", "rows": 65536},
    ]


def _between(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["line", "static", "static", "static", "moving", "moving", "tangent", "gradient", "network"])
    riemann = rng.choice(["hllc", "hllc", "hll"])
    if kind == "line":
        return {"kind": kind, "cells": _between(rng, 200, 4096), "limiter": rng.choice(["face", "minmod", "vanleer"]), "riemann": riemann,
                "steps": rng.randint(16, 64)}
    if kind == "network":
        return {"kind": kind, "rows": _between(rng, 1000, 500000)}
    dim = rng.choice([2, 3, 3])
    top = {"static": 120, "moving": 88, "tangent": 80, "gradient": 56}[kind]
    n = _between(rng, 14, top) if dim == 3 else _between(rng, 40, 6 * top)
    if kind == "tangent":
        return {"kind": kind, "dim": dim, "n": n, "riemann": riemann}
    if kind == "gradient":
        return {"kind": kind, "dim": dim, "n": n, "riemann": riemann, "steps": rng.randint(2, 5), "every": rng.randint(1, 3)}
    case = {"kind": kind, "dim": dim, "n": n, "precision": rng.choice(["double", "double", "grad32", "grad16"]), "riemann": riemann, "hll": 0.0}
    if kind == "static":
        case["steps"] = rng.randint(2, 4)
    else:
        case["limiter"] = rng.choice(["face", "face", "learned"])
        if case["limiter"] == "learned":
            case["precision"] = "double"
    if riemann == "hllc" and case["precision"] == "double" and case.get("limiter", "face") == "face" and rng.random() < 0.3:
        case["hll"] = 1.0
    return case


# ------------------------------------------------------------------------------------------------------------- inputs


def _rng(seed):
    return np.random.Generator(np.random.MT19937(seed))


def _waves(rng, x, count=4, top=3):
    """A smooth periodic field of unit order: `count` plane waves of whole wave numbers up to `top`."""
    out = np.zeros(len(x))
    for _ in range(count):
        k = rng.integers(-top, top + 1, x.shape[1])
        k[rng.integers(x.shape[1])] = rng.integers(1, top + 1)
        out += rng.uniform(0.3, 1.0) * np.sin(2 * np.pi * (x @ k + rng.uniform()))
    return out / count


def _state(m, seed, calm=False):
    """Q of a flow in motion on mesh m. 3D: waves in every variable and a blast of 50 times the pressure; 2D: a shear layer
    (density 2 against 1, velocities +-0.5) with waves; calm: waves alone (a differentiable flow)."""
    rng = _rng(seed + 1000)
    D, N = m["dim"], m["cells"]
    x = m["positions"] + m["centroid"]
    W = np.empty((N, D + 2))
    W[:, 0] = 1 + 0.2 * _waves(rng, x)
    for a in range(D):
        W[:, 1 + a] = 0.3 * _waves(rng, x)
    W[:, D + 1] = 1 + 0.2 * _waves(rng, x)
    if not calm and D == 3:
        d = x - rng.uniform(0.3, 0.7, D)
        d -= np.round(d)
        W[np.sqrt((d * d).sum(axis=1)) < 0.2, D + 1] *= 50.0
    if not calm and D == 2:
        layer = np.tanh((0.25 - np.abs(x[:, 1] % 1.0 - 0.5)) / 0.02)
        W[:, 0] *= 1.5 + 0.5 * layer
        W[:, 1] += 0.5 * layer
        W[:, D + 1] *= 2.5
    return problems.conserved_rows(W, GAMMA) * m["volume"][:, None]


def _mesh(case, seed):
    return meshlib.build(problems.jittered_lattice(case["n"], case["dim"], 0.25, seed + 1), 1.0)


def _rule(dim):
    return "luna" if dim == 2 else "arepo"


def _courant(dim):
    return 0.4 if dim == 2 else 0.3


def _rows(case, seed):
    """A training batch: features as the sweep records them (scale-free, within [-8, 8]), targets in [0, 1], weights."""
    rng = _rng(seed)
    x = np.clip(rng.normal(0.3, 0.8, (case["rows"], learned.FEATURES)), -8, 8).astype(np.float32)
    bits = (x.view(np.uint32) >> 16).astype(np.uint16)
    target = np.clip(0.8 - 0.4 * x[:, 8] + 0.2 * x[:, 3] + rng.normal(0, 0.1, case["rows"]), 0, 1)  # a fraction that falls with the jump
    return bits, target.astype(np.float32), rng.uniform(0, 1, case["rows"]).astype(np.float32)


def _line(case, seed):
    pb = problems.problem_1d("sod")
    keys, step, period = problems.line_keys(problems.line_points(case["cells"], pb.L, 0.5, seed + 1), pb.L)
    q0 = problems.line_initial_state(pb, keys, step, period)
    a, b, vol = (np.array(v) for v in problems.line_cells(keys, step, period, pb.periodic))
    rng = _rng(seed + 1000)  # a pressure ripple, so that the whole line moves
    q0[:, 2] *= 1 + 0.1 * np.sin(2 * np.pi * (rng.integers(2, 6) * 0.5 * (a + b) + rng.uniform()))
    return pb, keys, step, period, q0, vol


def prepare(case, seed):
    kind = case["kind"]
    if kind == "line":
        pb, keys, step, period, q0, _ = _line(case, seed)
        line = hydro.Line(keys, period, step, pb.gamma, periodic=pb.periodic, walls=pb.walls, limiter=case["limiter"], riemann=case["riemann"])
        return {"kind": kind, "line": line, "q0": q0, "steps": case["steps"]}
    if kind == "network":
        x, t, w = learned.device_rows(*_rows(case, seed))
        return {"kind": kind, "trainer": learned.Trainer(params=_params(seed)), "x": x, "t": t, "w": w, "sum": float(w.sum().item())}
    dim = case["dim"]
    m = _mesh(case, seed)
    q0 = _state(m, seed, calm=kind in ("tangent", "gradient", "moving_adjoint"))
    s = {"kind": kind, "courant": _courant(dim)}
    if kind in ("static", "tangent", "gradient"):
        fv = hydro.FiniteVolume(m, GAMMA, riemann=case["riemann"], step_rule=_rule(dim), precision=case.get("precision", "double"),
                                hll_compression=case.get("hll", 0.0))
        s.update(fv=fv, solver=autograd.Solver(fv), q0=torch.tensor(q0, device="cuda"))
        if kind == "static":
            s["steps"] = case["steps"]
        else:
            fv.set_state(q0)
            s["dt"] = fv.time_step(s["courant"])
            s["dq"] = torch.tensor(_rows_like(q0, seed), device="cuda")
            if kind == "gradient":
                s["steps"], s["every"] = case["steps"], case["every"]
        return s
    fv = hydro.FiniteVolume(m, GAMMA, riemann=case["riemann"], step_rule=_rule(dim), motion="moving", precision=case.get("precision", "double"),
                            hll_compression=case.get("hll", 0.0), limiter=case.get("limiter", "face"))
    if case.get("limiter") == "learned":
        fv.set_limiter_network(learned.default_params())
    fv.set_state(q0)
    dt = fv.time_step(s["courant"])
    m1 = meshlib.build(fv.moving_begin(dt), 1.0)
    fv.moving_finish(m1, dt)
    if kind == "moving":
        s.update(fv=fv, solver=autograd.Solver(fv), q0=torch.tensor(q0, device="cuda"), mesh0=hydro.DeviceMesh(m), mesh1=hydro.DeviceMesh(m1))
        return s
    rng = _rng(seed + 2000)
    s.update(fv=fv, q0=q0, dt=dt, mesh0=m, mesh1=m1, qbar=_rows_like(q0, seed), xbar=rng.normal(size=(m["cells"], dim)))
    return s


def _params(seed):
    """Parameters in the middle of training: the shipped network's with seeded noise."""
    p = learned.default_params()
    return p + _rng(seed + 1000).normal(0, 0.02, p.size).astype(np.float32)


def _rows_like(q, seed):
    """A tangent (or bar) of Q of the size of Q itself."""
    return _rng(seed + 2000).normal(size=q.shape) * np.abs(q).mean(axis=0, keepdims=True)


def run(s):
    kind = s["kind"]
    if kind == "line":
        s["line"].set_state(s["q0"])
        dt, dts = s["line"].time_step(0.4, "luna"), []
        for _ in range(s["steps"]):
            dts.append(dt)
            dt = s["line"].step_and_time_step(dt, 0.4)
        return {"q": s["line"].state(), "dt": np.array(dts)}
    if kind == "network":
        loss, grad = s["trainer"].gradient(s["x"], s["t"], s["w"], s["sum"])
        return {"loss": loss, "gradient": grad, "fraction": s["trainer"].forward(s["x"])}
    fv = s["fv"]
    if kind == "static":
        s["solver"].set_state(s["q0"])
        dts = []
        for _ in range(s["steps"]):
            dts.append(fv.time_step(s["courant"]))
            fv.step(dts[-1])
        return {"q": s["solver"].state(), "dt": np.array(dts)}
    if kind == "moving":
        fv.set_geometry(s["mesh0"])
        s["solver"].set_state(s["q0"])
        dt = fv.time_step(s["courant"])
        fv.moving_begin(dt, positions=False)
        fv.set_geometry(s["mesh1"])
        fv.moving_finish(None, dt)
        return {"q": s["solver"].state(), "dt": dt, "fallbacks": fv.fallbacks()}
    if kind == "tangent":
        s["solver"].set_state(s["q0"])
        dq = s["dq"].clone()
        torch.cuda.synchronize()
        dt = fv.time_step_tangent(s["courant"], dq)
        fv.step_tangent(dt, dq)
        return {"q": s["solver"].state(), "dq": dq, "dt": dt}
    if kind == "gradient":
        q = s["q0"].clone().requires_grad_()
        out = autograd.rollout(q, s["solver"], [s["dt"]] * s["steps"], every=s["every"])
        (out * s["dq"]).sum().backward()
        return {"q": out.detach(), "gradient": q.grad}
    fv.set_state(s["q0"])
    qbar, xbar = fv.moving_adjoint(s["dt"], s["mesh0"], s["mesh1"], s["qbar"], s["xbar"])
    return {"qbar": qbar, "xbar": xbar}


# ------------------------------------------------------------------------------------------------------ what a pass needs


def _faces(case):
    """Faces per cell of a jittered lattice's Voronoi mesh (7.78 in 3D, 3 in 2D)."""
    return 7.78 if case["dim"] == 3 else 3.0


def work(case):
    """Each array a pass's phases need read once and each result written once (FP64 but for the gradient rows' type):
    per cell Q, W with c_s, the gradients, the cell's geometry; per face the face's geometry and its flux."""
    kind = case["kind"]
    if kind == "line":
        return {"bytes": case["steps"] * case["cells"] * (2 * 24 + 8), "flops": case["steps"] * case["cells"] * 400}
    if kind == "network":
        macs = 16 * 64 + 64 * 64 + 64
        return {"bytes": case["rows"] * (2 * 32 + 8 + 4), "flops": case["rows"] * macs * 2 * 4}
    D, V, N = case["dim"], case["dim"] + 2, float(case["n"] ** case["dim"])
    f = _faces(case)
    grad = {"double": 8, "grad32": 4, "grad16": 2}[case.get("precision", "double")] * V * D
    cell = 8 * (2 * D + 2)  # position, centroid, volume, radius
    prim, q = 8 * (V + 1), 8 * V
    face = 8 * 2 * D + 8  # area vector, centroid, the two cells
    sweep = cell + prim + grad + 2 * f * (4 + 8 * (D + 1))
    flux = f * (face + q) + cell + prim + grad
    update = 2 * f * 4 + f * q + 2 * q + prim + 8
    flops = (2 * f * (120 if D == 3 else 70) + f * (300 if D == 3 else 180) + 400) * N
    if kind == "static":
        return {"bytes": case["steps"] * N * (sweep + flux + update), "flops": case["steps"] * flops}
    if kind == "moving":
        geometry = f * face + 2 * f * (4 + 4 + 4 + 8 * (D + 1)) + 2 * cell
        limiter = 2 * 32 * V + 2 * grad if case["limiter"] == "learned" else 0
        net = N * V * (16 * 64 + 64 * 64 + 64) * 2 if case["limiter"] == "learned" else 0
        return {"bytes": N * (sweep + 2 * (flux + update) + 2 * geometry + 8 * 6 * D + limiter), "flops": 1.6 * flops + net}
    if kind == "tangent":
        return {"bytes": N * 2 * (sweep + flux + update), "flops": 3 * flops}
    if kind == "gradient":
        forwards = case["steps"] + sum(1 for k in range(case["steps"]) if k % case["every"] != case["every"] - 1 and k != case["steps"] - 1)
        return {"bytes": N * (forwards + 3 * case["steps"]) * (sweep + flux + update), "flops": (forwards + 4 * case["steps"]) * flops}
    return {"bytes": N * 8 * (sweep + flux), "flops": 8 * flops}


def tolerance(case):
    """About four times what the path was seen to differ by from exact(), whose sums run in another order: forward steps in
    64 bits 7e-17 to 4e-16, derivatives 7e-16 to 3e-15, grad32 3e-9, grad16 2e-6 (their rows' own rounding), a step of the
    learned limiter 4e-7; its network's batch: FP32 sums in another order move a BF16 rounding here and there. max: a cell
    on a limiter's switch may take either side."""
    kind = case["kind"]
    if kind == "network":
        return {"rel": 4e-3, "max": 4e-2}
    if case.get("limiter") == "learned":
        return {"rel": 1.6e-6, "max": 1e-3}
    if case.get("precision") == "grad32":
        return {"rel": 1.2e-8, "max": 1e-5}
    if case.get("precision") == "grad16":
        return {"rel": 8e-6, "max": 8e-3}
    if kind in ("tangent", "gradient", "moving_adjoint"):
        return {"rel": 1.2e-14, "max": 1e-11}
    return {"rel": 1.6e-15, "max": 1e-12}


# ------------------------------------------------------------------------------------------- the scheme in plain torch


class _M:
    """A mesh as padded list tables (cells x longest list) of torch tensors."""

    def __init__(self, m, device):
        t = lambda a, k=torch.float64: torch.tensor(np.asarray(a), dtype=k, device=device)  # noqa: E731
        self.D, self.N = m["dim"], m["cells"]
        self.owner, self.neighbour = t(m["owner"], torch.int64), t(m["neighbour"], torch.int64)
        self.A, self.fc, self.c, self.V, self.x = t(m["area"]), t(m["face_centroid"]), t(m["centroid"]), t(m["volume"]), t(m["positions"])
        self.side = t(m["side"][: self.D])
        self.mag = (self.A * self.A).sum(1).sqrt()
        start, flat = t(m["start"], torch.int64), t(m["list"], torch.int64)
        count = start[1:] - start[:-1]
        k = torch.arange(int(count.max()), device=device)
        self.mask = k[None, :] < count[:, None]
        face = flat[(start[:-1, None] + k[None, :]).clamp(max=len(flat) - 1)]
        face = torch.where(face < 0, -face - 1, face)
        me = torch.arange(self.N, device=device)[:, None]
        self.face, self.owned = face, self.owner[face] == me
        self.other = torch.where(self.mask, torch.where(self.owned, self.neighbour[face], self.owner[face]), me)
        self.d = self.near(self.x[self.other] - self.x[:, None])
        # face centroids relative to the cell's centroid
        self.off = self.fc[face] + torch.where(self.owned[..., None], torch.zeros_like(self.d), self.d) - self.c[:, None]
        self.w = torch.where(self.mask, self.mag[face], torch.zeros_like(self.off[..., 0]))
        self.r = (self.V / math.pi).sqrt() if self.D == 2 else (3 * self.V / (4 * math.pi)) ** (1.0 / 3)

    def near(self, d):
        return d - self.side * torch.round(d / self.side)


def _primitives(q, V):
    U = q / V[:, None]
    v = U[:, 1:-1] / U[:, :1]
    P = (GAMMA - 1) * (U[:, -1] - 0.5 * U[:, 0] * (v * v).sum(1))
    W = torch.cat([U[:, :1], v, P[:, None]], 1)
    return W, (GAMMA * P / U[:, 0]).sqrt()


def _fit(M, W, limit=True):
    """The limited gradients (cells x V x D), the unlimited ones, the intercepts, the limiter's factors, the neighbours' range."""
    D, V, U = M.D, M.D + 2, M.D + 1
    X = [torch.ones_like(M.w)] + [M.d[..., a] + M.c[M.other][..., a] - M.c[:, None, a] for a in range(D)]
    S = [[(M.w * X[p] * X[s]).sum(1) for s in range(U)] for p in range(U)]
    L = [[None] * U for _ in range(U)]
    for p in range(U):
        for s in range(p + 1):
            v = S[s][p]
            for k in range(s):
                v = v - L[p][k] * L[s][k]
            L[p][s] = v.sqrt() if p == s else v / L[s][s]
    tiny = M.w < 1e-6 * M.w.sum(1, keepdim=True)
    use = M.mask & ~tiny
    g, g0, icpt, phi, lo, hi = [], [], [], [], [], []
    for v in range(V):
        Wn = W[:, v][M.other]
        dW = Wn - W[:, None, v]
        z = []
        for p in range(U):
            t = (M.w * X[p] * dW).sum(1)
            for k in range(p):
                t = t - L[p][k] * z[k]
            z.append(t / L[p][p])
        x = [None] * U
        for p in reversed(range(U)):
            t = z[p]
            for k in range(p + 1, U):
                t = t - L[k][p] * x[k]
            x[p] = t / L[p][p]
        grad = torch.stack(x[1:], 1)
        inf = torch.full_like(Wn, math.inf)
        low, high = torch.where(use, Wn, inf).amin(1), torch.where(use, Wn, -inf).amax(1)
        factor = torch.ones_like(low)
        if limit:
            dp = (grad[:, None] * M.off).sum(2)
            one = torch.ones_like(dp)
            up, down = use & (dp > 0) & (W[:, None, v] + dp > high[:, None]), use & (dp < 0) & (W[:, None, v] + dp < low[:, None])
            safe = torch.where(up | down, dp, one)
            room = torch.where(up, (high - W[:, v])[:, None].clamp(min=0), (low - W[:, v])[:, None].clamp(max=0))
            factor = torch.where(up | down, room / safe, one).amin(1)
        g.append(grad * factor[:, None])
        g0.append(grad)
        icpt.append(x[0])
        phi.append(factor)
        lo.append(low)
        hi.append(high)
    st = lambda a: torch.stack(a, 1)  # noqa: E731
    return st(g), st(g0), st(icpt), st(phi), st(lo), st(hi)


def _time_step(M, W, cs, w, courant):
    rel = W[:, 1:-1] if w is None else W[:, 1:-1] - w
    if M.D == 2:
        rate = ((rel.abs() + cs[:, None]) / (M.r * math.sqrt(math.pi))[:, None]).sum(1)
        return float((courant / rate).min())
    own = M.r / (cs + (rel * rel).sum(1).sqrt())
    dist = (M.d * M.d).sum(2).sqrt()
    dv = W[:, 1:-1][M.other] - W[:, None, 1:-1]
    vsig = cs[:, None] + cs[M.other] - (dv * M.d).sum(2) / torch.where(M.mask, dist, torch.ones_like(dist))
    pair = torch.where(M.mask & (vsig > 0), (dist + M.r[:, None]) / vsig, torch.full_like(dist, math.inf))
    return courant * min(float(own.min()), float(pair.min()))


def _point_velocity(M, W, cs):
    dist = torch.where(M.mask, (M.d * M.d).sum(2).sqrt(), torch.ones_like(M.w))
    angle = (M.w / math.pi).sqrt() if M.D == 3 else 0.5 * M.w
    worst = torch.where(M.mask, angle / (0.5 * dist), torch.zeros_like(dist)).amax(1)
    fraction = 0.5 * ((worst - 0.75 * 2.25) / (0.25 * 2.25)).clamp(0, 1)
    cd = (M.c * M.c).sum(1).sqrt()
    scale = torch.where(cd > 0, fraction * cs / torch.where(cd > 0, cd, torch.ones_like(cd)), torch.zeros_like(cd))
    return W[:, 1:-1] + M.c * scale[:, None]


def _half(W, g, dt):
    """W - dt/2 sum_d A_d(W) dW/dx_d of rows W (.. x V) and gradients g (.. x V x D)."""
    D = W.shape[1] - 2
    rho, P = W[:, 0], W[:, -1]
    v = W[:, 1:-1]
    div = sum(g[:, 1 + a, a] for a in range(D))
    along = lambda k: (v * g[:, k]).sum(1)  # noqa: E731
    A = [along(0) + rho * div] + [along(1 + k) + g[:, -1, k] / rho for k in range(D)] + [along(D + 1) + GAMMA * P * div]
    return W - 0.5 * dt * torch.stack(A, 1)


def _face_state(W, g, off, dt=None):
    out = (W if dt is None else _half(W, g, dt)) + (g * off[:, None]).sum(2)
    return torch.where(((out[:, 0] > 0) & (out[:, -1] > 0))[:, None], out, W)


def _flux(L, R, n, w, hll):
    """HLLC (or HLL where `hll`) in the frame of the face moving at w, back in the lab frame, per unit area."""
    def side(W):
        v = W[:, 1:-1] - w
        vn = (v * n).sum(1)
        rho, P = W[:, 0], W[:, -1]
        E = P / (GAMMA - 1) + 0.5 * rho * (v * v).sum(1)
        U = torch.cat([rho[:, None], rho[:, None] * v, E[:, None]], 1)
        F = torch.cat([(rho * vn)[:, None], (rho * vn)[:, None] * v + P[:, None] * n, ((E + P) * vn)[:, None]], 1)
        return rho, v, vn, P, (GAMMA * P / rho).sqrt(), E, U, F
    rl, vl, nl, pl, cl, El, Ul, Fl = side(L)
    rr, vr, nr, pr, cr, Er, Ur, Fr = side(R)
    SL, SR = torch.minimum(nl - cl, nr - cr), torch.maximum(nl + cl, nr + cr)
    dl, dr = rl * (SL - nl), rr * (SR - nr)
    SM = (pr - pl + dl * nl - dr * nr) / (dl - dr)

    def star(rho, v, vn, P, E, U, F, S, d):
        rs = d / (S - SM)
        Es = E / rho + (SM - vn) * (SM + P / d)
        Us = torch.cat([rs[:, None], rs[:, None] * (v + n * (SM - vn)[:, None]), (rs * Es)[:, None]], 1)
        return F + S[:, None] * (Us - U)
    pick = lambda c, a, b: torch.where(c[:, None], a, b)  # noqa: E731
    inside = pick(SM >= 0, star(rl, vl, nl, pl, El, Ul, Fl, SL, dl), star(rr, vr, nr, pr, Er, Ur, Fr, SR, dr))
    mean = (SR[:, None] * Fl - SL[:, None] * Fr + (SL * SR)[:, None] * (Ur - Ul)) / (SR - SL)[:, None]
    F = pick(SL >= 0, Fl, pick(SR <= 0, Fr, pick(hll, mean, inside)))
    energy = F[:, -1] + (w * F[:, 1:-1]).sum(1) + 0.5 * (w * w).sum(1) * F[:, 0]
    return torch.cat([F[:, :1], F[:, 1:-1] + w * F[:, :1], energy[:, None]], 1)


def _apply(M, q, F, dt):
    F = F * M.mag[:, None]
    return q - dt * torch.zeros_like(q).index_add(0, M.owner, F).index_add(0, M.neighbour, -F)


def _sides(M):
    o, j = M.owner, M.neighbour
    sep = M.near(M.x[j] - M.x[o])
    return o, j, sep, M.fc - M.c[o], M.fc - sep - M.c[j]


def _hll_faces(M, W, cs, g, case):
    if case["riemann"] == "hll":
        return torch.ones(len(M.owner), dtype=torch.bool, device=W.device)
    if not case.get("hll"):
        return torch.zeros(len(M.owner), dtype=torch.bool, device=W.device)
    flag = M.r * sum(g[:, 1 + a, a] for a in range(M.D)) / cs < -case["hll"]
    return flag[M.owner] | flag[M.neighbour]


def _static_step(M, q, dt, case, fitted=None):
    W, cs = _primitives(q, M.V)
    g = (fitted or _fit(M, W))[0]
    o, j, _, ro, rj = _sides(M)
    n = M.A / M.mag[:, None]
    F = _flux(_face_state(W[o], g[o], ro, dt), _face_state(W[j], g[j], rj, dt), n, torch.zeros_like(n), _hll_faces(M, W, cs, g, case))
    return _apply(M, q, F, dt)


def _moving_pass(M, q, W, g, what, dt, hll, c0=None):
    """One flux pass of a moving step over dt/2, on the mesh of t^n (c0 None) or of t^n+1 (c0: the centroids of t^n)."""
    o, j, sep, ro, rj = _sides(M)
    n = M.A / M.mag[:, None]
    dist = (sep * sep).sum(1).sqrt()
    cf = M.fc - 0.5 * sep
    speed = (cf * (what[o] - what[j])).sum(1) / dist
    far = (cf * cf).sum(1).sqrt()
    speed = torch.where(far > 0.9 * dist, speed * 0.9 * dist / far, speed)
    w = 0.5 * (what[o] + what[j]) + sep * (speed / dist)[:, None]
    if c0 is None:
        L, R = _face_state(W[o], g[o], ro), _face_state(W[j], g[j], rj)
    else:
        L = _face_state(W[o], g[o], ro + (M.c - c0)[o] + what[o] * dt, 2 * dt)
        R = _face_state(W[j], g[j], rj + (M.c - c0)[j] + what[j] * dt, 2 * dt)
    return _apply(M, q, _flux(L, R, n, w, hll), 0.5 * dt)


def _bf16(x):
    return x.to(torch.bfloat16).to(x.dtype)


def _network(params, x):
    """The limiter's MLP in 64 bits on rows x, with the weights' BF16 values (operands are stored so)."""
    H, K = learned.HIDDEN, learned.FEATURES
    cut = lambda a, b: params[a:b]  # noqa: E731
    W1, b1 = _bf16(cut(learned.P_W1, learned.P_B1)).reshape(H, K), cut(learned.P_B1, learned.P_W2)
    W2, b2 = _bf16(cut(learned.P_W2, learned.P_B2)).reshape(H, H), cut(learned.P_B2, learned.P_W3)
    h = torch.relu(torch.relu(x @ W1.T + b1) @ W2.T + b2)
    return torch.sigmoid(h @ cut(learned.P_W3, learned.P_B3) + params[learned.P_B3])


def _learned_fraction(M, W, cs, fit):
    """The learned limiter's fraction of each cell and variable (1 in troubled cells), from unrounded features."""
    g, g0, icpt, phi, lo, hi = fit
    N, V, D = g.shape
    scale = torch.stack([cs if 0 < v < V - 1 else W[:, v].abs() for v in range(V)], 1)
    S = hi - lo + 1e-12 * scale + 1e-300
    tiny = M.w < 1e-6 * M.w.sum(1, keepdim=True)
    dp = torch.stack([(g0[:, None, v] * M.off).sum(2) for v in range(V)], 2)
    dp = torch.where((M.mask & ~tiny)[..., None], dp, torch.zeros_like(dp))
    clip = lambda a: a.clamp(-8, 8)  # noqa: E731
    div = sum(g0[:, 1 + a, a] for a in range(D)) * M.r / cs
    if D == 2:
        curl = (g0[:, 2, 0] - g0[:, 1, 1]).abs()
    else:
        curl = ((g0[:, 3, 1] - g0[:, 2, 2]) ** 2 + (g0[:, 1, 2] - g0[:, 3, 0]) ** 2 + (g0[:, 2, 0] - g0[:, 1, 1]) ** 2).sqrt()
    mach = (W[:, 1:-1] ** 2).sum(1).sqrt() / cs
    count = M.mask.sum(1).to(W.dtype)
    # the faces whose clip changes the factor, in list order
    clips = torch.zeros_like(phi)
    for v in range(V):
        run = g0[:, v]
        for t in range(M.mask.shape[1]):
            use = (M.mask & ~tiny)[:, t]
            p = (run * M.off[:, t]).sum(1)
            up, down = use & (p > 0) & (W[:, v] + p > hi[:, v]), use & (p < 0) & (W[:, v] + p < lo[:, v])
            room = torch.where(up, (hi[:, v] - W[:, v]).clamp(min=0), (lo[:, v] - W[:, v]).clamp(max=0))
            hit = up | down
            run = run * torch.where(hit, room / torch.where(hit, p, torch.ones_like(p)), torch.ones_like(p))[:, None]
            clips[:, v] += hit
    same = lambda a: a[:, None].expand(N, V)  # noqa: E731
    rho_jump, p_jump = (hi[:, 0] - lo[:, 0]) / W[:, 0], (hi[:, -1] - lo[:, -1]) / W[:, -1]
    kind = lambda k: (torch.arange(V, device=W.device) == k).to(W.dtype)[None].expand(N, V)  # noqa: E731
    f = [phi, clip((hi - W) / S), clip((W - lo) / S), clip(dp.amax(1).clamp(min=0) / S), clip(-dp.amin(1).clamp(max=0) / S), clip(icpt / S),
         clips / count[:, None], same(phi.amin(1)), same(clip(rho_jump)), same(clip(p_jump)), same(clip(div)), same(clip(curl * M.r / cs)),
         same(clip(mach)), kind(0), kind(V - 1), clip(S / (scale + 1e-300))]
    params = torch.tensor(learned.default_params(), dtype=torch.float64, device=W.device)
    out = _network(params, torch.stack(f, 2).reshape(N * V, len(f))).reshape(N, V)
    troubled = ((div < -0.05) & (p_jump > 0.5)) | (lo[:, 0] < 0.1 * W[:, 0]) | (lo[:, -1] < 0.1 * W[:, -1])
    return torch.where(troubled[:, None], torch.ones_like(out), out)


def _exact_line(case, seed):
    """The Sod line in numpy: limited slopes, MUSCL-Hancock, the Riemann flux, LUNA's time step."""
    pb, keys, step, period, q, vol = _line(case, seed)
    gam = pb.gamma
    gaps = np.concatenate([[2 * keys[0]], np.diff(keys), [2 * (period - keys[-1])]]) * step
    c = 0.25 * (gaps[1:] - gaps[:-1])
    gl, gr = gaps[:-1], gaps[1:]
    copy = lambda a: np.concatenate([a[:1], a, a[-1:]])  # noqa: E731  (outflow walls)
    ce = np.concatenate([[-c[0]], c, [-c[-1]]])
    dL, dR = (-gl + ce[:-2] - c)[:, None], (gr + ce[2:] - c)[:, None]
    dts = []

    def prims(q):
        U = q / vol[:, None]
        return np.column_stack([U[:, 0], U[:, 1] / U[:, 0], (gam - 1) * (U[:, 2] - 0.5 * U[:, 1] ** 2 / U[:, 0])])

    def flux(L, R):
        rows = []
        for W in (L, R):
            E = W[:, 2] / (gam - 1) + 0.5 * W[:, 0] * W[:, 1] ** 2
            m = W[:, 0] * W[:, 1]
            rows.append((W[:, 0], W[:, 1], W[:, 2], np.sqrt(gam * W[:, 2] / W[:, 0]), E, np.column_stack([W[:, 0], m, E]),
                         np.column_stack([m, m * W[:, 1] + W[:, 2], (E + W[:, 2]) * W[:, 1]])))
        (rl, vl, pl, cl, El, Ul, Fl), (rr, vr, pr, cr, Er, Ur, Fr) = rows
        SL, SR = np.minimum(vl - cl, vr - cr), np.maximum(vl + cl, vr + cr)
        dl, dr = rl * (SL - vl), rr * (SR - vr)
        if case["riemann"] == "hll":
            mid = (SR[:, None] * Fl - SL[:, None] * Fr + (SL * SR)[:, None] * (Ur - Ul)) / (SR - SL)[:, None]
        else:
            SM = (pr - pl + dl * vl - dr * vr) / (dl - dr)
            mids = []
            for rho, v, P, E, U, F, S, d in ((rl, vl, pl, El, Ul, Fl, SL, dl), (rr, vr, pr, Er, Ur, Fr, SR, dr)):
                rs = d / (S - SM)
                Us = np.column_stack([rs, rs * SM, rs * (E / rho + (SM - v) * (SM + P / d))])
                mids.append(F + S[:, None] * (Us - U))
            mid = np.where((SM >= 0)[:, None], mids[0], mids[1])
        return np.where((SL >= 0)[:, None], Fl, np.where((SR <= 0)[:, None], Fr, mid))

    for _ in range(case["steps"]):
        W = prims(q)
        dt = 0.4 * float((vol / (np.abs(W[:, 1]) + np.sqrt(gam * W[:, 2] / W[:, 0]))).min())
        dts.append(dt)
        We = copy(W)
        left, right = We[:-2], We[2:]
        sL, sR = (left - W) / dL, (right - W) / dR
        with np.errstate(divide="ignore", invalid="ignore"):
            if case["limiter"] == "minmod":
                g = np.where(sL * sR > 0, np.where(np.abs(sL) < np.abs(sR), sL, sR), 0.0)
            elif case["limiter"] == "vanleer":
                g = np.where(sL * sR > 0, 2 * sL * sR / (sL + sR), 0.0)
            else:
                g = ((right - W) - (left - W)) / (dR - dL)
                lo, hi = np.minimum(left, right), np.maximum(left, right)
                for r in ((-0.5 * gl - c)[:, None], (0.5 * gr - c)[:, None]):
                    dp = g * r
                    g = np.where((dp > 0) & (W + dp > hi), g * np.maximum(hi - W, 0) / dp,
                                 np.where((dp < 0) & (W + dp < lo), g * np.minimum(lo - W, 0) / dp, g))
        A = np.column_stack([W[:, 1] * g[:, 0] + W[:, 0] * g[:, 1], W[:, 1] * g[:, 1] + g[:, 2] / W[:, 0],
                             W[:, 1] * g[:, 2] + gam * W[:, 2] * g[:, 1]])
        half = W - 0.5 * dt * A
        faces = []
        for r in ((-0.5 * gl - c)[:, None], (0.5 * gr - c)[:, None]):
            s = half + g * r
            faces.append(np.where(((s[:, 0] > 0) & (s[:, 2] > 0))[:, None], s, W))
        # an outflow wall's ghost face takes the cell's own state
        L = np.concatenate([W[:1], faces[1]])
        R = np.concatenate([faces[0], W[-1:]])
        F = flux(L, R)
        q = q - dt * (F[1:] - F[:-1])
    return {"q": q, "dt": np.array(dts)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "moving_adjoint":
        return None  # the geometry's derivative in the generators is the mesh library's: no plain-torch counterpart
    if kind == "line":
        return _exact_line(case, seed)
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "network":
        bits, t, w = _rows(case, seed)
        x = torch.tensor((bits.astype(np.uint32) << 16).view(np.float32), dtype=torch.float64, device=device)
        t, w = (torch.tensor(a, dtype=torch.float64, device=device) for a in (t, w))
        p = torch.tensor(_params(seed), dtype=torch.float64, device=device).requires_grad_()
        H, K = learned.HIDDEN, learned.FEATURES
        q = p + (torch.cat([_bf16(p[: learned.P_B1]), p[learned.P_B1:learned.P_W2], _bf16(p[learned.P_W2:learned.P_B2]),
                            p[learned.P_B2:]]) - p).detach()  # the BF16 weights' values, the gradient straight through
        h = torch.relu(x @ q[: H * K].reshape(H, K).T + q[learned.P_B1:learned.P_W2])
        h = torch.relu(h @ q[learned.P_W2:learned.P_B2].reshape(H, H).T + q[learned.P_B2:learned.P_W3])
        f = torch.sigmoid(h @ q[learned.P_W3:learned.P_B3] + q[learned.P_B3])
        loss = (w * (f - t) ** 2).sum() / w.sum()
        loss.backward()
        return {"loss": float(loss), "gradient": p.grad, "fraction": f.detach()}
    m = _mesh(case, seed)
    q0 = _state(m, seed, calm=kind in ("tangent", "gradient"))
    M = _M(m, device)
    q = torch.tensor(q0, device=device)
    courant = _courant(case["dim"])
    W, cs = _primitives(q, M.V)
    if kind == "static":
        dts = []
        for _ in range(case["steps"]):
            W, cs = _primitives(q, M.V)
            dts.append(_time_step(M, W, cs, None, courant))
            q = _static_step(M, q, dts[-1], case)
        return {"q": q, "dt": np.array(dts)}
    if kind == "moving":
        w = _point_velocity(M, W, cs)
        dt = _time_step(M, W, cs, w, courant)
        fit = _fit(M, W)
        g = fit[0]
        if case["limiter"] == "learned":
            g = g * _learned_fraction(M, W, cs, fit)[..., None]
        hll = _hll_faces(M, W, cs, g, case)
        step = m["step"]
        k0, k1 = torch.round(M.x / step), torch.round((M.x + dt * w) / step)
        what = (k1 - k0) * (step / dt)
        q = _moving_pass(M, q, W, g, what, dt, hll)
        period = torch.tensor([float(p) for p in m["period"]], dtype=torch.float64, device=device)
        m1 = meshlib.build((torch.remainder(k1, period) * step).cpu().numpy(), 1.0)
        M1 = _M(m1, device)
        if case.get("hll"):
            flag = M.r * sum(g[:, 1 + a, a] for a in range(M.D)) / cs < -case["hll"]
            hll = flag[M1.owner] | flag[M1.neighbour]
        else:
            hll = hll[:1].expand(len(M1.owner))
        q = _moving_pass(M1, q, W, g, what, dt, hll, c0=M.c)
        return {"q": q, "dt": dt, "fallbacks": None}
    dq = torch.tensor(_rows_like(q0, seed), device=device)
    dt = _time_step(M, W, cs, None, courant)
    if kind == "gradient":
        q.requires_grad_()
        out = q
        for _ in range(case["steps"]):
            out = _static_step(M, out, dt, case)
        (out * dq).sum().backward()
        return {"q": out.detach(), "gradient": q.grad}
    # forward mode as two reverses: d/du of u -> (J^T u) . dq
    q.requires_grad_()
    out = _static_step(M, q, dt, case)
    u = torch.zeros_like(out).requires_grad_()
    back, = torch.autograd.grad(out, q, u, create_graph=True)
    forward, = torch.autograd.grad(back, u, dq)
    return {"q": out.detach(), "dq": forward, "dt": dt}
