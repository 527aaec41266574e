"""Performance cases: what users of this framework run, through its public entry points.

A pass of a tissue case is one simulation call as a program makes it: upload a start, advance it, read the
state back (the reference's CLEulerUpdate does the three on every call).  Cases of one step also read the
forces, which a run of many steps leaves out: the force law jumps at its cut-offs (facing faces, 2 l0
adhesion, contact), so the force of a single vertex at the end of a long run says nothing about accuracy,
while the state does.

Kinds:
  tissue3d   3D monolayers of icosphere cells on the substrate (workloads.py's configurations)
  adjoint3d  forward trajectory and its discrete adjoint through torch.autograd (the differentiation form)
  tissue2d   2D polygon tissues, the reference's terms, overdamped Euler
  fire2d     FIRE minimisation of a batch of packings, fixed iterations
  disperse   the dispersal that every drop-in program starts with
"""
from __future__ import annotations

import math

import numpy as np
import torch

from opencl_dpm_amd import autograd, capi

DT3, DT2 = 0.002, 0.005


def listed():
    return [
        # the smallest call: one step of nine cells, as a smoke test or an interactive session makes it
        {"name": "t3_9x162_1step", "kind": "tissue3d", "tissues": 1, "side": 3, "ragged": False, "subdiv": 2,
         "steps": 1, "bits": 32, "terms": "reference"},
        # the drop-in's tissue: one 256-cell monolayer, every term, a plotting interval
        {"name": "t3_256x162", "kind": "tissue3d", "tissues": 1, "side": 16, "ragged": False, "subdiv": 2,
         "steps": 100, "bits": 32, "terms": "all"},
        # the benchmark's batch: 64 tissues of that shape
        {"name": "t3_64x256x162", "kind": "tissue3d", "tissues": 64, "side": 16, "ragged": False, "subdiv": 2,
         "steps": 200, "bits": 32, "terms": "all"},
        # a sweep of coarse tissues of uneven size, the reference's terms
        {"name": "t3_ragged_x42", "kind": "tissue3d", "tissues": 23, "side": 13, "ragged": True, "subdiv": 1,
         "steps": 100, "bits": 32, "terms": "reference"},
        # the precision workload in float: 4096 cells of 642 vertices
        {"name": "t3_4096x642", "kind": "tissue3d", "tissues": 1, "side": 64, "ragged": False, "subdiv": 3,
         "steps": 50, "bits": 32, "terms": "all"},
        # its all-double comparison run, a quarter of the tissue
        {"name": "t3_1024x642_f64", "kind": "tissue3d", "tissues": 1, "side": 32, "ragged": False, "subdiv": 3,
         "steps": 30, "bits": 64, "terms": "all"},
        # the differentiation workload: 64 cells, 200 steps forward and backward
        {"name": "adjoint_64x162", "kind": "adjoint3d", "side": 8, "subdiv": 2, "steps": 200, "every": 20,
         "bits": 32},
        # the reference's CPU-runnable 2D case
        {"name": "t2_16x24", "kind": "tissue2d", "tissues": 1, "cells": 16, "cells_hi": 16, "nv": 24, "nv_hi": 24,
         "ratio": 1.4, "phi": 0.6, "calA": 1.0, "Ka": 1.0, "Kb": 0.0, "Kat": 0.0, "steps": 1000, "bits": 32},
        # the reference's test2D.py tissue: 400 cells of 22 and 25 vertices, with attraction
        {"name": "t2_400_driver", "kind": "tissue2d", "tissues": 1, "cells": 400, "cells_hi": 400, "nv": 22,
         "nv_hi": 25, "ratio": 1.69, "phi": 0.81, "calA": 1.2, "Ka": 0.1, "Kb": 0.05, "Kat": 0.5, "steps": 200,
         "bits": 32},
        # a batch of uneven 2D tissues under the reference's terms
        {"name": "t2_512_batch", "kind": "tissue2d", "tissues": 512, "cells": 8, "cells_hi": 128, "nv": 16,
         "nv_hi": 64, "ratio": 1.4, "phi": 0.6, "calA": 1.02, "Ka": 1.0, "Kb": 0.01, "Kat": 0.1, "steps": 50,
         "bits": 32},
        # the batching form: FIRE in double on packings near jamming
        {"name": "fire_512_f64", "kind": "fire2d", "tissues": 512, "cells": 8, "cells_hi": 128, "nv": 16,
         "nv_hi": 64, "phi": 0.75, "iters": 100, "bits": 64},
        # set-up of a drop-in tissue: the soft-disk relaxation of its centres
        {"name": "disperse_100", "kind": "disperse", "cells": 100, "phi0": 0.9},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tissue3d", "tissue3d", "tissue3d", "adjoint3d", "tissue2d", "tissue2d", "fire2d", "disperse"])
    if kind == "tissue3d":
        subdiv = rng.choice([1, 2, 2, 3])
        bits = rng.choice([32, 32, 32, 64])
        side = _log(rng, 3, 40 if subdiv < 3 else 50)
        nv = 10 * 4 ** subdiv + 2
        tissues = _log(rng, 1, max(1, min(64, 2_000_000 // (side * side * nv))))
        most = {1: 3e8, 2: 4e8, 3: 1e8}[subdiv] / (5 if bits == 64 else 1) / (tissues * side * side * nv)
        return {"kind": kind, "tissues": tissues, "side": side, "ragged": rng.random() < 0.5, "subdiv": subdiv,
                "steps": max(1, min(200, int(most), _log(rng, 1, 200))), "bits": bits,
                "terms": rng.choice(["reference", "all"])}
    if kind == "adjoint3d":
        every = _log(rng, 2, 25)
        return {"kind": kind, "side": rng.randint(3, 9), "subdiv": rng.choice([1, 2]),
                "steps": every * rng.randint(1, max(1, 200 // every)), "every": every, "bits": rng.choice([32, 64])}
    if kind == "disperse":
        return {"kind": kind, "cells": _log(rng, 16, 100), "phi0": rng.choice([0.7, 0.8, 0.9])}
    if kind == "fire2d":
        lo = rng.randint(8, 40)
        return {"kind": kind, "tissues": _log(rng, 1, 512), "cells": lo, "cells_hi": rng.randint(lo, 128), "nv": 16,
                "nv_hi": rng.randint(16, 64), "phi": rng.choice([0.5, 0.65, 0.75]), "iters": _log(rng, 10, 100),
                "bits": rng.choice([32, 64])}
    one = rng.random() < 0.5
    lo = _log(rng, 6, 700) if one else rng.randint(8, 60)
    nlo = rng.randint(12, 30)
    return {"kind": kind, "tissues": 1 if one else _log(rng, 2, 512), "cells": lo,
            "cells_hi": lo if one else rng.randint(lo, 128), "nv": nlo, "nv_hi": rng.randint(nlo, 30 if one else 64),
            "ratio": rng.choice([1.4, 1.69]), "phi": rng.choice([0.6, 0.81]), "calA": rng.choice([1.0, 1.02, 1.2]),
            "Ka": rng.choice([0.1, 1.0]), "Kb": rng.choice([0.0, 0.05]), "Kat": rng.choice([0.0, 0.5]),
            "steps": _log(rng, 20, 200) if one and lo > 100 else _log(rng, 10, 50), "bits": 32}


# ------------------------------------------------------------------ inputs

_SPHERE = {}


def _icosphere(subdiv):
    if subdiv not in _SPHERE:
        t = (1 + 5 ** 0.5) / 2
        V = [np.array(p, float) / math.hypot(1, t) for p in
             ((-1, t, 0), (1, t, 0), (-1, -t, 0), (1, -t, 0), (0, -1, t), (0, 1, t), (0, -1, -t), (0, 1, -t),
              (t, 0, -1), (t, 0, 1), (-t, 0, -1), (-t, 0, 1))]
        F = [(0, 11, 5), (0, 5, 1), (0, 1, 7), (0, 7, 10), (0, 10, 11), (1, 5, 9), (5, 11, 4), (11, 10, 2), (10, 7, 6),
             (7, 1, 8), (3, 9, 4), (3, 4, 2), (3, 2, 6), (3, 6, 8), (3, 8, 9), (4, 9, 5), (2, 4, 11), (6, 2, 10),
             (8, 6, 7), (9, 8, 1)]
        for _ in range(subdiv):
            mid, G = {}, []

            def m(a, b):
                k = (min(a, b), max(a, b))
                if k not in mid:
                    p = V[a] + V[b]
                    V.append(p / np.linalg.norm(p))
                    mid[k] = len(V) - 1
                return mid[k]

            for a, b, c in F:
                x, y, z = m(a, b), m(b, c), m(c, a)
                G += [(a, x, z), (b, y, x), (c, z, y), (x, y, z)]
            F = G
        _SPHERE[subdiv] = np.array(V, np.float32), np.array(F, np.int32)
    return _SPHERE[subdiv]


def _sides(case):
    if not case.get("ragged"):
        return [case["side"]] * case.get("tissues", 1)
    return [3 + (7 * k + 5) % max(1, case["side"] - 2) for k in range(case["tissues"])]


def _in3(case, seed):
    """Monolayers on the substrate: radius U(0.9, 1.1), spacing 2.4, jitter 0.1."""
    rng = np.random.Generator(np.random.PCG64(seed))
    V, F = _icosphere(case["subdiv"])
    sides = _sides(case)
    C = sum(s * s for s in sides)
    r = rng.uniform(0.9, 1.1, C).astype(np.float32)
    g = np.concatenate([np.stack(np.meshgrid(np.arange(s), np.arange(s)), -1).reshape(-1, 2) for s in sides])
    c = np.empty((C, 3), np.float32)
    c[:, :2] = (g + 0.5) * 2.4 + rng.uniform(-0.1, 0.1, (C, 2))
    c[:, 2] = r
    X = (V[None] * r[:, None, None] + c[:, None, :]).reshape(-1, 3)
    v0 = (4 / 3 * np.pi * r.astype(np.float64) ** 3).astype(np.float32)
    a0 = ((6 * np.sqrt(np.pi) * v0.astype(np.float64)) ** (2 / 3) / len(F)).astype(np.float32)
    cb = np.concatenate([[0], np.cumsum([s * s for s in sides])]).astype(np.int32)
    return dict(V=V, F=F, X=X, v0=v0, a0=a0, cb=cb, L=[np.float32(2.4 * s) for s in sides])


def _mask3(case):
    if case["kind"] == "adjoint3d":  # the adjoint covers every term but vertex adhesion
        return capi.DPM3D_ALL & ~capi.DPM3D_ADHESION
    return capi.DPM3D_ALL if case["terms"] == "all" else capi.DPM3D_REFERENCE


_K3 = dict(Kv=1.0, Ka=0.5, Ks=0.2, Kb=0.01, Kre=1.0, Kat=0.1)


def _ncells2(case):
    n = case["cells_hi"] - case["cells"] + 1
    return [case["cells"] + (41 * k) % n for k in range(case["tissues"])]


def _in2(case, seed):
    """Bidisperse regular polygons on a jittered grid, small and large in turn."""
    rng = np.random.Generator(np.random.PCG64(seed))
    ratio, calA = case.get("ratio", 1.4), case.get("calA", 1.02)
    X, nvs, a0s, l0s, rs, Ls = [], [], [], [], [], []
    for n in _ncells2(case):
        cols = int(math.ceil(math.sqrt(n)))
        rows = -(-n // cols)
        i, j = np.arange(n) % cols, np.arange(n) // cols
        big = (i + j) % 2 == 1
        r = np.where(big, math.sqrt(ratio), 1.0)
        nv = np.where(big, case["nv"], case["nv_hi"]) if n == case["cells_hi"] == case["cells"] \
            else case["nv"] + (np.arange(n) * 13 + n) % (case["nv_hi"] - case["nv"] + 1)
        a0 = 0.5 * nv * r ** 2 * np.sin(2 * np.pi / nv)
        l0 = 2 * np.sqrt(np.pi * calA * (nv * np.tan(np.pi / nv) / np.pi) * a0) / nv
        L = math.sqrt(a0.sum() / case["phi"])
        c = np.stack([(i + 0.5) * L / cols, (j + 0.5) * L / rows], 1) + rng.uniform(-0.08, 0.08, (n, 2))
        turn = rng.uniform(0, 2 * np.pi, n)
        own = np.repeat(np.arange(n), nv)
        k = np.arange(len(own)) - np.repeat(np.cumsum(nv) - nv, nv)
        th = turn[own] + 2 * np.pi * (k + 1) / nv[own]
        X.append(c[own] + r[own, None] * np.stack([np.cos(th), np.sin(th)], 1))
        nvs.append(nv), a0s.append(a0), l0s.append(l0), rs.append(r), Ls.append(np.float32(L))
    f = lambda v: np.concatenate(v).astype(np.float32)
    return dict(X=f(X), nv=np.concatenate(nvs).astype(np.int32), a0=f(a0s), l0=f(l0s), r0=f(rs), L=Ls,
                cb=np.concatenate([[0], np.cumsum([len(v) for v in nvs])]).astype(np.int32))


def _in_disperse(case, seed):
    """test2D.py's radii, centres at random in the tissue's box."""
    rng = np.random.Generator(np.random.PCG64(seed))
    r = np.where(np.arange(case["cells"]) % 2 == 0, 1.0, 1.3).astype(np.float32)
    L = float(np.float32(math.sqrt(float((np.pi * r.astype(np.float64) ** 2).sum())) / case["phi0"]))
    X, Y = (rng.uniform(0, L, (2, len(r)))).astype(np.float32)
    return r, L, X, Y


# -------------------------------------------------------------- the passes

def prepare(case, seed):
    kind = case["kind"]
    if kind == "disperse":
        return dict(case=case, args=_in_disperse(case, seed))
    if kind in ("tissue3d", "adjoint3d"):
        m = _in3(case, seed)
        t = capi.Tissues3D(m["F"], m["cb"], _K3["Kv"], _K3["Ka"], _K3["Ks"], m["v0"], m["a0"], m["L"], _K3["Kre"],
                           Kat=_K3["Kat"], Kb=_K3["Kb"], ks_grad=9.0 if kind == "adjoint3d" else None,
                           mask=_mask3(case), nv=len(m["V"]), precision=case["bits"])
        if kind == "adjoint3d":
            full = lambda v: torch.full((t.C,), v, dtype=torch.float64, requires_grad=True)
            X0 = torch.tensor(m["X"], dtype=torch.float64, requires_grad=True)
            return dict(case=case, t=t, C=t.C, theta=[full(_K3[k]) for k in ("Kv", "Ka", "Kb", "Ks")], X0=X0)
    else:
        m = _in2(case, seed)
        fire = kind == "fire2d"
        Kb = np.where(np.arange(len(m["nv"])) % 2, 0.01, 0.0) if fire else case["Kb"]
        t = capi.Tissues2D(m["cb"], m["nv"], 1.0 if fire else case["Ka"], 1.0, Kb, m["a0"], m["l0"], m["r0"], m["L"],
                           Kre=1.0, Kat=0.0 if fire else case["Kat"],
                           mask=capi.DPM2D_CONSERVATIVE if fire else capi.DPM2D_ALL, precision=case["bits"])
    return dict(case=case, t=t, X=m["X"].astype(np.float64) if case["bits"] == 64 else m["X"])


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "disperse":
        X, Y, (iters, capped) = capi.disperse(*state["args"])
        return {"X": X, "Y": Y, "iterations": int(iters)}
    t = state["t"]
    if kind == "adjoint3d":
        X0 = state["X0"]
        for p in state["theta"] + [X0]:
            p.grad = None
        XN = autograd.trajectory(t, *state["theta"], X0, case["steps"], DT3, case["every"])
        loss = autograd.com_displacement_loss(XN, X0.detach(), state["C"])
        loss.backward()
        return {"XN": XN.detach(), "loss": loss.detach(), "theta": torch.stack([p.grad for p in state["theta"]]),
                "X0": X0.grad}
    t.set_positions(state["X"])
    if kind == "fire2d":
        st = t.fire(max_iter=case["iters"], ftol=0.0)
        return {"X": t.positions(), "energy": st["energy"]}
    t.euler(case["steps"], DT3 if kind == "tissue3d" else DT2)
    out = {"X": t.positions()}
    if kind == "tissue3d":
        if case["steps"] == 1:
            out["F"] = t.forces()
        out["volume"] = t.cell_stats()[0]
    return out


def work(case):
    """Positions read once and written once; a vertex-step's arithmetic counted at about 500 operations in 3D
    (ring of six springs, volume, bending, substrate, adhesion pairs) and 200 in 2D (neighbours, near vertices)."""
    kind = case["kind"]
    if kind == "disperse":
        return {"bytes": 20.0 * case["cells"], "flops": case["cells"] * 6 * 40 * 1000.0}
    size = case["bits"] / 8
    if kind in ("tissue3d", "adjoint3d"):
        n = sum(s * s for s in _sides(case)) * (10 * 4 ** case["subdiv"] + 2)
        back = 4 if kind == "adjoint3d" else 1
        return {"bytes": 6 * size * n * back, "flops": 500.0 * n * case["steps"] * back}
    n = sum(_ncells2(case)) * (case["nv"] + case["nv_hi"]) / 2
    return {"bytes": 4 * size * n, "flops": 200.0 * n * case.get("steps", case.get("iters"))}


# ------------------------------------------------- the same in 64 bits (torch)

def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a, dtype=torch.float64):
    return torch.as_tensor(np.asarray(a), dtype=dtype, device=_dev())


def _unit(v):
    n = v.square().sum(-1, keepdim=True)
    return v / torch.where(n > 0, n, torch.ones_like(n)).sqrt()


class _Exact3:
    """One 3D tissue in double: X [C, nv, 3]."""

    def __init__(self, V, F, v0, a0, L, mask, ksg):
        self.nv, self.F, self.L, self.mask, self.ksg = len(V), _t(F, torch.long), float(L), mask, ksg
        self.v0, self.a0 = _t(v0), _t(a0)
        self.l0 = (4 * self.a0).sqrt() / math.sqrt(3.0)
        E = np.unique(np.sort(np.concatenate([F[:, [0, 1]], F[:, [1, 2]], F[:, [2, 0]]]), 1), axis=0)
        lap = np.zeros((self.nv, self.nv))
        lap[E[:, 0], E[:, 1]] = lap[E[:, 1], E[:, 0]] = 1
        lap -= np.diag(lap.sum(1))
        self.lap = _t(lap)

    def forces(self, X, Kv, Ka, Kb, Ks, Kre=_K3["Kre"], Kat=_K3["Kat"]):
        C, F, l0 = len(X), self.F, self.l0[:, None]
        com = X.mean(1)
        P = [X[:, F[:, k]] for k in range(3)]
        out = torch.zeros_like(X)
        rel = [p - com[:, None] for p in P]
        vol = (torch.linalg.cross(rel[0], rel[1]) * rel[2]).sum((1, 2)).abs() / 6
        kv = (-Kv * (vol / self.v0 - 1) / 6)[:, None, None]
        sc = (Ka * self.a0.sqrt() / self.l0 * 0.3)[:, None, None]
        e = [P[1] - P[0], P[2] - P[1], P[0] - P[2]]
        ln = [x.square().sum(-1, keepdim=True).sqrt() for x in e]
        s = [x / n * (n / l0[:, :, None] - 1) for x, n in zip(e, ln)]
        down = _unit(torch.linalg.cross(e[0], -e[2]).detach())[..., 2] < float(np.float32(-0.1))
        for k in range(3):
            f = kv * torch.linalg.cross(rel[(k + 1) % 3], rel[(k + 2) % 3]) + sc * (s[k] - s[(k + 2) % 3])
            p = P[k]
            ks = Ks[:, None] * (1 + self.ksg * (p[..., 0] - self.L * (p[..., 0] / self.L).floor().detach()) / self.L)
            z, h = p[..., 2], p[..., 2].abs()
            w = _unit(torch.stack([p[..., 0] - com[:, None, 0], p[..., 1] - com[:, None, 1],
                                   -com[:, None, 2].expand_as(z)], -1))
            push = torch.where(h < 2 * l0, ks * (1 - h / l0), torch.zeros_like(h))[..., None] * w
            push = push + torch.stack([torch.zeros_like(z)] * 2 + [torch.where(z < 0, ks * h, torch.zeros_like(h))], -1)
            out = out.index_add(1, F[:, k], f + torch.where(down[..., None], push, torch.zeros_like(push)))
        if self.mask & 32:
            out = out - Kb[:, None, None] * (self.lap @ (self.lap @ X))
        Xd, cd = X.detach(), com.detach()
        r = (Xd - cd[:, None]).square().sum(-1).amax(1).sqrt()
        D = cd[:, None] - cd[None]
        shift = self.L * (D / self.L).round()
        dist = (D - shift).square().sum(-1).sqrt()
        touch = dist < r[:, None] + r[None] + 2.5 * self.l0.max() * 1.01
        touch.fill_diagonal_(False)
        pi, pj = touch.nonzero(as_tuple=True)
        if (self.mask & 8) and len(pi):
            near = (Xd[pi] - cd[pj, None] - shift[pi, pj, None]).square().sum(-1).sqrt() < r[pj, None] + 0.6 * self.l0.max()
            q, v = near.nonzero(as_tuple=True)
            parts = [torch.zeros_like(X).reshape(-1, 3)]
            for at in torch.arange(len(q), device=q.device).split(20000):
                a, b, w = pi[q[at]], pj[q[at]], v[at]
                p = X[a, w]
                u = [_unit(X[b][:, F[:, k]] + shift[a, b][:, None] - p[:, None]) for k in range(3)]
                den = 1 + (u[0] * u[1]).sum(-1) + (u[1] * u[2]).sum(-1) + (u[2] * u[0]).sum(-1)
                num = (u[0] * torch.linalg.cross(u[1], u[2])).sum(-1)
                ok = den >= 1e-8
                om = torch.where(ok, 2 * torch.atan2(num, torch.where(ok, den, torch.ones_like(den))),
                                 torch.zeros_like(num)).sum(-1) / (4 * math.pi)
                g = torch.where(om.abs() < 1e-6, torch.zeros_like(om), om.abs()) * 0.5 * Kre
                parts.append(torch.zeros_like(parts[0]).index_add(0, a * self.nv + w, g[:, None] * _unit(com[a] - p)))
            out = out + sum(parts).reshape(X.shape)
        if self.mask & 16:
            flat = out.reshape(-1, 3).clone()
            for at in torch.arange(len(pi), device=pi.device).split(max(1, 12_000_000 // self.nv ** 2)):
                a, b = pi[at], pj[at]
                d = X[b][:, None] - X[a][:, :, None]
                d = d - self.L * (d / self.L).round()
                n = d.square().sum(-1).sqrt()
                la = self.l0[a][:, None, None]
                k = torch.where((n < 2 * la) & (n > 1e-12), Kat * 0.5 * (1 / la - 1 / n.clamp(min=1e-12)), torch.zeros_like(n))
                f = k[..., None] * d
                own = torch.arange(self.nv, device=X.device)
                flat.index_add_(0, (a[:, None] * self.nv + own).reshape(-1), -f.sum(2).reshape(-1, 3))
                flat.index_add_(0, (b[:, None] * self.nv + own).reshape(-1), f.sum(1).reshape(-1, 3))
            out = flat.reshape(X.shape)
        return out, vol


def _exact3(case, seed):
    m = _in3(case, seed)
    nv, sides = len(m["V"]), _sides(case)
    if case["steps"] * len(m["v0"]) * 4 * nv * nv > 1.2e10 or case["steps"] * len(sides) > 800:
        return None
    Xs, Fs, vols = [], [], []
    for k in range(len(sides)):
        a, b = m["cb"][k], m["cb"][k + 1]
        T = _Exact3(m["V"], m["F"], m["v0"][a:b], m["a0"][a:b], m["L"][k], _mask3(case), 0.0)
        X = _t(m["X"]).reshape(-1, nv, 3)[a:b]
        K = [_t(np.full(b - a, np.float32(_K3[q]))) for q in ("Kv", "Ka", "Kb", "Ks")]
        for _ in range(case["steps"]):
            f, _v = T.forces(X, *K, Kat=float(np.float32(_K3["Kat"])))
            X = X + float(np.float32(DT3)) * f
        r = X - X.mean(1, keepdim=True)
        P = [r[:, T.F[:, q]] for q in range(3)]
        vols.append((torch.linalg.cross(P[0], P[1]) * P[2]).sum((1, 2)).abs() / 6)
        Xs.append(X.reshape(-1, 3)), Fs.append(f.reshape(-1, 3))
    out = {"X": torch.cat(Xs).cpu().numpy(), "volume": torch.cat(vols).cpu().numpy()}
    if case["steps"] == 1:
        out["F"] = torch.cat(Fs).cpu().numpy()
    return out


def _exact_adjoint(case, seed):
    m = _in3(case, seed)
    T = _Exact3(m["V"], m["F"], m["v0"], m["a0"], m["L"][0], _mask3(case), 9.0)
    th = [_t(np.full(len(m["v0"]), np.float32(_K3[q]))).requires_grad_() for q in ("Kv", "Ka", "Kb", "Ks")]
    X0 = _t(m["X"]).requires_grad_()
    X = X0.reshape(len(m["v0"]), -1, 3)
    for _ in range(case["steps"]):
        X = X + float(np.float32(DT3)) * T.forces(X, *th)[0]
    loss = torch.linalg.norm(X.mean(1) - X0.detach().reshape(X.shape).mean(1), dim=1).mean()
    loss.backward()
    return {"XN": X.detach().reshape(-1, 3).cpu(), "loss": loss.detach().cpu(),
            "theta": torch.stack([p.grad for p in th]).cpu(), "X0": X0.grad.cpu()}


class _Exact2:
    """One 2D tissue in double: X [V, 2]."""

    def __init__(self, nv, a0, l0, r0, L, Ka, Kb, Kat, fire):
        nv = np.asarray(nv)
        b = np.concatenate([[0], np.cumsum(nv)])
        own = np.repeat(np.arange(len(nv)), nv)
        k = np.arange(len(own)) - b[own]
        step = lambda s: _t(b[own] + (k + s) % nv[own], torch.long)
        self.n = {s: step(s) for s in (-2, -1, 1, 2)}
        self.own, self.C, self.L, self.fire, self.Kat = _t(own, torch.long), len(nv), float(L), fire, Kat
        self.nv, self.a0, self.l0, self.r0 = _t(nv), _t(a0), _t(l0), _t(r0)
        self.Ka, self.Kb = _t(Ka), _t(Kb)
        self.other = self.own[:, None] != self.own[None]
        self.ind = torch.zeros(len(own), len(nv), device=_dev())
        self.ind[torch.arange(len(own)), self.own] = 1

    def sum_cell(self, v):
        return torch.zeros((self.C,) + v.shape[1:], dtype=v.dtype, device=v.device).index_add_(0, self.own, v)

    def forces(self, X):
        o, L = self.own, self.L
        xm, xp, xm2, xp2 = (X[self.n[s]] for s in (-1, 1, -2, 2))
        a2 = self.sum_cell((xm[:, 0] + X[:, 0]) * (xm[:, 1] - X[:, 1]))
        strain = (0.5 * a2.abs() / self.a0 - 1)[o]
        c = (self.Ka / self.a0.sqrt())[o] * 0.5 * strain
        dy, dx = xm[:, 1] - xp[:, 1], xm[:, 0] - xp[:, 0]
        if self.fire:
            sg = torch.where(a2 < 0, -1.0, 1.0)[o]
            F = torch.stack([-c * sg * dy, c * sg * dx], 1)
        else:
            F = torch.stack([c * dy, c * dx], 1)
        e, em = xp - X, X - xm
        n, nm = e.norm(dim=1, keepdim=True), em.norm(dim=1, keepdim=True)
        l0 = self.l0[o][:, None]
        F = F + (self.a0 / self.l0).sqrt()[o][:, None] * ((n / l0 - 1) * e / n - (nm / l0 - 1) * em / nm)
        F = F + self.Kb[o][:, None] * (2 * (e - em) - (em - (xm - xm2)) - ((xp2 - xp) - e))
        U = 0.5 * (self.Ka * self.a0.sqrt() * (0.5 * a2.abs() / self.a0 - 1) ** 2).sum()
        U = U + 0.5 * ((self.a0 * self.l0).sqrt()[o] * (n[:, 0] / l0[:, 0] - 1) ** 2).sum()
        U = U + 0.5 * (self.Kb[o] * (e - em).square().sum(1)).sum()
        if self.fire or self.Kat:
            d = X[None] - X[:, None]
            d = d - L * (d / L).round()
            n = d.square().sum(-1).sqrt()
            if self.fire:
                sig = 0.5 * (l0 + l0.T)
                hit = self.other & (n < sig) & (n > 0)
                ov = 1 - n / sig
                k = torch.where(hit, -ov / (sig * n.clamp(min=1e-30)), torch.zeros_like(n))
                U = U + 0.25 * torch.where(hit, ov * ov, torch.zeros_like(n)).sum()
            else:
                k = torch.where(self.other & (n < l0), self.Kat / self.nv[o][:, None] / l0, torch.zeros_like(n))
            F = F + (k[..., None] * d).sum(1)
        if not self.fire:
            di = X[:, None] - X[None]
            dj = X[:, None] - X[self.n[-1]][None]
            big = (di.abs() > L) | (dj.abs() > L)
            rnd = lambda q: torch.stack([(q[..., 0] / L).floor(), (q[..., 1] / L).round()], -1)
            di, dj = (torch.where(big, q - L * rnd(q), q) for q in (di, dj))
            st = (di[..., 1] > 0) != (dj[..., 1] > 0)
            den = torch.where(st, dj[..., 1] - di[..., 1], torch.ones_like(di[..., 1]))
            cr = st & (0 < (dj[..., 0] - di[..., 0]) * -di[..., 1] / den + di[..., 0]) & self.other
            over = ((cr.float() @ self.ind).long() % 2).any(1)
            d = (self.sum_cell(X) / self.nv[:, None])[o] - X
            d = d - L * (d / L).round()
            n = d.norm(dim=1, keepdim=True)
            F = F + torch.where(over[:, None], 0.5 * (1 - n / (2 * self.r0[o][:, None])) * d / n.clamp(min=1e-30),
                                torch.zeros_like(F))
        return F, U


def _exact2(case, seed):
    m = _in2(case, seed)
    fire = case["kind"] == "fire2d"
    steps = case["iters"] if fire else case["steps"]
    ends = np.concatenate([[0], np.cumsum(m["nv"])])
    V = [ends[m["cb"][k + 1]] - ends[m["cb"][k]] for k in range(case["tissues"])]
    if steps * case["tissues"] > 3000 or steps * sum(float(v) ** 2 for v in V) > 4e10:
        return None
    f32 = lambda v: float(np.float32(v))
    Xs, Us = [], []
    for k in range(case["tissues"]):
        a, b = m["cb"][k], m["cb"][k + 1]
        Kb = np.where(np.arange(a, b) % 2, np.float32(0.01), 0.0) if fire else np.full(b - a, f32(case["Kb"]))
        T = _Exact2(m["nv"][a:b], m["a0"][a:b], m["l0"][a:b], m["r0"][a:b], m["L"][k],
                    np.full(b - a, 1.0 if fire else f32(case["Ka"])), Kb, 0.0 if fire else f32(case["Kat"]), fire)
        X = _t(m["X"][ends[a]:ends[b]])
        if not fire:
            for _ in range(steps):
                X = X + f32(DT2) * T.forces(X)[0]
        else:  # Bitzek et al. 2006, the library's defaults
            v, dt, al, pos = torch.zeros_like(X), 0.01, 0.1, 0
            for _ in range(steps):
                F, _u = T.forces(X)
                P = float((F * v).sum())
                if P > 0:
                    v = (1 - al) * v + al * float(v.norm() / F.norm()) * F
                    if pos > 5:
                        dt, al = min(dt * 1.1, 0.1), al * 0.99
                    pos += 1
                elif P < 0:
                    v, dt, al, pos = torch.zeros_like(v), dt * 0.5, 0.1, 0
                v = v + dt * F
                X = X + dt * v
            Us.append(float(T.forces(X)[1]))
        Xs.append(X)
    out = {"X": torch.cat(Xs).cpu().numpy()}
    if fire:
        out["energy"] = np.array(Us)
    return out


def exact(case, seed):
    """None for dispersal (its float sums decide where it stops) and where the pairs take too long."""
    if case["kind"] == "disperse":
        return None
    if case["kind"] == "adjoint3d":
        return _exact_adjoint(case, seed)
    return _exact3(case, seed) if case["kind"] == "tissue3d" else _exact2(case, seed)
