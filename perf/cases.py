"""The workloads whose speed is followed: the material-point update on device
planes, load increments of one volume element, whole jobs, and served jobs.

Every case goes through the entry points that a program of a user calls
(include/solver_cpp_amd.h through its ctypes description, ``Rve`` and
``Server``).  Microstructures are periodic Voronoi grains in the 1e-5 m cube of
the grid examples with uniform orientations; the load is the example's uniaxial
tension (1e-3/s, 0.5 s an increment).

Kinds
  mp     sc_mp_update_noalloc: the update (and the consistent tangent, where it
         is asked for) of n points whose planes the caller owns, for hosts that
         bring their own solver.  The points are in plastic flow: random
         orientations, hardened slip resistances, a stress whose resolved
         shears lie at the slip resistances, and a step that goes on with the
         flow to within a few tenths.
  inc    one load increment of a context that a program keeps: forward,
         solution, coordinates, and F, P, the average stress and the average
         stiffness read back.  The increment is solved again from its converged
         start (the step that a cut-back takes), so each pass has the same work.
  job    a short load case from nothing: context, init, increments, fields.
  serve  independent jobs of uneven grids sent to the batched job server at
         once, their average stresses and stress fields read back.
"""
from __future__ import annotations

import ctypes as C
import math
import os

import numpy as np
import torch

from solver_cpp_amd.capi import SC_FIELD, Library, MpDevicePlanes, ptr
from solver_cpp_amd.geometry import EXAMPLE_NUMERICS
from solver_cpp_amd.rve import Rve, RveSpec, tension_x
from solver_cpp_amd.serving import Server, rotation_to

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBRARY = os.path.join(ROOT, "solver_cpp_amd", "_build", "libsolver_cpp_amd.so")
PRECISION = {"fp64": 0, "mixed": 1}
RATE, DT = 1.0e-3, 0.5  # examples/grid/tensionX.yaml: 1/s, s
WARM = 6                # increments that a kept context has behind it: elastic, the knee, settled plastic flow
EVALUATIONS = 10        # residual evaluations of a plastic increment (4 to 14 by grid and increment)

_lib = None


def library() -> Library:
    global _lib
    if _lib is None:
        _lib = Library(LIBRARY, boundary=True)
    return _lib


def listed():
    return [
        # a handful of points from a host that steps single integration points: launch and latency
        dict(name="mp_60", kind="mp", n=60, tangent=False, n_sl=20.0, a_sl=2.25),
        # a finite-element host's element block, ragged, with the tangent its assembly needs
        dict(name="mp_4097_tangent", kind="mp", n=4097, tangent=True, n_sl=20.0, a_sl=2.25),
        # another material: its exponents (quarters, then any) are not the compiled-in ones
        dict(name="mp_9261_n10_tangent", kind="mp", n=9261, tangent=True, n_sl=10.0, a_sl=2.0),
        # the largest call that the entry point takes
        dict(name="mp_32768", kind="mp", n=32768, tangent=False, n_sl=20.0, a_sl=2.25),
        # the small configuration (16^3 / 20 grains): bound by launches and round trips
        dict(name="inc_16", kind="inc", nx=16, ny=16, nz=16, grains=20, precision="fp64"),
        # an uneven grid, lengths that are not powers of two among them, in the mixed form
        dict(name="inc_27x40x22_mixed", kind="inc", nx=27, ny=40, nz=22, grains=60, precision="mixed"),
        # the drop-in configuration (64^3 / 200 grains)
        dict(name="inc_64", kind="inc", nx=64, ny=64, nz=64, grains=200, precision="fp64"),
        # a large grid of the serving stream's edges (2^a 3^b) without a power of two
        dict(name="inc_108x96x72", kind="inc", nx=108, ny=96, nz=72, grains=350, precision="fp64"),
        # the headline configuration (128^3 / 1000 grains), both arithmetic forms
        dict(name="inc_128_mixed", kind="inc", nx=128, ny=128, nz=128, grains=1000, precision="mixed"),
        dict(name="inc_128", kind="inc", nx=128, ny=128, nz=128, grains=1000, precision="fp64"),
        # a whole small job, set-up included
        dict(name="job_32", kind="job", nx=32, ny=32, nz=32, grains=40, precision="fp64", increments=3),
        # the batched workload: edges from {16, 24, 32, 48}, random tension directions
        dict(name="serve_24", kind="serve", jobs=24, increments=2, precision="fp64"),
    ]


def _smooth(e: float) -> int:
    """The nearest grid length whose prime factors are at most 13."""
    def ok(m):
        for f in (2, 3, 5, 7, 11, 13):
            while m % f == 0:
                m //= f
        return m == 1
    return min((m for m in range(4, 129) if ok(m)), key=lambda m: (abs(m - e), m))


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(("mp", "mp", "inc", "inc", "inc", "job", "serve"))
    precision = rng.choice(("fp64", "mixed"))
    if kind == "mp":
        n_sl, a_sl = rng.choice(((20.0, 2.25), (20.0, 2.25), (10.0, 2.0), (17.3, 1.7)))
        return dict(kind="mp", n=int(_log_uniform(rng, 32, 32768)), tangent=rng.random() < 0.5, n_sl=n_sl, a_sl=a_sl)
    if kind == "serve":
        return dict(kind="serve", jobs=rng.randint(4, 24), increments=rng.randint(1, 2), precision=precision)
    top = 128 if kind == "inc" else 48
    edge = [_smooth(_log_uniform(rng, 8, top)) for _ in range(3)]
    if rng.random() < 0.5:
        edge = edge[:1] * 3
    n = edge[0] * edge[1] * edge[2]
    c = dict(kind=kind, nx=edge[0], ny=edge[1], nz=edge[2], grains=rng.randint(2, max(3, min(1000, n // 200))),
             precision=precision)
    if kind == "job":
        c["increments"] = rng.randint(1, 4)
    return c


def _edges(case):
    """Edge, grains and seed offset of each job of a serve case (part of the case: the same for every seed)."""
    r = np.random.default_rng(1000 + case["jobs"])
    return [(int(r.choice((16, 24, 32, 48))), int(r.integers(10, 201)), j) for j in range(case["jobs"])]


def work(case):
    """Bytes: every residual evaluation reads and writes the material-point state once (139 values a cell) and its
    spectral part reads 9 and writes 9 values a cell; the fields that are read back once more.  Flops: about 5 Newton
    iterations of 1500 and 1.5 state iterations of 1000 operations a point and evaluation, 20000 for a tangent."""
    if case["kind"] == "mp":
        n = case["n"]
        values = 78 + 69 + (81 if case["tangent"] else 0)
        return {"bytes": n * (8 * values + 4), "flops": n * (9500 + (20000 if case["tangent"] else 0))}
    if case["kind"] == "serve":
        cells, incs = sum(e ** 3 for e, _, _ in _edges(case)), case["increments"]
    else:
        cells, incs = case["nx"] * case["ny"] * case["nz"], case.get("increments", 1)
    spectral = 18 * (8 if case["precision"] == "fp64" else 4)
    each = incs * (EVALUATIONS * (8 * 139 + spectral) + 8 * 60) + 2 * 8 * 18
    return {"bytes": cells * each, "flops": cells * incs * (EVALUATIONS * 9500 + 20000)}


# ---- inputs --------------------------------------------------------------------
def _grains(cells, grains, seed):
    """(material_at, orientations): periodic Voronoi grains of the unit cube, x fastest, and unit quaternions."""
    rng = np.random.default_rng(seed)
    points = torch.from_numpy(rng.random((grains, 3))).cuda()
    d2 = []
    for axis, n in enumerate(cells):
        d = ((torch.arange(n, device="cuda", dtype=torch.float64) + 0.5) / n)[:, None] - points[None, :, axis]
        d2.append((d - d.round()) ** 2)
    at = torch.empty(cells[::-1], dtype=torch.int32, device="cuda")
    for z in range(cells[2]):
        at[z] = (d2[2][z] + d2[1][:, None, :] + d2[0][None, :, :]).argmin(dim=2)
    q = rng.normal(size=(grains, 4))
    q[q[:, 0] < 0] *= -1.0
    return at.cpu().numpy().reshape(-1), q / np.linalg.norm(q, axis=1, keepdims=True)


SIZE = (1.0e-5, 1.0e-5, 1.0e-5)
_SLIP = np.array([  # cF <110>{111}: direction, normal
    (0, 1, -1, 1, 1, 1), (-1, 0, 1, 1, 1, 1), (1, -1, 0, 1, 1, 1), (0, -1, -1, -1, -1, 1),
    (1, 0, 1, -1, -1, 1), (-1, 1, 0, -1, -1, 1), (0, -1, 1, 1, -1, -1), (-1, 0, -1, 1, -1, -1),
    (1, 1, 0, 1, -1, -1), (0, 1, 1, -1, 1, -1), (1, 0, -1, -1, 1, -1), (-1, -1, 0, -1, 1, -1)], dtype=float)
_SCHMID = np.einsum("si,sj->sij", _SLIP[:, :3], _SLIP[:, 3:]) / math.sqrt(6.0)
_HTYPE = np.array([  # slip-slip interaction types (reacting, acting)
    (1, 2, 2, 4, 7, 5, 3, 5, 5, 4, 6, 7), (2, 1, 2, 7, 4, 5, 6, 4, 7, 5, 3, 5), (2, 2, 1, 5, 5, 3, 6, 7, 4, 7, 6, 4),
    (4, 7, 6, 1, 2, 2, 4, 6, 7, 3, 5, 5), (7, 4, 6, 2, 1, 2, 5, 3, 5, 6, 4, 7), (5, 5, 3, 2, 2, 1, 7, 6, 4, 6, 7, 4),
    (3, 5, 5, 4, 6, 7, 1, 2, 2, 4, 7, 6), (6, 4, 7, 5, 3, 5, 2, 1, 2, 7, 4, 6), (6, 7, 4, 7, 6, 4, 2, 2, 1, 5, 5, 3),
    (4, 6, 7, 3, 5, 5, 4, 7, 6, 1, 2, 2), (5, 3, 5, 6, 4, 7, 7, 4, 6, 2, 1, 2), (7, 6, 4, 6, 7, 4, 5, 5, 3, 2, 2, 1)])
# examples/grid/material.yaml
_C11, _C12, _C44 = 106.75e9, 60.41e9, 28.34e9
_XI_0, _XI_INF, _H0, _GDOT0 = 31.0e6, 63.0e6, 75.0e6, 1.0e-3
_HV = np.array((1, 1, 1.4, 1.4, 1.4, 1.4, 1.4))


def _stiffness(E):
    """C : E of the cubic stiffness, (..., 3, 3), E not taken to be symmetric."""
    tr = E.diagonal(dim1=-2, dim2=-1).sum(-1)
    S = _C44 * (E + E.transpose(-1, -2))
    d = _C12 * tr[..., None] + (_C11 - _C12) * E.diagonal(dim1=-2, dim2=-1)
    return S - torch.diag_embed(S.diagonal(dim1=-2, dim2=-1)) + torch.diag_embed(d)


def _points(case, seed):
    """Inputs of an mp case as (n, 3, 3) and (n, 12) tensors in host memory."""
    n, rng = case["n"], np.random.default_rng(seed)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a))  # noqa: E731
    eye = torch.eye(3, dtype=torch.float64)
    P = T(_SCHMID)
    O = torch.linalg.qr(T(rng.normal(size=(n, 3, 3))))[0]
    O = O * torch.linalg.det(O)[:, None, None]
    D = T(0.01 * rng.normal(size=(n, 3, 3)))  # plastic distortion so far
    Fp0 = (eye + D) @ O
    Fp0 = Fp0 / torch.linalg.det(Fp0)[:, None, None] ** (1.0 / 3.0)
    xi0 = T(_XI_0 + (_XI_INF - _XI_0) * (rng.uniform(0.05, 0.5, (n, 1)) + rng.uniform(0.0, 0.1, (n, 12))))
    gamma0 = T(rng.uniform(0.0, 0.02, (n, 12)))
    # a stress whose largest resolved shear is near its slip resistance: flow at the load's rate
    S = T(rng.normal(size=(n, 3, 3)))
    S = S + S.transpose(1, 2)
    S = S - S.diagonal(dim1=1, dim2=2).mean(1)[:, None, None] * eye
    tau = torch.einsum("nij,sij->ns", S, P).abs() / xi0
    S = S * (T(rng.uniform(0.92, 0.97, n)) * (20.0 / case["n_sl"]) ** 0.1 / tau.amax(1))[:, None, None]
    d = S.diagonal(dim1=1, dim2=2)
    E = S / (2.0 * _C44)
    E = E - torch.diag_embed(E.diagonal(dim1=1, dim2=2)) + torch.diag_embed(d / (_C11 - _C12))
    U = eye + E
    Fe0 = O.transpose(1, 2) @ U
    S0 = _stiffness(0.5 * (U.transpose(1, 2) @ U - eye))
    tau = torch.einsum("nij,sij->ns", S0, P)
    gdot = torch.sign(tau) * _GDOT0 * (tau.abs() / xi0) ** case["n_sl"]
    Lp0 = torch.einsum("ns,sij->nij", gdot, P)
    F0 = Fe0 @ Fp0
    step = eye + DT * (Lp0 * T(rng.uniform(0.8, 1.2, (n, 1, 1))) + T(5e-5 * rng.normal(size=(n, 3, 3))))
    F = Fe0 @ step @ Fp0
    Lp = Lp0 * T(rng.uniform(0.8, 1.2, (n, 1, 1)))
    return dict(F=F, F0=F0, Fp0=Fp0, Lp0=Lp0, S0=S0, xi0=xi0, gamma0=gamma0, Lp=Lp)


def _planes(t):
    """(n, 3, 3) -> 9 planes, component i + 3j in plane i + 3j; (n, 12) -> 12 planes."""
    n = t.shape[0]
    return (t.transpose(1, 2).reshape(n, 9) if t.dim() == 3 else t).t().contiguous()


def _materials(lib, case):
    m, p, _ = lib.defaults()
    m.n_sl, m.a_sl = case["n_sl"], case["a_sl"]
    return m, p


def _prepare_mp(case, seed):
    lib, n = library(), case["n"]
    s = {"kind": "mp", "lib": lib, "n": n}
    x = {k: _planes(v).cuda() for k, v in _points(case, seed).items()}
    s["guess"] = x["Lp"].clone()  # the caller's Newton start: Lp of its last evaluation
    for k, c in dict(P=9, Fp=9, S=9, Fe=9, xi=12, gamma=12).items():
        x[k] = torch.zeros((c, n), dtype=torch.float64, device="cuda")
    if case["tangent"]:
        x["dPdF"] = torch.zeros((81, n), dtype=torch.float64, device="cuda")
    x["broken"] = torch.zeros(n, dtype=torch.int32, device="cuda")
    s["x"] = x
    s["planes"] = MpDevicePlanes(**{k: v.data_ptr() for k, v in x.items()})
    s["material"] = _materials(lib, case)
    return s


def _run_mp(s):
    lib, x, (m, p) = s["lib"], s["x"], s["material"]
    x["Lp"].copy_(s["guess"])
    lib.check(lib.sc_mp_update_noalloc(s["n"], DT, C.byref(m), C.byref(p), C.byref(s["planes"]),
                                       torch.cuda.current_stream().cuda_stream), "sc_mp_update_noalloc")
    return {k: x[k] for k in ("Lp", "P", "Fp", "S", "Fe", "xi", "gamma", "broken", "dPdF") if k in x}


def _pinned(n):
    return torch.zeros(n, dtype=torch.float64, pin_memory=True).numpy()


def _prepare_inc(case, seed):
    cells = (case["nx"], case["ny"], case["nz"])
    at, q = _grains(cells, case["grains"], seed)
    rve = Rve(library(), cells, SIZE, at, q, precision=PRECISION[case["precision"]], **EXAMPLE_NUMERICS)
    rve.init()
    load = tension_x(t=60 * DT, N=60, rate=RATE)
    for i in range(WARM + 1):
        rve.forward(False, i > 0, DT, DT if i else 1.0, (60 - i) * DT, load)
        rve.calculate_solution()
        rve.update_coords()
    return {"kind": "inc", "rve": rve, "load": load, "left": (60 - WARM) * DT,
            "F": _pinned(9 * rve.N), "P": _pinned(9 * rve.N)}


def _read(rve, name, out):
    rve.lib.check(rve.lib.sc_rve_get_field(rve.h, SC_FIELD[name], ptr(out), out.size), f"get_field {name}")
    return out


def _answer(rve, F, P):
    sc = rve.scalars()
    return dict(F=_read(rve, "F", F), P=_read(rve, "P", P), P_av=np.array(sc.P_av), C=np.array(sc.C_volAvg))


def _run_inc(s):
    rve = s["rve"]
    rve.forward(True, True, DT, DT, s["left"], s["load"])
    sol = rve.calculate_solution()
    rve.update_coords()
    return dict(_answer(rve, s["F"], s["P"]), converged=int(sol.converged))


def _prepare_job(case, seed):
    cells = (case["nx"], case["ny"], case["nz"])
    at, q = _grains(cells, case["grains"], seed)
    n = cells[0] * cells[1] * cells[2]
    return {"kind": "job", "cells": cells, "at": at, "q": q, "precision": PRECISION[case["precision"]],
            "load": tension_x(t=case["increments"] * DT, N=case["increments"], rate=RATE),
            "F": _pinned(9 * n), "P": _pinned(9 * n), "Fp": _pinned(9 * n), "xi": _pinned(12 * n)}


def _run_job(s):
    rve = Rve(library(), s["cells"], SIZE, s["at"], s["q"], precision=s["precision"], **EXAMPLE_NUMERICS)
    rve.init()
    rve.loop_over_loadcase([s["load"]])
    out = dict(_answer(rve, s["F"], s["P"]), Fp=_read(rve, "Fp", s["Fp"]), xi=_read(rve, "xi", s["xi"]))
    rve.close()
    return out


def _prepare_serve(case, seed):
    lib, rng, jobs = library(), np.random.default_rng(seed), []
    for e, g, j in _edges(case):
        at, q = _grains((e, e, e), g, seed + 7919 * (j + 1))
        spec = RveSpec(lib, (e, e, e), SIZE, at, q, precision=PRECISION[case["precision"]], **EXAMPLE_NUMERICS)
        n = case["increments"]
        jobs.append((spec, [tension_x(t=n * DT, N=n, rate=RATE, rot_q=rotation_to(rng.normal(size=3)))]))
    total = sum(spec.N for spec, _ in jobs)
    return {"kind": "serve", "server": Server(lib, 64 << 30, case["jobs"], batched=True), "jobs": jobs,
            "increments": case["increments"], "P": _pinned(9 * total)}


def _run_serve(s):
    srv, sent = s["server"], []
    for spec, load in s["jobs"]:
        job = srv.add_job(spec, load, keep_resident=True)
        sent.append((job, spec.N, [srv.submit(job) for _ in range(s["increments"])]))
    P_av, status, at = [], [], 0
    for job, n, requests in sent:
        for r in requests:
            got = srv.wait(r)
            P_av.append(list(got.P_av))
            status.append(int(got.status))
        field = s["P"][at:at + 9 * n]
        srv.lib.check(srv.lib.sc_server_get_field(srv.h, job, SC_FIELD["P"], ptr(field), 9 * n), "get_field")
        srv.remove_job(job)
        at += 9 * n
    return dict(P_av=np.array(P_av), P=s["P"], status=np.array(status))


_PREPARE = dict(mp=_prepare_mp, inc=_prepare_inc, job=_prepare_job, serve=_prepare_serve)
_RUN = dict(mp=_run_mp, inc=_run_inc, job=_run_job, serve=_run_serve)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["kind"]](state)


# ---- the material point in plain torch, 64 bits ------------------------------------
def _kinetics(S, xi, n_sl):
    tau = torch.einsum("nij,sij->ns", S, torch.from_numpy(_SCHMID))
    x = tau.abs() / xi
    return _GDOT0 * x ** n_sl * torch.where(tau > 0, 1.0, -1.0), _GDOT0 * n_sl * x ** (n_sl - 1) / xi


def _dot_state(S, xi, case):
    h = torch.from_numpy(_HV[_HTYPE - 1])
    dg = _kinetics(S, xi, case["n_sl"])[0].abs()
    x = 1.0 - xi / _XI_INF
    return torch.cat((_H0 * torch.copysign(x.abs() ** case["a_sl"], x) * (dg @ h.t()), dg), dim=1)


def _hooke(Fe):
    return _stiffness(0.5 * (Fe.transpose(1, 2) @ Fe - torch.eye(3, dtype=torch.float64)))


def _newton(A, Lp, xi, case):
    """The plastic velocity gradient of each point: Newton with the solver's stopping rule and line search."""
    P = torch.from_numpy(_SCHMID)
    eye = torch.eye(3, dtype=torch.float64)
    n = A.shape[0]
    Lp, old, d, step = Lp.clone(), Lp.clone(), torch.zeros_like(Lp), torch.ones(n, dtype=torch.float64)
    rold = torch.zeros(n, dtype=torch.float64)
    todo = torch.arange(n)
    for it in range(1, 41):
        a, lp = A[todo], Lp[todo]
        Fe = a @ (eye - DT * lp)
        g, c = _kinetics(_hooke(Fe), xi[todo], case["n_sl"])
        Lc = torch.einsum("ns,sij->nij", g, P)
        res = lp - Lc
        norm = res.flatten(1).norm(dim=1)
        go = ~(norm < (1e-6 * torch.maximum(lp.flatten(1).norm(dim=1), Lc.flatten(1).norm(dim=1))).clamp_min(1e-8))
        todo, a, lp, Fe, c, res, norm = todo[go], a[go], lp[go], Fe[go], c[go], res[go], norm[go]
        if todo.numel() == 0:
            return Lp
        back = norm >= rold[todo] if it > 1 else torch.zeros_like(norm, dtype=torch.bool)
        b, f = todo[back], todo[~back]
        step[b] = 0.5 * step[b]
        Lp[b] = old[b] + d[b] * step[b][:, None, None]
        if f.numel() == 0:
            continue
        rold[f], old[f], step[f] = norm[~back], lp[~back], 1.0
        K = _stiffness(P)  # P_s : C
        G = Fe[~back].transpose(1, 2) @ a[~back]
        V = torch.einsum("nmp,sml->nspl", G, K)
        J = torch.eye(9, dtype=torch.float64) + DT * torch.einsum(
            "ns,si,nsj->nij", c[~back], P.reshape(12, 9), V.reshape(-1, 12, 9))
        d[f] = -torch.linalg.solve(J, res[~back].reshape(-1, 9)).reshape(-1, 3, 3)
        Lp[f] = Lp[f] + d[f]
    raise ValueError("a point's stress integration did not converge")


def _update(x, case):
    """homogenization_mechanical_response of points that need no substeps."""
    eye = torch.eye(3, dtype=torch.float64)
    n = x["F"].shape[0]
    iFp0 = torch.linalg.inv(x["Fp0"])
    A = x["F"] @ iFp0
    Lp, S = x["Lp"].clone(), x["S0"].clone()
    start = torch.cat((x["xi0"], x["gamma0"]), dim=1)
    dot = _dot_state(S, x["xi0"], case)
    state = start + dot * DT
    last1, atol = torch.zeros_like(dot), torch.tensor([1.0] * 12 + [1e-6] * 12, dtype=torch.float64)
    todo = torch.arange(n)
    for it in range(20):
        last2 = last1[todo] if it else torch.zeros_like(dot)
        last1[todo] = dot[todo]
        Lp[todo] = _newton(A[todo], Lp[todo], state[todo, :12], case)
        S[todo] = _hooke(A[todo] @ (eye - DT * Lp[todo]))
        w0, w1 = _dot_state(S[todo], state[todo, :12], case), last1[todo]
        p12, p22, p01 = ((w0 - w1) * (w1 - last2)).sum(1), ((w1 - last2) ** 2).sum(1), (w0 * w1).sum(1)
        damp = (torch.minimum(p01, p12) < 0) & (p22 > 0)
        z = torch.where(damp, 0.75 + 0.25 * torch.tanh(2.0 + 4.0 * p12 / p22), torch.ones_like(p12))[:, None]
        dot[todo] = w0 * z + w1 * (1.0 - z)
        r = state[todo] - start[todo] - dot[todo] * DT
        state[todo] = state[todo] - r
        todo = todo[(r.abs() > torch.maximum(atol, 1e-6 * state[todo].abs())).any(1)]
        if todo.numel() == 0:
            break
    iFp = iFp0 @ (eye - DT * Lp)
    Fp = torch.linalg.inv(iFp)
    Fe = x["F"] @ iFp
    return dict(Lp=Lp, S=S, P=Fe @ S @ iFp.transpose(1, 2), Fe=Fe, xi=state[:, :12], gamma=state[:, 12:],
                Fp=Fp / torch.linalg.det(Fp)[:, None, None] ** (1.0 / 3.0))


def _tangent(x, o, case):
    """The consistent tangent dP/dF(k,l,p,o) as 81 planes k + 3l + 9p + 27o."""
    P = torch.from_numpy(_SCHMID)
    n = x["F"].shape[0]
    iFp, iFp0 = torch.linalg.inv(o["Fp"]), torch.linalg.inv(x["Fp0"])
    c = _kinetics(o["S"], o["xi"], case["n_sl"])[1]
    H = o["Fe"].transpose(1, 2) @ x["F"] @ iFp0
    U = _stiffness(torch.einsum("nij,sjl->nsil", H, P))
    L = torch.eye(9, dtype=torch.float64) + DT * torch.einsum("ns,nsi,sj->nij", c, U.reshape(n, 12, 9), P.reshape(12, 9))
    R = _stiffness(torch.einsum("npm,nor->npomr", o["Fe"], iFp)).reshape(n, 9, 9)  # row: (p,o), column: (i,j)
    dS = torch.linalg.solve(L, R.transpose(1, 2)).transpose(1, 2).reshape(n, 3, 3, 3, 3)  # p,o,i,j
    w = -DT * c[:, None, None, :] * torch.einsum("sij,npoij->npos", P, dS)
    diFp = torch.einsum("nij,npos,sjk->npoik", iFp0, w, P)
    SiT = o["S"] @ iFp.transpose(1, 2)
    F = x["F"]
    G = iFp @ SiT
    d = torch.einsum("nij,npojk,nkl->npoil", F, diFp, SiT)
    d = d + torch.einsum("nij,npojk,nlk->npoil", F @ iFp, dS, iFp)
    d = d + torch.einsum("nij,npolj->npoil", F @ iFp @ o["S"], diFp)
    for p in range(3):
        d[:, p, :, p, :] += G
    return d.permute(2, 1, 4, 3, 0).reshape(81, n)  # o slowest, then p, l, k


def exact(case, seed):
    """An increment's fields have no value but the solver's own: its iteration stops at loose tolerances."""
    if case["kind"] != "mp":
        return None
    with torch.no_grad():
        x = _points(case, seed)
        o = _update(x, case)
        out = {k: _planes(o[k]) for k in ("Lp", "P", "Fp", "S", "Fe", "xi", "gamma")}
        out["broken"] = None
        if case["tangent"]:
            out["dPdF"] = _tangent(x, o, case)
    return out
