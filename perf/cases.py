"""The work that programs have this library do, as cases to be timed and compared: time steps of flow cases from a
one-dimensional tube to a 256^3 box, on the parity path (the default, the reference's bits) and on the performance
path, several cases served at once, batches of stiff chemistry cells, and a reacting box.

A pass of a flow case is what a program does with a case that it keeps on the device: the state goes up, `steps` RK3
steps run, the state comes down.  A pass of a chemistry batch is upload, integration over dt, download.  Every pass
starts from the same state, so passes can be repeated and their outputs compared.

exact() gives the same results for the cases of one calorically perfect gas on uniform boxes from whole-array
statements in double precision (torch), without this library.
"""
import ctypes
import dataclasses
import functools
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "mose-gpu_amd"))

from mosegpu import PATH_FAST, PATH_FUSED, Context, DeviceCase, DeviceChem, cases, chem, serve  # noqa: E402
from mosegpu.core import Layout, ThermoTables, dptr, lib  # noqa: E402

PATHS = {"parity": PATH_FUSED, "fast": PATH_FAST}
GAMMA = cases.CP_AIR / (cases.CP_AIR - cases.R_AIR)


def listed():
    return [
        # a shock tube, the smallest call: a thousand cells on the default path, launches and latency
        {"name": "sod-1000", "kind": "sod", "n": 1000, "steps": 100, "path": "parity"},
        # two-dimensional four-quadrant problems at both ends of what is served (n in 64..1024), an odd size at the top
        {"name": "riemann2d-64", "kind": "riemann2d", "n": 64, "steps": 40, "path": "fast"},
        {"name": "riemann2d-1023", "kind": "riemann2d", "n": 1023, "steps": 20, "path": "fast"},
        # viscous Taylor-Green boxes: the smallest served, an uneven odd one on the parity path, the benchmark's
        {"name": "tgv-48", "kind": "tgv", "n1": 48, "n2": 48, "n3": 48, "steps": 20, "path": "fast"},
        {"name": "tgv-101x97x89", "kind": "tgv", "n1": 101, "n2": 97, "n3": 89, "steps": 10, "path": "parity"},
        {"name": "tgv-256", "kind": "tgv", "n1": 256, "n2": 256, "n3": 256, "steps": 10, "path": "fast"},
        # uneven blocks with a wall, far field and Spalart-Allmaras: a production-like mesh, and a small one on the
        # parity path
        {"name": "lattice-3x2x2", "kind": "lattice", "b1": 3, "b2": 2, "b3": 2, "wmin": 24, "wmax": 72,
         "solver": "LMRoe", "steps": 10, "path": "fast"},
        {"name": "lattice-2x2x2", "kind": "lattice", "b1": 2, "b2": 2, "b3": 2, "wmin": 9, "wmax": 32,
         "solver": "HLLC", "steps": 20, "path": "parity"},
        # a server's mix: two- and three-dimensional cases of different sizes stepping at the same time
        {"name": "served-6", "kind": "served", "count": 6, "n2d": 300, "n3d": 72, "steps": 20},
        # batches of hydrogen-air cells over a microsecond, both integrators
        {"name": "rodas-16384", "kind": "chem", "method": "rodas", "cells": 16384, "dt": 1e-6},
        {"name": "radau5-4096", "kind": "chem", "method": "radau5", "cells": 4096, "dt": 1e-6},
        # Strang-split steps of a viscous reacting box: nine species, chemistry on the resident state
        {"name": "reacting-20x16x12", "kind": "reacting", "n1": 20, "n2": 16, "n3": 12, "viscous": True, "steps": 2},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sod", "riemann2d", "riemann2d", "tgv", "tgv", "tgv", "lattice", "lattice", "served", "chem",
                       "chem", "reacting"])
    path = rng.choice(["parity", "fast"])
    if kind == "sod":
        return {"kind": kind, "n": _log(rng, 60, 4000), "steps": rng.randint(50, 150), "path": path}
    if kind == "riemann2d":
        return {"kind": kind, "n": _log(rng, 48, 1024), "steps": rng.randint(8, 24), "path": path}
    if kind == "tgv":
        n = _log(rng, 24, 200)
        return {"kind": kind, "n1": n, "n2": max(9, n + rng.randint(-n // 8, n // 8)),
                "n3": max(9, n + rng.randint(-n // 8, n // 8)), "steps": rng.randint(5, 10), "path": path}
    if kind == "lattice":
        wmin = rng.randint(8, 24)
        return {"kind": kind, "b1": rng.randint(1, 3), "b2": rng.randint(1, 2), "b3": rng.randint(1, 2), "wmin": wmin,
                "wmax": wmin + rng.randint(4, 48), "solver": rng.choice(["HLLC", "AUSM+", "LMRoe", "HLLE"]),
                "steps": rng.randint(5, 10), "path": path}
    if kind == "served":
        return {"kind": kind, "count": rng.randint(2, 8), "n2d": _log(rng, 64, 400), "n3d": _log(rng, 32, 80),
                "steps": rng.randint(8, 20)}
    if kind == "chem":
        return {"kind": kind, "method": rng.choice(["rodas", "radau5"]), "cells": _log(rng, 100, 8192),
                "dt": math.exp(rng.uniform(math.log(5e-8), math.log(1e-6)))}
    return {"kind": kind, "n1": rng.randint(6, 20), "n2": rng.randint(6, 16), "n3": rng.randint(5, 12),
            "viscous": rng.random() < 0.5, "steps": 1}


# ------------------------------------------------------------------------------------------------------------
# initial fields [nprim, n3, n2, n1] of the interior, from the seed alone
# ------------------------------------------------------------------------------------------------------------
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _noise(shape, seed):
    """Uniform in [-1, 1]."""
    g = torch.Generator(device=_device())
    g.manual_seed(seed)
    return torch.rand(shape, dtype=torch.float64, device=_device(), generator=g) * 2.0 - 1.0


def _centres(n, length=1.0):
    return (torch.arange(n, dtype=torch.float64, device=_device()) + 0.5) * (length / n)


def sod_field(n, seed):
    r = np.random.Generator(np.random.PCG64(seed))
    q = torch.zeros(5, 1, 1, n, dtype=torch.float64, device=_device())
    left = _centres(n) < 0.5
    q[0] = torch.where(left, 1.0 + 0.2 * r.uniform(), 0.125 + 0.05 * r.uniform())
    q[4] = torch.where(left, 1.0 + 0.2 * r.uniform(), 0.1 + 0.05 * r.uniform())
    return q


def riemann2d_field(n, seed):
    """Four seeded quadrant states: density and pressure in [0.3, 2], a speed of at most 0.7."""
    r = np.random.Generator(np.random.PCG64(seed))
    right = (_centres(n) >= 0.5)[None, :].expand(n, n)
    upper = (_centres(n) >= 0.5)[:, None].expand(n, n)
    q = torch.zeros(5, 1, n, n, dtype=torch.float64, device=_device())
    for k in range(4):
        rho, p = r.uniform(0.3, 2.0, size=2)
        speed, angle = r.uniform(0.0, 0.7), r.uniform(0.0, 2 * math.pi)
        here = (right == bool(k & 1)) & (upper == bool(k & 2))
        for s, v in ((0, rho), (1, speed * math.cos(angle)), (2, speed * math.sin(angle)), (4, p)):
            q[s, 0][here] = v
    return q


TGV = {"mach": 0.1, "re": 1600.0, "T0": 300.0, "p0": 101325.0, "prandtl": 0.72, "cfl": 0.4, "vnn": 0.5}
TGV["V0"] = TGV["mach"] * math.sqrt(GAMMA * cases.R_AIR * TGV["T0"])
TGV["rho0"] = TGV["p0"] / (cases.R_AIR * TGV["T0"])


def tgv_field(n1, n2, n3, seed):
    """The vortex of mosegpu.cases.taylor_green (isothermal start) with a seeded velocity perturbation of 1e-3 V0."""
    V0, rho0 = TGV["V0"], TGV["rho0"]
    x = _centres(n1, 2 * math.pi)[None, None, :]
    y = _centres(n2, 2 * math.pi)[None, :, None]
    z = _centres(n3, 2 * math.pi)[:, None, None]
    q = torch.empty(5, n3, n2, n1, dtype=torch.float64, device=_device())
    q[4] = TGV["p0"] + rho0 * V0 ** 2 / 16.0 * (torch.cos(2 * x) + torch.cos(2 * y)) * (torch.cos(2 * z) + 2.0)
    q[0] = q[4] / (cases.R_AIR * TGV["T0"])
    q[1:4] = 1e-3 * V0 * _noise((3, n3, n2, n1), seed)
    q[1] += V0 * torch.sin(x) * torch.cos(y) * torch.cos(z)
    q[2] -= V0 * torch.cos(x) * torch.sin(y) * torch.cos(z)
    return q


# ------------------------------------------------------------------------------------------------------------
# states
# ------------------------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=4)
def _mesh(kind, *size):
    """The mesh, records and scheme of a flow case: what a program reads from its case files."""
    if kind == "sod":
        return cases.sod(size[0])
    if kind == "riemann2d":
        return cases.riemann2d(size[0])
    if kind == "tgv":
        return cases.taylor_green(dims=size, cfl=TGV["cfl"])
    if kind == "lattice":
        b1, b2, b3, wmin, wmax, solver = size
        return cases.channel_lattice(nb=(b1, b2, b3), wmin=wmin, wmax=wmax, riemann=solver)
    return cases.reacting_box(size[:3], viscous=size[3], T_range=(1200.0, 1700.0))


def _pinned(shape):
    return torch.zeros(shape, dtype=torch.float64, pin_memory=torch.cuda.is_available())


class Flow:
    """A flow case on the device, its initial state and the buffer of its results in pinned host memory."""

    def __init__(self, mesh, field, path, tile):
        layout = mesh.layout
        start = _pinned((mesh.nprim, layout.NC))
        self.start, self.result = start.numpy(), _pinned((mesh.nprim, layout.NC)).numpy()
        if field is None:
            self.start[...] = mesh.P
        else:
            # the ghost rows (filled by the first step) start as the nearest cells
            padded = torch.nn.functional.pad(field[None], (2,) * 6, mode="replicate")[0]
            start.copy_(padded.reshape(mesh.nprim, layout.NC))
        self.case = dataclasses.replace(mesh, P=self.start)
        self.ctx = Context(self.case.tables)
        self.dc = DeviceCase(self.ctx, self.case)
        self.dc.upload(self.start)
        if tile is not None:
            self.dc.tune(path, tile)       # (0, 0, 0): the autotuner; None: the path and the tile of a new case

    def outputs(self, report):
        self.ctx.check(lib().mose_state_download(self.ctx.h, self.dc.id, dptr(self.result)), "mose_state_download")
        lay = self.case.layout
        return {"dt": report.dt, "state": [lay.interior(self.result, b) for b in range(lay.nb)]}

    def close(self):
        self.ctx.close()


class State:
    def __init__(self, steps=0):
        self.steps, self.flows, self.chem, self.chem_ctx = steps, [], None, None

    def __del__(self):
        for f in self.flows:
            f.close()
        if self.chem is not None:
            self.chem.destroy()
        if self.chem_ctx is not None:
            self.chem_ctx.close()


def _served(case):
    """The cases of a served mix: alternately two- and three-dimensional, of different sizes."""
    out = []
    for q in range(case["count"]):
        if q % 2 == 0:
            n = max(32, int(case["n2d"] * (1.0 - 0.11 * q)))
            out.append(("riemann2d", n))
        else:
            n = max(16, int(case["n3d"] * (1.0 - 0.07 * q)))
            out.append(("tgv", n, n, n))
    return out


def _field(item, seed):
    return {"sod": sod_field, "riemann2d": riemann2d_field, "tgv": tgv_field}[item[0]](*item[1:], seed)


def _item(case):
    return (case["kind"], case["n1"], case["n2"], case["n3"]) if case["kind"] == "tgv" else (case["kind"], case["n"])


def prepare(case, seed):
    kind = case["kind"]
    st = State(case.get("steps", 0))
    st.kind = kind
    if kind in ("sod", "riemann2d", "tgv"):
        item = _item(case)
        tune = None if kind == "sod" and case["path"] == "parity" else (0, 0, 0)
        st.flows = [Flow(_mesh(*item), _field(item, seed), PATHS[case["path"]], tune)]
    elif kind == "served":
        for q, item in enumerate(_served(case)):
            mesh = _mesh(*item)
            st.flows.append(Flow(mesh, _field(item, seed + 1000 * q), PATH_FAST, serve.serve_tile(mesh, PATH_FAST)))
    elif kind == "lattice":
        mesh = _mesh(kind, case["b1"], case["b2"], case["b3"], case["wmin"], case["wmax"], case["solver"])
        P = mesh.P.copy()
        P[1:4] += 1e-3 * mesh.meta["U"] * _noise((3, mesh.layout.NC), seed).cpu().numpy()
        P[5] *= 1.0 + 0.1 * _noise((mesh.layout.NC,), seed + 1).cpu().numpy()
        st.flows = [Flow(dataclasses.replace(mesh, P=P), None, PATHS[case["path"]], (0, 0, 0))]
    elif kind == "chem":
        mech = chem.h2_air_mechanism()
        # RADAU5 users keep to temperatures where its simplified Newton iteration converges
        lo = 900.0 if case["method"] == "rodas" else 1100.0
        st.cells = chem.h2_air_cells(case["cells"], seed=seed, T_range=(lo, 2500.0))
        st.chem_ctx = Context(ThermoTables(mech.wm, mech.cp, mech.h, names=mech.names))
        st.chem = DeviceChem(st.chem_ctx, mech, case["cells"])
        st.dt, st.opts = case["dt"], chem.ode_opts(method={"rodas": 1, "radau5": 2}[case["method"]])
    else:
        mesh = _mesh(kind, case["n1"], case["n2"], case["n3"], case["viscous"])
        own = cases.reacting_box((case["n1"], case["n2"], case["n3"]), viscous=case["viscous"], T_range=(1200.0, 1700.0),
                                 seed=seed)
        st.flows = [Flow(dataclasses.replace(mesh, P=own.P), None, PATH_FUSED, (0, 0, 0))]
        f = st.flows[0]
        st.chem_ctx = Context(f.case.tables)
        st.chem = DeviceChem(st.chem_ctx, chem.h2_air_mechanism(), 1)
        f.dc.chem_attach(st.chem, chem.ode_opts())
    return st


def run(state):
    if state.kind == "chem":
        state.chem.upload(state.cells)
        state.chem.advance(state.dt, state.opts)
        cells, hr, idid, nstep = state.chem.download()
        return {"cells": cells, "hr": hr, "idid": idid, "nstep": nstep}
    for f in state.flows:
        f.dc.upload(f.start)
    if state.kind != "served":
        f = state.flows[0]
        return f.outputs(f.dc.step(state.steps))
    for f in state.flows:
        f.dc.launch(state.steps)
    left, reports = list(enumerate(state.flows)), {}
    while left:
        still = []
        for q, f in left:
            rep = f.dc.poll()
            if rep is None:
                still.append((q, f))
            else:
                reports[q] = rep
        left = still
    return [f.outputs(reports[q]) for q, f in enumerate(state.flows)]


# ------------------------------------------------------------------------------------------------------------
# work
# ------------------------------------------------------------------------------------------------------------
def _flow_work(cells, steps, ndir, nprim, viscous, rans):
    """Per cell-stage: the stage input and the step base read, the output written, and the geometry read once (12 face
    normals and areas, 3 lengths, the volume, 9 metric terms if viscous, the wall distance with RANS); per step the
    time step; the state up and down once.  Arithmetic: a MUSCL + Riemann face, a viscous face, an update."""
    geo = 4 * ndir + ndir + 1 + (9 if viscous else 0) + (1 if rans else 0)
    scale = nprim / 5.0
    flops = ndir * (330 + (210 if viscous else 0)) * scale + 130 * scale + (150 if rans else 0)
    return {"bytes": cells * (steps * (3 * 8 * (3 * nprim + geo) + 8 * (nprim + 12)) + 16 * nprim),
            "flops": cells * steps * (3 * flops + 60)}


def _rodas_steps(dt):
    """Mean step attempts per hydrogen-air cell at rtol 1e-8 (about 240 over 5e-8 s, 1400 over 2e-7 s, 2800 over
    1e-6 s)."""
    x = math.log(dt)
    return float(np.exp(np.interp(x, np.log([5e-8, 2e-7, 1e-6]), np.log([240.0, 1400.0, 2800.0]))))


# a right-hand side: 19 rates of progress of about 25 operations, nine productions over the reactions, the energy
RHS = 900.0
RODAS_STEP = 16 * RHS + 700 + 6 * 200 + 300            # 16 right-hand sides, one 10 x 10 LU, six solves
RADAU_STEP = 11 * RHS + 3 * 4 * RHS + 700 * 5 + 4 * 1000   # Jacobian, about four Newton iterations, both LUs


def work(case):
    kind, steps = case["kind"], case.get("steps", 0)
    if kind == "sod":
        return _flow_work(case["n"], steps, 1, 5, False, False)
    if kind == "riemann2d":
        return _flow_work(case["n"] ** 2, steps, 2, 5, False, False)
    if kind == "tgv":
        return _flow_work(case["n1"] * case["n2"] * case["n3"], steps, 3, 5, True, False)
    if kind == "lattice":
        rng = np.random.Generator(np.random.PCG64(7))    # the widths of cases.channel_lattice
        w = [rng.integers(case["wmin"], case["wmax"] + 1, size=case[b]) for b in ("b1", "b2", "b3")]
        return _flow_work(int(np.prod([x.sum() for x in w])), steps, 3, 6, True, True)
    if kind == "served":
        both = [_flow_work(i[1] ** 2, steps, 2, 5, False, False) if i[0] == "riemann2d"
                else _flow_work(i[1] ** 3, steps, 3, 5, True, False) for i in _served(case)]
        return {k: sum(w[k] for w in both) for k in ("bytes", "flops")}
    if kind == "chem":
        per = _rodas_steps(case["dt"]) * RODAS_STEP if case["method"] == "rodas" else 400 * RADAU_STEP
        return {"bytes": case["cells"] * (2 * 10 * 8 + 16), "flops": case["cells"] * per}
    cells = case["n1"] * case["n2"] * case["n3"]
    w = _flow_work(cells, 2 * steps, 3, 13, case["viscous"], False)     # two half transport steps per step
    return {"bytes": w["bytes"], "flops": w["flops"] + cells * steps * 1500.0 * RODAS_STEP}


# ------------------------------------------------------------------------------------------------------------
# the same results in whole-array statements (a calorically perfect gas, h = cp T, on a uniform box)
# ------------------------------------------------------------------------------------------------------------
def _shift(q, axis, k):
    return torch.roll(q, -k, dims=axis)


def _minmod(x, y):
    return torch.where(x * y < 0, torch.zeros_like(x), torch.where(x.abs() > y.abs(), y, x))


def _albada(x, y):
    return (y * y * x + y * x * x) / (x * x + y * y + 1e-300)


def _prim_to_cons(q):
    c = torch.empty_like(q)
    c[0] = q[0]
    c[1:4] = q[0] * q[1:4]
    c[4] = q[4] / (GAMMA - 1.0) + 0.5 * q[0] * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2)
    return c


def _cons_to_prim(c):
    q = torch.empty_like(c)
    q[0] = c[0]
    q[1:4] = c[1:4] / c[0]
    q[4] = (GAMMA - 1.0) * (c[4] - 0.5 * c[0] * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2))
    return q


def _physical(q, d):
    """The Euler flux along direction d and the total enthalpy."""
    un = q[1 + d]
    h0 = GAMMA / (GAMMA - 1.0) * q[4] / q[0] + 0.5 * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2)
    f = torch.stack([q[0] * un, q[0] * un * q[1], q[0] * un * q[2], q[0] * un * q[3], q[0] * un * h0])
    f[1 + d] += q[4]
    return f, h0


def _roe(L, R, hL, hR):
    """Velocity [3], total enthalpy and sound speed of the Roe state."""
    sl, sr = torch.sqrt(L[0]), torch.sqrt(R[0])
    vel = (sl * L[1:4] + sr * R[1:4]) / (sl + sr)
    h = (sl * hL + sr * hR) / (sl + sr)
    return vel, h, torch.sqrt((GAMMA - 1.0) * (h - 0.5 * (vel ** 2).sum(0)))


def _hllc(L, R, d):
    fL, hL = _physical(L, d)
    fR, hR = _physical(R, d)
    vel, _, a = _roe(L, R, hL, hR)
    uL, uR = L[1 + d], R[1 + d]
    aL, aR = torch.sqrt(GAMMA * L[4] / L[0]), torch.sqrt(GAMMA * R[4] / R[0])
    s1 = torch.minimum(uL - aL, vel[d] - a).clamp(max=0.0)
    s4 = torch.maximum(uR + aR, vel[d] + a).clamp(min=0.0)
    ss = (R[4] - L[4] + L[0] * uL * (s1 - uL) - R[0] * uR * (s4 - uR)) / (L[0] * (s1 - uL) - R[0] * (s4 - uR))
    ps = L[0] * (uL - s1) * (uL - ss) + L[4]

    def side(q, f, s, u):
        c = _prim_to_cons(q)
        star = torch.stack([c[k] * (s - u) for k in range(5)])
        star[1 + d] += ps - q[4]
        star[4] += ps * ss - q[4] * u
        return f + s * (star / (s - ss) - c)

    left = torch.where(s1 >= 0.0, fL, side(L, fL, s1, uL))
    right = torch.where(s4 <= 0.0, fR, side(R, fR, s4, uR))
    return torch.where((s1 >= 0.0) | (ss >= 0.0), left, right)


def _roe_flux(L, R, d):
    """Roe's flux: the acoustic, entropy and shear waves by their strengths."""
    fL, hL = _physical(L, d)
    fR, hR = _physical(R, d)
    vel, h, a = _roe(L, R, hL, hR)
    rho, un = torch.sqrt(L[0] * R[0]), vel[d]
    dp, du = R[4] - L[4], R[1:4] - L[1:4]
    w1 = (un - a).abs() * 0.5 * (dp / a ** 2 - rho * du[d] / a)
    w5 = (un + a).abs() * 0.5 * (dp / a ** 2 + rho * du[d] / a)
    w4 = un.abs() * (R[0] - L[0] - dp / a ** 2)
    ws = un.abs() * rho
    shear = du.clone()
    shear[d] = 0.0
    diss = torch.empty_like(fL)
    diss[0] = w1 + w4 + w5
    diss[1:4] = (w1 + w4 + w5) * vel + ws * shear
    diss[1 + d] += (w5 - w1) * a
    diss[4] = (w1 + w5) * h + (w5 - w1) * a * un + w4 * 0.5 * (vel ** 2).sum(0) + ws * (vel * shear).sum(0)
    return 0.5 * (fL + fR) - 0.5 * diss


def _half_slopes(q, axis, limiter):
    """Half the limited difference of each cell along axis of the periodic (or padded) field."""
    return 0.5 * limiter(_shift(q, axis, 1) - q, q - _shift(q, axis, -1))


def _euler_residual(q, width):
    """The residual of HLLC + minmod between extrapolation faces; q [5, n3, n2, n1], directions with one cell have no
    net flux."""
    res = torch.zeros_like(q)
    for d in range(3):
        axis, n = 3 - d, q.shape[3 - d]
        if n < 2:
            continue
        first, last = q.narrow(axis, 0, 1), q.narrow(axis, n - 1, 1)
        lo = 3 * first - 3 * q.narrow(axis, 1, 1) + q.narrow(axis, 2, 1)      # the cubic ghost cell
        hi = 3 * last - 3 * q.narrow(axis, n - 2, 1) + q.narrow(axis, n - 3, 1)
        e = torch.cat([lo, q, hi], axis)
        s = _half_slopes(e, axis, _minmod).narrow(axis, 1, n)
        f = _hllc((q + s).narrow(axis, 0, n - 1), (q - s).narrow(axis, 1, n - 1), d)
        f = torch.cat([_physical(first, d)[0], f, _physical(last, d)[0]], axis)
        res += (f.narrow(axis, 1, n) - f.narrow(axis, 0, n)) / width[d]
    return res


def _viscosity(T):
    """The Sutherland law of the vortex on whole kelvins, linear between them."""
    def law(t):
        return (TGV["rho0"] * TGV["V0"] / TGV["re"]) * (t / TGV["T0"]) ** 1.5 * (TGV["T0"] + 110.4) / (t + 110.4)
    t = torch.floor(T)
    return law(t) + (law(t + 1.0) - law(t)) * (T - t)


def _tgv_residual(q, width):
    """The residual of Roe + van Albada and the central viscous fluxes on the periodic box."""
    res = torch.zeros_like(q)
    T = q[4] / (q[0] * cases.R_AIR)
    fields = torch.cat([q[1:4], T[None]])                 # u, v, w, T
    for d in range(3):
        axis = 3 - d
        s = _half_slopes(q, axis, _albada)
        f = _roe_flux(q + s, _shift(q - s, axis, 1), d)
        mid = 0.5 * (q + _shift(q, axis, 1))
        mu = _viscosity(mid[4] / (mid[0] * cases.R_AIR))
        grad = []
        for e in range(3):
            if e == d:
                grad.append((_shift(fields, axis, 1) - fields) / width[d])
            else:
                c = _shift(fields, 3 - e, 1) - _shift(fields, 3 - e, -1)
                grad.append(0.25 * (c + _shift(c, axis, 1)) / width[e])
        div = grad[0][0] + grad[1][1] + grad[2][2]
        power = mu * cases.CP_AIR / TGV["prandtl"] * grad[d][3]
        for e in range(3):
            tau = mu * (grad[d][e] + grad[e][d])
            if e == d:
                tau = tau - 2.0 / 3.0 * mu * div
            f[1 + e] -= tau
            power = power + tau * mid[1 + e]
        f[4] -= power
        res += (f - _shift(f, axis, -1)) / width[d]
    return res


def _time_step(q, width, ndir, cfl, vnn):
    a = torch.sqrt(GAMMA * q[4] / q[0])
    dt = min(float((width[d] / (q[1 + d].abs() + a)).min()) * cfl for d in range(ndir))
    if vnn:
        mu = _viscosity(q[4] / (q[0] * cases.R_AIR))
        dt = min([dt] + [float((q[0] * width[d] ** 2 * vnn / mu).min()) for d in range(ndir)])
    return dt


def _march(item, steps, seed):
    q = _field(item, seed)
    if item[0] == "tgv":
        width = [2 * math.pi / n for n in item[1:]]
        residual, ndir, cfl, vnn = _tgv_residual, 3, TGV["cfl"], TGV["vnn"]
    else:
        width = [1.0 / item[1]] * 3
        residual, ndir, cfl, vnn = _euler_residual, (1 if item[0] == "sod" else 2), 0.5, 0.0
    dt = 0.0
    for _ in range(steps):
        dt = _time_step(q, width, ndir, cfl, vnn)
        base = _prim_to_cons(q)
        for weight in (1.0, 0.25, 2.0 / 3.0):
            c = base + weight * (_prim_to_cons(q) - base - dt * residual(q, width))
            q = _cons_to_prim(c)
    return {"dt": dt, "state": [q]}


def exact(case, seed):
    if case["kind"] == "served":
        return [_march(item, case["steps"], seed + 1000 * q) for q, item in enumerate(_served(case))]
    if case["kind"] in ("sod", "riemann2d", "tgv"):
        return _march(_item(case), case["steps"], seed)
    return None     # the walled channels and the stiff integrations take far longer than this in whole-array form
