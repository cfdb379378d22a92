"""One- and two-stage Runge-Kutta schemes against the oracle, bit for bit on the parity path: the only stage of a
one-stage scheme starts from and ends in the state buffer, and its tiles read their neighbours' cells, which other tiles
of the same launch write."""
import numpy as np
import pytest

import mosegpu
from mosegpu import Context, DeviceCase, cases
from mosegpu.core import BC_EXTRAPOLATION, BC_NONE, BC_SYMMETRY, BC_WALL_ADIABATIC
from oracle_bind import OracleCase
from test_gpu_walls_sa import interiors, run_device

pytestmark = pytest.mark.gpu

PER, SYM, WA, EX, NO = "periodic", BC_SYMMETRY, BC_WALL_ADIABATIC, BC_EXTRAPOLATION, BC_NONE


def box(dims, faces, viscous, n_rk, integration="cons"):
    case = cases.box_case(dims, dict(zip(range(1, 7), faces)), extent=(1.0, 0.8, 0.9), viscous=viscous,
                          mu_of_T=cases.sutherland(2e-3, 300.0) if viscous else None, limiter="vanleer",
                          ndir=sum(d > 1 for d in dims), n_rk=n_rk, integration=integration)
    rng = np.random.Generator(np.random.PCG64(29))
    V = case.layout.interior(case.P, 0)
    V[0] = 1.1 + 0.1 * rng.uniform(-1, 1, V[0].shape)
    for q in range(3):
        V[1 + q] = 20.0 * rng.uniform(-1, 1, V[0].shape)
    V[4] = 1e5 * (1.0 + 0.05 * rng.uniform(-1, 1, V[0].shape))
    cases.fill_ghosts_nearest(case.layout, case.P)
    return case


def agree(case, steps, path, tile):
    Pg, rep, _ = run_device(case, steps, path, tile)
    Po = case.P.copy()
    dts = OracleCase(case).step(Po, steps)
    got, want = interiors(case, Pg), interiors(case, Po)
    if path != mosegpu.PATH_FAST:
        assert np.array_equal(got, want)
        assert abs(rep.time - dts.sum()) <= 1e-15 * dts.sum()
        return
    speed = np.sqrt((want[1:4] ** 2).sum(axis=0)) + np.sqrt(want[4] / want[0])
    for q in range(5):
        scale = speed.max() if 1 <= q <= 3 else np.abs(want[q]).max()
        assert np.abs(got[q] - want[q]).max() <= 1e-12 * scale


@pytest.mark.parametrize("n_rk", [1, 2])
@pytest.mark.parametrize("path", [mosegpu.PATH_FUSED, mosegpu.PATH_FAST, mosegpu.PATH_PLAIN])
@pytest.mark.parametrize("dims,faces,viscous,tile", [
    ((37, 28, 12), (PER, PER, PER, PER, PER, PER), True, (8, 8, 4)),
    ((37, 28, 12), (PER, PER, SYM, EX, WA, EX), True, (8, 4, 4)),
    ((34, 26, 10), (NO, WA, PER, PER, PER, PER), False, (32, 8, 1)),
    ((130, 70, 1), (EX, SYM, PER, PER, NO, NO), False, (16, 8, 1)),
    ((300, 1, 1), (EX, EX, NO, NO, NO, NO), False, (128, 1, 1))])
def test_stage_counts(gpu_ready, dims, faces, viscous, tile, path, n_rk):
    print(f"rk stages: {n_rk} {dims} path {path}", flush=True)
    agree(box(dims, faces, viscous, n_rk), 5, path, (0, 0, 0) if path == mosegpu.PATH_PLAIN else tile)


@pytest.mark.parametrize("path", [mosegpu.PATH_FUSED, mosegpu.PATH_PLAIN])
def test_one_stage_primitive_update(gpu_ready, path):
    agree(box((37, 28, 12), (PER, PER, SYM, EX, WA, EX), True, 1, "prim"), 5, path,
          (8, 4, 4) if path == mosegpu.PATH_FUSED else (0, 0, 0))


@pytest.mark.parametrize("path,tile", [(mosegpu.PATH_FUSED, (8, 4, 4)), (mosegpu.PATH_PLAIN, (0, 0, 0))])
def test_one_stage_turbulent_channel(gpu_ready, path, tile):
    """SA on eight blocks: the source reads its neighbours in the plain path's update too.  The bar is the SA cases'."""
    case = cases.channel_lattice(nb=(2, 2, 2), wmin=9, wmax=14, seed=11)
    case.scheme.n_rk = 1
    Pg, _, _ = run_device(case, 4, path, tile)
    Po = case.P.copy()
    OracleCase(case).step(Po, 4)
    got, want = interiors(case, Pg), interiors(case, Po)
    for q in range(6):
        assert np.abs(got[q] - want[q]).max() <= 1e-12 * max(np.abs(want[q]).max(), 1e-300)


def test_one_stage_replays(gpu_ready):
    """The captured step of a one-stage scheme, several calls on one state, equals the eager launches."""
    case = box((37, 28, 12), (PER, PER, SYM, EX, WA, EX), True, 1)
    out = []
    for graph in (True, False):
        ctx = Context(case.tables)
        dc = DeviceCase(ctx, case)
        dc.upload(case.P)
        dc.tune(mosegpu.PATH_FUSED, (8, 8, 4), graph=graph)
        for n in (1, 3, 2):
            dc.step(n)
        out.append(interiors(case, dc.download()))
        dc.destroy()
        ctx.close()
    assert np.array_equal(out[0], out[1])
    Po = case.P.copy()
    OracleCase(case).step(Po, 6)
    assert np.array_equal(out[0], interiors(case, Po))
