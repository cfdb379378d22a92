"""The ghost rows of a download, as include/mose_gpu.h states them: those that the last step's first stage filled (of
the state that the step started from), or, where an inviscid case has no-flux faces of a direction of one cell, those
of the state returned."""
import numpy as np
import pytest

import mosegpu
from mosegpu import Context, DeviceCase
from mosegpu.core import BC_EXTRAPOLATION, BC_NONE, BC_SYMMETRY, BC_WALL_ADIABATIC
from oracle_bind import OracleCase
from test_gpu_boundary_plan import seeded
from test_gpu_walls_sa import run_device

pytestmark = pytest.mark.gpu

PER, SYM, WA, EX, NO = "periodic", BC_SYMMETRY, BC_WALL_ADIABATIC, BC_EXTRAPOLATION, BC_NONE


def ghost_layers(case, P):
    """The ghosts behind the faces of the one block, without its edges and corners; behind symmetry faces only the first
    layer is filled."""
    v, typ = case.layout.block_view(P, 0), {int(r["f"]): int(r["typ"]) for r in case.records}
    out = []
    for f in range(1, 7):
        ax = 3 - (f - 1) // 2
        for g in (0, 1):
            if typ[f] == SYM and g == 1:
                continue
            idx = [slice(None)] + [slice(2, -2)] * 3
            idx[ax] = 1 - g if f % 2 == 1 else v.shape[ax] - 2 + g
            out.append(v[tuple(idx)].copy())
    return out


@pytest.mark.parametrize("steps", [1, 3])
@pytest.mark.parametrize("dims,faces,viscous,returned", [
    ((7, 6, 5), (SYM, EX, PER, PER, WA, NO), True, False),
    ((7, 6, 5), (SYM, EX, PER, PER, WA, NO), False, False),
    ((9, 7, 1), (EX, SYM, PER, PER, NO, NO), True, False),
    ((9, 7, 1), (EX, SYM, PER, PER, SYM, NO), False, False),      # no plan: every stage fills every ghost
    ((9, 7, 1), (EX, SYM, PER, PER, NO, NO), False, True),
    ((11, 1, 1), (EX, EX, NO, NO, NO, NO), False, True)])
def test_ghosts_of_a_download(gpu_ready, dims, faces, viscous, returned, steps):
    case = seeded(dims, faces, viscous)
    print(f"download ghosts: {dims} {faces} viscous {viscous} steps {steps}", flush=True)
    Pg, _, _ = run_device(case, steps, mosegpu.PATH_FUSED, (8, 4, 4) if viscous or dims[2] > 1 else (0, 0, 0))
    oracle = OracleCase(case)
    Po = case.P.copy()
    oracle.step(Po, steps if returned else steps - 1)
    oracle.fill_ghosts(Po)
    for got, want in zip(ghost_layers(case, Pg), ghost_layers(case, Po)):
        assert np.array_equal(got, want)


def test_plain_steps_after_fused_ones(gpu_ready):
    """The plain path fills every ghost, whatever path the steps before took."""
    case = seeded((9, 7, 1), (EX, SYM, PER, PER, NO, NO), False)
    print("download ghosts: two fused steps, one plain", flush=True)
    ctx = Context(case.tables)
    dc = DeviceCase(ctx, case)
    dc.upload(case.P)
    dc.step(2)
    dc.tune(mosegpu.PATH_PLAIN)
    dc.step(1)
    Pg = dc.download()
    dc.destroy()
    ctx.close()
    oracle = OracleCase(case)
    Po = case.P.copy()
    oracle.step(Po, 2)
    oracle.fill_ghosts(Po)
    for got, want in zip(ghost_layers(case, Pg), ghost_layers(case, Po)):
        assert np.array_equal(got, want)
