"""The planned boundary kernel of the fused paths (ghosts and increments of every record in one launch, transverse
neighbours on block edges taken from the interior) against the oracle, bit for bit: faces of every type side by side, so
that the edge neighbours of viscous connection and symmetry records lie behind each other kind of face, on boxes that
leave workgroups partly filled and on boxes of one cell in a direction."""
import numpy as np
import pytest

import mosegpu
from mosegpu import cases
from mosegpu.core import BC_EXTRAPOLATION, BC_NONE, BC_SYMMETRY, BC_WALL_ADIABATIC, BC_WALL_ISOTHERMAL
from oracle_bind import OracleCase
from test_gpu_walls_sa import run_device

pytestmark = pytest.mark.gpu

PER, SYM, WA, WI, EX, NO = "periodic", BC_SYMMETRY, BC_WALL_ADIABATIC, BC_WALL_ISOTHERMAL, BC_EXTRAPOLATION, BC_NONE
FACES = {
    "periodic": (PER, PER, PER, PER, PER, PER),
    "periodic-symmetry-wall": (PER, PER, SYM, SYM, WA, WI),
    "symmetry-extrapolation": (SYM, EX, PER, PER, EX, SYM),
    "wall-symmetry-none": (WI, WA, SYM, EX, NO, NO),
}


def seeded(dims, faces, viscous, limiter="vanalbada", riemann="HLLC"):
    case = cases.box_case(dims, dict(zip(range(1, 7), faces)), extent=(1.0, 0.8, 0.9), viscous=viscous,
                          mu_of_T=cases.sutherland(2e-3, 300.0) if viscous else None, riemann=riemann, limiter=limiter,
                          ndir=sum(d > 1 for d in dims))
    rng = np.random.Generator(np.random.PCG64(17))
    V = case.layout.interior(case.P, 0)
    V[0] = 1.1 + 0.1 * rng.uniform(-1, 1, V[0].shape)
    for q in range(3):
        V[1 + q] = 20.0 * rng.uniform(-1, 1, V[0].shape)
    V[4] = 1e5 * (1.0 + 0.05 * rng.uniform(-1, 1, V[0].shape))
    cases.fill_ghosts_nearest(case.layout, case.P)
    return case


@pytest.mark.parametrize("viscous", [False, True], ids=["euler", "viscous"])
@pytest.mark.parametrize("dims", [(3, 3, 3), (5, 4, 7), (17, 9, 6)])
@pytest.mark.parametrize("name", list(FACES))
def test_faces_side_by_side(gpu_ready, name, dims, viscous):
    case = seeded(dims, FACES[name], viscous)
    print(f"boundary plan: {name} {dims} viscous {viscous}", flush=True)
    Pg, rep, _ = run_device(case, 3, mosegpu.PATH_FUSED, (8, 4, 4))
    Po = case.P.copy()
    OracleCase(case).step(Po, 3)
    assert np.array_equal(case.layout.interior(Pg, 0), case.layout.interior(Po, 0))


@pytest.mark.parametrize("viscous", [False, True], ids=["euler", "viscous"])
@pytest.mark.parametrize("dims,faces", [((9, 7, 1), (PER, PER, WA, EX, NO, NO)), ((9, 7, 1), (SYM, EX, PER, PER, EX, EX)),
                                        ((11, 1, 1), (EX, EX, NO, NO, NO, NO))])
def test_one_cell_directions(gpu_ready, dims, faces, viscous):
    case = seeded(dims, faces, viscous)
    print(f"boundary plan: {dims} faces {faces} viscous {viscous}", flush=True)
    Pg, rep, _ = run_device(case, 3, mosegpu.PATH_FUSED)
    Po = case.P.copy()
    OracleCase(case).step(Po, 3)
    assert np.array_equal(case.layout.interior(Pg, 0), case.layout.interior(Po, 0))
    if faces[4] == NO:      # ghosts behind no-flux faces: the cell's values, whenever they were filled
        v = case.layout.block_view(Pg, 0)
        assert np.all(np.isfinite(v[:, 0, 2:-2, 2:-2]))
        if not viscous:
            for g in (0, 1, 3, 4):
                assert np.array_equal(v[:, g, 2:-2, 2:-2], v[:, 2, 2:-2, 2:-2])
