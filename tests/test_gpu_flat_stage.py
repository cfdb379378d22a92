"""The stage kernel of blocks one cell thick in k (inviscid, one species) against the oracle: rows and planes that leave
tiles partly filled, every limiter and solver, both workgroup forms (a thread per face while all tiles are resident, a
thread per cell beyond), the default tile, and tiles that the general kernels take instead (a tile across the one-cell
direction)."""
import numpy as np
import pytest

import mosegpu
from mosegpu.core import BC_EXTRAPOLATION, BC_NONE, BC_SYMMETRY, BC_WALL_ADIABATIC
from oracle_bind import OracleCase
from test_gpu_boundary_plan import seeded
from test_gpu_walls_sa import run_device

pytestmark = pytest.mark.gpu

PER, SYM, WA, EX, NO = "periodic", BC_SYMMETRY, BC_WALL_ADIABATIC, BC_EXTRAPOLATION, BC_NONE
PLANE, ROW, BOX2 = (EX, SYM, WA, EX, NO, NO), (EX, EX, NO, NO, NO, NO), (PER, PER, PER, PER, EX, EX)


def agree(case, tile, steps, paths=(mosegpu.PATH_FUSED, mosegpu.PATH_FAST)):
    Po = case.P.copy()
    OracleCase(case).step(Po, steps)
    want = case.layout.interior(Po, 0)
    for path in paths:
        Pg, rep, _ = run_device(case, steps, path, tile)
        got = case.layout.interior(Pg, 0)
        if path == mosegpu.PATH_FUSED:
            assert np.array_equal(got, want)
        else:
            for q in range(5):
                scale = np.abs(want[1:4]).max() if 1 <= q <= 3 else np.abs(want[q]).max()
                assert np.abs(got[q] - want[q]).max() <= 1e-12 * scale


@pytest.mark.parametrize("dims,faces", [((17, 9, 1), PLANE), ((31, 33, 1), BOX2), ((3, 3, 1), PLANE), ((130, 5, 1), BOX2),
                                        ((3, 40, 1), PLANE), ((257, 1, 1), ROW), ((5, 1, 1), ROW), ((129, 1, 1), ROW)])
@pytest.mark.parametrize("tile", [(16, 8, 1), (32, 8, 1), (128, 1, 1), (256, 1, 1), (2, 64, 1), (1, 128, 1), (8, 8, 4)])
def test_tiles_and_edges(gpu_ready, dims, faces, tile):
    print(f"flat stage: {dims} tile {tile}", flush=True)
    # the performance path refuses 256 x 1 x 1 (the general kernel's LDS)
    paths = (mosegpu.PATH_FUSED,) if tile == (256, 1, 1) else (mosegpu.PATH_FUSED, mosegpu.PATH_FAST)
    agree(seeded(dims, faces, False), tile, 3, paths)


@pytest.mark.parametrize("riemann", ["HLLC", "HLLE", "SLAU", "AUSM+", "LMRoe"])
@pytest.mark.parametrize("limiter", ["minmod", "vanleer", "vanalbada", "mc", "superbee"])
@pytest.mark.parametrize("tile", [(16, 8, 1), (16, 16, 1)])
def test_limiters_and_solvers(gpu_ready, tile, limiter, riemann):
    print(f"flat stage: {limiter} {riemann} tile {tile}", flush=True)
    paths = (mosegpu.PATH_FUSED,) if riemann == "SLAU" else (mosegpu.PATH_FUSED, mosegpu.PATH_FAST)
    agree(seeded((21, 18, 1), PLANE, False, limiter, riemann), tile, 2, paths)


@pytest.mark.parametrize("dims,faces,tile", [((321, 320, 1), BOX2, (16, 8, 1)), ((98500, 1, 1), ROW, (128, 1, 1))])
def test_more_tiles_than_resident(gpu_ready, dims, faces, tile):
    print(f"flat stage: {dims} tile {tile}", flush=True)
    agree(seeded(dims, faces, False), tile, 1)
