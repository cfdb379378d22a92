"""Symmetry and connection faces of a direction of one cell, where a record's neighbour along the normal is the ghost
behind the opposite face: the fused paths against the oracle (the parity path bit for bit), as a plane closed by two
symmetry faces, a wedge whose faces are tilted, mixed pairs, and a block one cell thick between two others.  Every
uploaded ghost row holds NaN: a stage that reads a ghost before its record has filled it does not stay finite."""
import numpy as np
import pytest

import mosegpu
from mosegpu import cases
from mosegpu.cases import Case, block_records, box_nodes, make_scheme
from mosegpu.core import (BC_CONNECTION, BC_EXTRAPOLATION, BC_NONE, BC_SYMMETRY, BC_WALL_ADIABATIC, Layout,
                          metrics_build, records_tangent)
from oracle_bind import OracleCase
from test_gpu_walls_sa import run_device

pytestmark = pytest.mark.gpu

PER, SYM, WA, EX, NO = "periodic", BC_SYMMETRY, BC_WALL_ADIABATIC, BC_EXTRAPOLATION, BC_NONE


def seed_state(case):
    """Density, three velocity components and pressure of every cell from a seed, NaN in every ghost row."""
    case.P[...] = np.nan
    rng = np.random.Generator(np.random.PCG64(23))
    for b in range(case.layout.nb):
        V = case.layout.interior(case.P, b)
        V[0] = 1.1 + 0.1 * rng.uniform(-1, 1, V[0].shape)
        for q in range(3):
            V[1 + q] = 20.0 * rng.uniform(-1, 1, V[0].shape)
        V[4] = 1e5 * (1.0 + 0.05 * rng.uniform(-1, 1, V[0].shape))
    return case


def sutherland_if(viscous):
    return cases.sutherland(2e-3, 300.0) if viscous else None


def agree(case, tile, steps=3):
    Po = case.P.copy()
    OracleCase(case).step(Po, steps)
    for path in (mosegpu.PATH_FUSED, mosegpu.PATH_FAST):
        Pg, rep, _ = run_device(case, steps, path, tile)
        for b in range(case.layout.nb):
            got, want = case.layout.interior(Pg, b), case.layout.interior(Po, b)
            assert np.all(np.isfinite(want))
            if path == mosegpu.PATH_FUSED:
                assert np.array_equal(got, want)
                continue
            for q in range(5):
                scale = np.abs(want[1:4]).max() if 1 <= q <= 3 else np.abs(want[q]).max()
                assert np.abs(got[q] - want[q]).max() <= 1e-12 * scale


@pytest.mark.parametrize("limiter", ["minmod", "vanalbada"])
@pytest.mark.parametrize("viscous", [False, True], ids=["euler", "viscous"])
@pytest.mark.parametrize("k", [(SYM, SYM), (SYM, NO), (NO, SYM)], ids=["sym-sym", "sym-none", "none-sym"])
@pytest.mark.parametrize("shape", ["box", "wedge"])
def test_plane_closed_by_symmetry(gpu_ready, shape, k, viscous, limiter):
    dims = (9, 7, 1)
    nodes = None
    if shape == "wedge":      # the thickness grows with y, so neither face's normal is an axis
        nodes = box_nodes(*dims, (0.0, 0.0, 0.0), (1.0, 0.8, 1.0))
        nodes[..., 2] = (nodes[..., 2] - 0.4) * (0.2 + 0.3 * nodes[..., 1])
    case = cases.box_case(dims, dict(zip(range(1, 7), (PER, PER, WA, EX) + k)), extent=(1.0, 0.8, 0.9), viscous=viscous,
                          mu_of_T=sutherland_if(viscous), nodes=nodes, limiter=limiter, ndir=2)
    print(f"one-cell faces: {shape} {k} viscous {viscous} {limiter}", flush=True)
    agree(seed_state(case), (8, 8, 4) if viscous else (16, 8, 1))


@pytest.mark.parametrize("viscous", [False, True], ids=["euler", "viscous"])
def test_row_closed_by_symmetry(gpu_ready, viscous):
    case = cases.box_case((11, 1, 1), dict(zip(range(1, 7), (EX, SYM, SYM, SYM, SYM, SYM))), extent=(1.0, 0.1, 0.1),
                          viscous=viscous, mu_of_T=sutherland_if(viscous), limiter="vanalbada", ndir=1)
    print(f"one-cell faces: row viscous {viscous}", flush=True)
    agree(seed_state(case), (8, 4, 4) if viscous else (128, 1, 1))


@pytest.mark.parametrize("middle", ["between", "end"])
@pytest.mark.parametrize("viscous", [False, True], ids=["euler", "viscous"])
def test_block_one_cell_thick_receives(gpu_ready, viscous, middle):
    """Block 0 is one cell thick along i: between blocks 1 and 2 (a receiver on both sides), or at the end of block 1
    with a symmetry face behind it.  Its neighbours close on their other side (block 0 cannot be a donor)."""
    both = middle == "between"
    dims = [(1, 5, 4), (4, 5, 4)] + ([(3, 5, 4)] if both else [])
    ext = [(0.25, 0.8, 0.6), (1.0, 0.8, 0.6), (0.9, 0.8, 0.6)]
    lo = [(1.0, 0.0, 0.0), (0.0, 0.0, 0.0), (1.25, 0.0, 0.0)]
    nodes = [box_nodes(*d, o, tuple(a + e for a, e in zip(o, x))) for d, o, x in zip(dims, lo, ext)]
    side = {3: SYM, 4: EX, 5: NO, 6: EX}
    to = {1: (1, 2, lambda i, j, k: (np.full_like(i, 4), j, k), False),
          2: (2, 1, lambda i, j, k: (np.full_like(i, 1), j, k), False)}
    recs = [block_records(0, dims[0], {1: BC_CONNECTION, 2: BC_CONNECTION if both else SYM, **side}, to),
            block_records(1, dims[1], {1: EX, 2: SYM, **side})]
    if both:
        recs.append(block_records(2, dims[2], {1: SYM, 2: EX, **side}))
    rec = np.ascontiguousarray(np.concatenate(recs))
    layout = Layout(dims)
    records_tangent(layout, nodes, rec)
    geom = metrics_build(layout, nodes, rec, ndir=3)
    tables = cases.air_tables(sutherland_if(viscous), prandtl=0.72)
    sch = make_scheme(limiter="vanalbada", riemann="HLLC", viscous=viscous, ndir=3, prandtl=0.72 if viscous else 0.0)
    case = Case("thin", tables, sch, layout, nodes, rec, geom, np.zeros((5, layout.NC)), 3)
    print(f"one-cell faces: thin block, {middle}, viscous {viscous}", flush=True)
    agree(seed_state(case), (8, 4, 4))
