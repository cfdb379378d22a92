"""The tile that serving gives a case, without a GPU: it fits the LDS of a workgroup for every species count, viscosity,
dimension and path, and where the plane kernel does not run it is never the plane kernel's larger tile."""
from types import SimpleNamespace

import pytest

from mosegpu import PATH_FAST, PATH_FUSED, PATH_PLAIN, cases, serve

LDS = 160 * 1024      # a gfx950 workgroup's


def case(dims, nsc=1, nrans=0, viscous=False):
    return SimpleNamespace(layout=SimpleNamespace(dims=[dims]),
                           scheme=cases.make_scheme(nsc=nsc, nrans=nrans, viscous=viscous))


@pytest.mark.parametrize("path", [PATH_FUSED, PATH_FAST])
@pytest.mark.parametrize("nsc,nrans,viscous", [(1, 0, False), (1, 0, True), (1, 1, True), (4, 0, False), (4, 0, True),
                                               (9, 0, False), (9, 0, True)])
@pytest.mark.parametrize("dims", [(5, 1, 1), (1000, 1, 1), (200000, 1, 1), (64, 64, 1), (313, 314, 1), (1024, 1024, 1),
                                  (9, 8, 7), (256, 256, 256)])
def test_tile_fits(dims, nsc, nrans, viscous, path):
    c = case(dims, nsc, nrans, viscous)
    t = serve.serve_tile(c, path)
    assert t[0] * t[1] * t[2] in (128, 256)
    assert serve.tile_lds(c, path, t) <= LDS
    if nsc == 9 and viscous:
        assert t[0] * t[1] * t[2] == 128      # larger ones are refused
    if nsc > 1 or viscous:
        assert t != (32, 8, 1)


def test_plane_kernel_tiles():
    """32 x 8 x 1 once 16 x 8 x 1 tiles are more than three workgroups per compute unit."""
    assert serve.serve_tile(case((1024, 1024, 1)), PATH_FAST) == (32, 8, 1)
    assert serve.serve_tile(case((256, 256, 1)), PATH_FAST) == (16, 8, 1)
    assert serve.serve_tile(case((256, 256, 1)), PATH_FAST, cus=64) == (32, 8, 1)
    assert serve.serve_tile(case((48, 48, 48), viscous=True), PATH_FAST) == (8, 8, 4)
    assert serve.serve_tile(case((48, 48, 48), viscous=True), PATH_PLAIN) == (0, 0, 0)


def test_refused_tiles_by_their_bytes():
    """The tiles that the rule gave these cases before do not fit: 256 x 1 x 1 for viscous rows, 32 x 8 x 1 for planes of
    four and nine species, 128 x 1 x 1 for rows of nine on the performance path."""
    for c, path, t in ((case((1000, 1, 1), viscous=True), PATH_FUSED, (256, 1, 1)),
                       (case((1000, 1, 1), viscous=True), PATH_FAST, (256, 1, 1)),
                       (case((1024, 1024, 1), nsc=4), PATH_FAST, (32, 8, 1)),
                       (case((1024, 1024, 1), nsc=9), PATH_FUSED, (32, 8, 1)),
                       (case((1000, 1, 1), nsc=9), PATH_FAST, (128, 1, 1))):
        assert serve.tile_lds(c, path, t) > LDS
        assert serve.serve_tile(c, path) != t
