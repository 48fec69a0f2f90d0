"""The 4th-order and LES right-hand sides at the edges of their tiles, bit for bit
against the oracle: 64 x cells per wavefront with the cells beside them (a
last tile of 2 cells, of 8, an exact tile, less than one tile), four rows
per workgroup (one, two or three of them past the top), runs of z planes with remainders and with every plane a periodic neighbour of the others."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_parity4 import interior4, make_pair, random_state

pytestmark = pytest.mark.gpu

GRIDS = [(450, 9, 8), (72, 21, 27), (64, 8, 4), (8, 7, 5), (128, 18, 45)]


@pytest.fixture(scope="module")
def O(oracle_mod):
    return oracle_mod


@pytest.mark.parametrize("grid", GRIDS, ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("half", [False, True], ids=["channel", "half"])
def test_rhs4_tiles_bitwise(O, grid, half):
    from channel3d_amd import lib as L
    nx, ny, nz = grid
    base = cases.HALF4 if half else cases.SMALL4
    o, g = make_pair(O, dict(base, nxc=nx, nyc=ny, nzc=nz, u_crf=0.3))
    random_state(O, o, g, seed=nx)
    o.call("PMcoeUpdate", 2)
    g.PMcoeUpdate(2)
    rz = np.zeros((nx + 4, ny + 2, nz + 4), order="F")
    o.call("clcRhsXYZ", o.field(O.UX), o.field(O.UY), o.field(O.UZ), o.field(O.ARR1),
           o.field(O.ARR2), rz, o.field(O.HISTX), o.field(O.HISTY), o.field(O.HISTZ),
           o.field(O.PR))
    g.clcRhsXYZ(L.UX, L.UY, L.UZ, L.ARR1, L.ARR2, L.HALOARR, L.HISTX, L.HISTY, L.HISTZ, L.PR)
    for fid, gid in ((O.ARR1, L.ARR1), (O.ARR2, L.ARR2), (O.HISTX, L.HISTX), (O.HISTY, L.HISTY),
                     (O.HISTZ, L.HISTZ)):
        assert np.abs(g.download(gid) - o.field(fid)).max() == 0.0, fid
    assert np.abs(interior4(g.download(L.HALOARR)) - interior4(rz)).max() == 0.0
    assert g.diagnostics()["PrGradNow"] == o.scalar(O.S_PRGRADNOW)
    g.close()
    o.close()


@pytest.mark.parametrize("grid", GRIDS, ids=lambda v: "x".join(map(str, v)))
def test_rhs_les_tiles_bitwise(O, grid):
    from channel3d_amd import lib as L
    from tests import test_gpu_parity as P2
    nx, ny, nz = grid
    o, g = P2.make_pair(O, dict(cases.SMALL, nxc=nx, nyc=ny, nzc=nz, les_type=3, filter_type=1),
                        laminar=False)
    P2.random_state(O, o, g, seed=ny)
    u = (o.field(O.UX), o.field(O.UY), o.field(O.UZ))
    nut = o.field(O.NUT)
    o.call("Clc_SGS_Vis", *u, nut)
    g.upload(L.NUT, nut)
    o.call("PMcoeUpdate", 2)
    g.PMcoeUpdate(2)
    rx, ry = (np.zeros((nx, ny, nz), order="F") for _ in range(2))
    rz = np.zeros((nx + 3, ny + 3, nz + 3), order="F")
    o.call("clcRhsX_les", *u, rx, o.field(O.HISTX), o.field(O.PR), nut)
    o.call("clcRhsY_les", *u, ry, o.field(O.HISTY), o.field(O.PR), nut)
    o.call("clcRhsZ_les", *u, rz, o.field(O.HISTZ), o.field(O.PR), nut)
    g.clcRhsX(L.UX, L.UY, L.UZ, L.ARR1, L.HISTX, L.PR)
    g.clcRhsY(L.UX, L.UY, L.UZ, L.ARR2, L.HISTY, L.PR)
    g.clcRhsZ(L.UX, L.UY, L.UZ, L.HALOARR, L.HISTZ, L.PR)
    for gid, ref in ((L.ARR1, rx), (L.ARR2, ry), (L.HALOARR, rz), (L.HISTX, o.field(O.HISTX)),
                     (L.HISTY, o.field(O.HISTY)), (L.HISTZ, o.field(O.HISTZ))):
        got = g.download(gid)
        if gid == L.HALOARR:
            got, ref = P2.interior(got), P2.interior(ref)
        assert np.abs(got - ref).max() == 0.0, gid
    g.close()
    o.close()
