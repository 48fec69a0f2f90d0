"""The LES wall-normal solves at the edges of their segments (8 rows: one row,
one segment, a row more, two and three segments and a remainder) and of their
64-line workgroups, bit for bit against the oracle.  Divisions by a shared
reciprocal round like divisions, so the comparison stays exact."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_parity import interior, make_pair, periodic_fill, random_state

pytestmark = pytest.mark.gpu

GRIDS = [(16, 3, 8), (18, 8, 9), (10, 9, 12), (16, 16, 8), (20, 17, 15), (36, 31, 10)]


@pytest.fixture(scope="module")
def O(oracle_mod):
    return oracle_mod


@pytest.mark.parametrize("grid", GRIDS, ids=lambda v: "x".join(map(str, v)))
def test_les_solves_bitwise(O, grid):
    from channel3d_amd import lib as L, synth
    nx, ny, nz = grid
    o, g = make_pair(O, dict(cases.SMALL, nxc=nx, nyc=ny, nzc=nz, les_type=3, filter_type=1),
                     laminar=False)
    random_state(O, o, g, seed=ny)
    nut = o.field(O.NUT)
    o.call("Clc_SGS_Vis", o.field(O.UX), o.field(O.UY), o.field(O.UZ), nut)
    g.upload(L.NUT, nut)
    o.call("PMcoeUpdate", 2)
    g.PMcoeUpdate(2)
    r = [synth.random_interior(nx, ny, nz, 5, 1 + q, 0.01) for q in range(2)]
    r.append(periodic_fill(synth.random_halo(nx, ny, nz, 5, 3, 0.01)))
    duy = synth.uniform_pm1(5, 4, (nx, nz)) * 1e-3
    for gid, a in ((L.ARR1, r[0]), (L.ARR2, r[1]), (L.HALOARR, r[2]), (L.DUY_YM, duy)):
        g.upload(gid, a)
    o.call("clcU1Hat_les", o.field(O.UX), np.asfortranarray(r[0].copy()), nut)
    o.call("clcU2Hat_les", o.field(O.UY), np.asfortranarray(r[1].copy()), np.asfortranarray(duy),
           nut)
    o.call("clcU3Hat_les", o.field(O.UZ), np.asfortranarray(r[2].copy()), nut)
    g.clcU1Hat(L.UX, L.ARR1)
    g.clcU2Hat(L.UY, L.ARR2, L.DUY_YM)
    g.clcU3Hat(L.UZ, L.HALOARR)
    for fid, gid in ((O.UX, L.UX), (O.UY, L.UY), (O.UZ, L.UZ)):
        assert np.abs(interior(g.download(gid)) - interior(o.field(fid))).max() == 0.0
    g.close()
    o.close()
