"""The eddy viscosity at the edges of its tiles: 64 x cells with one or two cells
beside them (a last tile of 2 cells, of 8, an exact tile, less than one tile),
rows past the top, runs of z planes with a remainder and grids on which each
plane is a periodic neighbour of the others.  MTS uses correctly rounded
operations only and equals the oracle bit for bit; WALE's powers are square roots
on the device and pow on the host, a few ulp each, so 1e-14 of the maximum."""
import numpy as np
import pytest

from tests import cases
from tests.test_gpu_parity import make_pair, random_state, relerr

pytestmark = pytest.mark.gpu

GRIDS = [(450, 9, 8), (72, 21, 27), (64, 8, 4), (8, 7, 5), (128, 18, 45)]


@pytest.fixture(scope="module")
def O(oracle_mod):
    return oracle_mod


@pytest.mark.parametrize("grid", GRIDS, ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("les_type", [2, 3], ids=["wale", "mts"])
def test_sgs_tiles(O, grid, les_type):
    from channel3d_amd import lib as L
    nx, ny, nz = grid
    o, g = make_pair(O, dict(cases.SMALL, nxc=nx, nyc=ny, nzc=nz, les_type=les_type,
                             filter_type=1), laminar=False)
    random_state(O, o, g, seed=ny)
    o.call("Clc_SGS_Vis", o.field(O.UX), o.field(O.UY), o.field(O.UZ), o.field(O.NUT))
    g.Clc_SGS_Vis(L.UX, L.UY, L.UZ, L.NUT)
    sl = (slice(1, nx + 1), slice(0, ny + 2), slice(1, nz + 1))
    err = relerr(g.download(L.NUT)[sl], o.field(O.NUT)[sl])
    assert err == 0.0 if les_type == 3 else err < 1e-14, err
    g.close()
    o.close()
