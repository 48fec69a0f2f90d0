"""The run-time transform plan at its edges, pressure solves at 1e-12 against the
oracle: lengths of a single pass, a partial last tile of lines, three and four
butterflies per thread (lengths 2 m and 3 m with full tiles), one line per
workgroup, and the longest line but one factor."""
import numpy as np
import pytest

from tests.test_gpu_parity import interior, make_pair, relerr

pytestmark = pytest.mark.gpu

BASE = dict(xlx=3.0, yly=2.0, zlz=1.0, xnu=1.0 / 1500.0, dt=0.004, gamma=1.3, ubulk=1.0)
# (nx, ny, nz): transforms of nx / 2 and nz
GRIDS = [(16, 5, 8), (10, 7, 9), (30, 5, 25), (300, 9, 150), (108, 6, 450), (486, 5, 270),
         (4050, 4, 10), (20, 4, 2430), (7680, 4, 6)]


@pytest.fixture(scope="module")
def O(oracle_mod):
    return oracle_mod


@pytest.mark.parametrize("grid", GRIDS, ids=lambda v: "x".join(map(str, v)))
def test_ppe_lengths(O, grid, monkeypatch):
    from channel3d_amd import lib as L, synth
    monkeypatch.setenv("C3D_FFT_PLAN", "runtime")
    nx, ny, nz = grid
    o, g = make_pair(O, dict(BASE, nxc=nx, nyc=ny, nzc=nz), laminar=False)
    f = synth.ppe_rhs(nx, ny, nz, seed=nx)
    ph = np.zeros((nx + 3, ny + 3, nz + 3), order="F")
    o.call("clcPPE", np.asfortranarray(f.copy()), ph)
    g.upload(L.ARR1, f)
    g.clcPPE(L.ARR1, L.HALOARR)
    assert relerr(interior(g.download(L.HALOARR)), interior(ph)) < 1e-12
    g.close()
    o.close()
