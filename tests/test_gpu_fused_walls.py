"""The substep's walls inside its kernels: with moving and blowing walls, no-slip
and free-slip, the fused substeps (wall rows of uy taken by the pressure source,
ghosts written by the projection, the flow-rate and divergence reductions in
slots) equal the routines called one at a time, ghost rows included.  The same
operations on the same operands: bit for bit, in FP64 and in FP32.  Row counts
below, at and above a workgroup's four rows; both kernel variants (C3D_NT).  A
second set of grids runs over the edges of the 64-cell tiles, the segments of the
sweeps and the z runs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BASE = dict(xlx=4.0, yly=2.0, zlz=2.0, xnu=1 / 500.0, dt=0.004, gamma=1.3,
            ubulk=1.0, uxbc=(0, 0, 0.2, -0.1, 0, 0), uzbc=(0, 0, -0.05, 0.3, 0, 0))
KINDS = {
    "channel": dict(uybc=(0, 0, 0.02, 0.02, 0, 0)),
    "freeslip": dict(bc=(0, 0, -1, -2, 0, 0)),
    "bottom_freeslip": dict(bc=(0, 0, -2, -1, 0, 0)),
    "les": dict(les_type=2, filter_type=1, uybc=(0, 0, 0.01, 0.01, 0, 0)),
    "mts": dict(les_type=3, filter_type=0, bc=(0, 0, -1, -2, 0, 0)),
    "fourth": dict(order=4),
    "half": dict(order=4, bc=(0, 0, -1, -2, 0, 0)),
}


def _routines(g, ns, order, les):
    from channel3d_amd import lib as L
    u, p = (L.UX, L.UY, L.UZ), L.PR
    g.PMcoeUpdate(ns)
    g.Update_uy_ym()
    if order == 4:
        g.clcRhsXYZ(*u, L.ARR1, L.ARR2, L.HALOARR, L.HISTX, L.HISTY, L.HISTZ, p)
    else:
        g.clcRhsX(*u, L.ARR1, L.HISTX, p)
        g.clcRhsY(*u, L.ARR2, L.HISTY, p)
        g.clcRhsZ(*u, L.HALOARR, L.HISTZ, p)
    g.clcU1Hat(L.UX, L.ARR1)
    g.clcU2Hat(L.UY, L.ARR2, L.DUY_YM)
    g.clcU3Hat(L.UZ, L.HALOARR)
    g.SetBC_and_UpdateHaloForPrSrc(*u, L.UY_YM)
    div = g.clcPrSrc(*u, L.ARR1, None if order == 4 else p)
    g.clcPPE(L.ARR1, L.HALOARR)
    g.SetBC_and_UpdateHalo_pr(L.HALOARR)
    g.FluidVelUpdate(L.HALOARR, *u)
    g.PressureUpdate(p, L.HALOARR)
    g.SetBC_and_UpdateHalo(*u, L.UY_YM)
    g.SetBC_and_UpdateHalo_pr(p)
    return div


def _check(kind, nx, ny, nz, fp32):
    from channel3d_amd import Channel, lib as L
    case = dict(BASE, nxc=nx, nyc=ny, nzc=nz, **KINDS[kind])
    les = "les_type" in case
    out = []
    for fused in (False, True):
        with Channel(case, precision=L.FP32 if fp32 else L.FP64) as g:
            rng = np.random.default_rng(ny)
            h = 2 if g.order == 4 else 1
            for f in (L.UX, L.UY, L.UZ):
                a = np.zeros(g.shape(L.HALO), order="F")
                a[h:h + nx, 1:ny + 1, h:h + nz] = rng.uniform(-0.2, 1.0, (nx, ny, nz))
                g.upload(f, a)
            g.project()
            if les:
                g.Clc_SGS_Vis()
            divs = []
            for ns in (1, 2, 3):
                if fused:
                    g.substep(ns)
                    divs.append(g.diagnostics()["divmax1"])
                else:
                    divs.append(_routines(g, ns, g.order, les))
            d = g.diagnostics()
            out.append(([g.download(f) for f in (L.UX, L.UY, L.UZ, L.PR, L.HISTX, L.HISTY,
                                                 L.HISTZ)], divs,
                        (d["PrGradNow"], d["PrGradAver"])))
    for a, b in zip(out[0][0], out[1][0]):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)
    assert out[0][1] == out[1][1]
    assert out[0][2] == out[1][2]


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("ny", [3, 8, 13])
@pytest.mark.parametrize("nt", ["0", "1"])
@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
def test_fused_equals_routines(monkeypatch, kind, ny, nt, fp32):
    monkeypatch.setenv("C3D_NT", nt)
    _check(kind, 24, ny, 20, fp32)


# (nx, ny, nz): a last tile of 2 x cells, of 8, an exact tile, less than one tile
GRIDS = [(450, 9, 8), (72, 21, 27), (64, 8, 4), (8, 7, 5), (128, 18, 45)]


@pytest.mark.parametrize("grid", GRIDS, ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("kind", ["channel", "les", "mts", "fourth"])
@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
def test_fused_tile_edges(kind, grid, fp32):
    _check(kind, *grid, fp32)


@pytest.mark.parametrize("kind", ["channel", "freeslip", "les"])
@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
def test_fused_source_pass(monkeypatch, kind, fp32):
    """the same where the x length has a run-time transform plan and the source
    is a pass of its own"""
    monkeypatch.setenv("C3D_FFT_PLAN", "runtime")
    for ny, nt in ((13, "0"), (5, "1")):
        monkeypatch.setenv("C3D_NT", nt)
        _check(kind, 24, ny, 20, fp32)
