"""FP32 contexts' routines against FP64 contexts' on the same (FP32) inputs, at the
edges of the tiles, segments and z runs: right-hand sides, wall-normal solves, eddy
viscosity, source, projection and pressure update of every scheme.

Bound: a result takes fewer than 64 FP32 roundings, each at most 2^-24 of the
largest value (random inputs of one size: no partial sum is larger than that by
more than what the roundings cancel).  The eddy viscosity raises its
invariants to powers up to 5/2 after removing their trace: another factor 4.  A cell that read
a wrong neighbour would be off by the order of its own value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOUND = 64 * 2.0 ** -24
GRIDS = [(450, 9, 8), (72, 21, 27), (64, 8, 4), (8, 7, 5), (128, 18, 45)]
BASE = dict(xlx=4.0, yly=2.0, zlz=2.0, xnu=1 / 500.0, dt=0.004, gamma=1.3, ubulk=1.0,
            uxbc=(0, 0, 0.25, -0.125, 0, 0))
KINDS = {"channel": {}, "wale": dict(les_type=2), "mts": dict(les_type=3, filter_type=0),
         "fourth": dict(order=4), "half": dict(order=4, bc=(0, 0, -1, -2, 0, 0))}


def _run(case, prec, grid):
    from channel3d_amd import Channel, lib as L
    nx, ny, nz = grid
    out = {}
    with Channel(case, precision=prec) as g:
        rng = np.random.default_rng(nx + ny)
        h = 2 if g.order == 4 else 1
        cut = (slice(h, h + nx), slice(0, ny + 2), slice(h, h + nz))

        def halo():
            a = np.zeros(g.shape(L.HALO), order="F")
            a[cut] = rng.uniform(-1, 1, (nx, ny + 2, nz)).astype(np.float32)
            return a

        def inner(scale=1.0):
            return np.asfortranarray(scale * rng.uniform(-1, 1, (nx, ny, nz)).astype(np.float32))

        def take(name, f):
            a = g.download(f)
            out[name] = a if a.shape == (nx, ny, nz) else a[cut][:, 1:ny + 1]

        u, p = (L.UX, L.UY, L.UZ), L.PR
        for f in u + (p,):
            g.upload(f, halo())
        for f in (L.HISTX, L.HISTY, L.HISTZ):
            g.upload(f, inner())
        if "les_type" in case:
            g.Clc_SGS_Vis()
            out["nut"] = g.download(L.NUT)[cut]
        g.PMcoeUpdate(2)
        g.Update_uy_ym()
        if g.order == 4:
            g.clcRhsXYZ(*u, L.ARR1, L.ARR2, L.HALOARR, L.HISTX, L.HISTY, L.HISTZ, p)
        else:
            g.clcRhsX(*u, L.ARR1, L.HISTX, p)
            g.clcRhsY(*u, L.ARR2, L.HISTY, p)
            g.clcRhsZ(*u, L.HALOARR, L.HISTZ, p)
        for name, f in (("rx", L.ARR1), ("ry", L.ARR2), ("rz", L.HALOARR), ("hx", L.HISTX),
                        ("hy", L.HISTY), ("hz", L.HISTZ)):
            take(name, f)
        for f in (L.ARR1, L.ARR2):
            g.upload(f, inner(0.125))
        g.upload(L.HALOARR, halo())
        g.clcU1Hat(L.UX, L.ARR1)
        g.clcU2Hat(L.UY, L.ARR2, L.DUY_YM)
        g.clcU3Hat(L.UZ, L.HALOARR)
        for name, f in zip(("u1", "u2", "u3"), u):
            take(name, f)
        for f in u:
            g.upload(f, halo())
        g.SetBC_and_UpdateHaloForPrSrc(*u, L.UY_YM)
        out["div"] = np.array([g.clcPrSrc(*u, L.ARR1, None if g.order == 4 else p)])
        take("src", L.ARR1)
        g.upload(L.HALOARR, halo())
        g.SetBC_and_UpdateHalo_pr(L.HALOARR)
        g.FluidVelUpdate(L.HALOARR, *u)
        g.PressureUpdate(p, L.HALOARR)
        g.SetBC_and_UpdateHalo(*u, L.UY_YM)
        g.SetBC_and_UpdateHalo_pr(p)
        for name, f in zip(("v1", "v2", "v3", "p"), u + (p,)):
            out[name] = g.download(f)[cut]
    return out


@pytest.mark.parametrize("grid", GRIDS, ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("kind", list(KINDS))
def test_fp32_routines(kind, grid):
    from channel3d_amd import lib as L
    case = dict(BASE, nxc=grid[0], nyc=grid[1], nzc=grid[2], **KINDS[kind])
    a, b = _run(case, L.FP64, grid), _run(case, L.FP32, grid)
    err = {k: np.abs(a[k] - b[k]).max() / np.abs(a[k]).max() for k in a}
    print({k: "%.1e" % v for k, v in err.items()})
    assert all(np.isfinite(v).all() for v in b.values())
    bad = {k: v for k, v in err.items() if not v <= BOUND * (4 if k == "nut" else 1)}
    assert not bad, bad
