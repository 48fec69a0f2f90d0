"""The FP64 residual passes of the refined solves at the edges of their tiles:
64 x cells per wavefront (a last tile of 2 cells, one exact tile, less than a
tile), blocks of 4 and 8 rows in workgroups of 16 and 32, z chunks with
remainders.  A cell whose residual is wrong keeps the FP32 solve's error, so
the refined solution must approach the FP64 solve of the same source (which
the oracle tests cover) everywhere.  Bounds: a sweep multiplies the error by at
most the FP32 solve's relative error, FP32's eps times the condition number of
the operator: for the pressure's worst line, the y operator's largest entry
(about ny^2) over the smallest non-zero wavenumber term (1 in these boxes; the
mean mode's line is solved in FP64 and has a test of its own); below 20 for the
velocity operator.  What remains is FP64 rounding (1e-12)."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(450, 33, 12), (128, 31, 50), (64, 32, 18), (72, 17, 25), (64, 16, 64)]


def _channel(nx, ny, nz):
    from channel3d_amd import Channel
    return Channel(dict(nxc=nx, nyc=ny, nzc=nz, xlx=2 * math.pi, yly=2.0, zlz=math.pi,
                        xnu=1.0e-4, dt=0.001, gamma=1.2, ubulk=1.0))


def _fields(g, nb, compatible):
    rng = np.random.default_rng(3)
    out = []
    for _ in range(nb):
        f = rng.standard_normal((g.nxc, g.nyc, g.nzc))
        if compatible:
            d = np.diff(np.asarray(g.yp[1:g.nyc + 2]))
            f -= (f.mean(axis=(0, 2)) * d).sum() / d.sum()
        out.append(np.asfortranarray(f))
    return out


# the (0, 0) mode's line moves through LDS 256 rows at a time: one row more, two chunks
# and a remainder
LONG = [(16, 257, 8), (16, 530, 8), (16, 256, 8)]


@pytest.mark.parametrize("grid", GRIDS + LONG, ids=lambda v: "x".join(map(str, v)))
def test_pressure_refinement(grid):
    from channel3d_amd import lib as L
    with _channel(*grid) as g:
        src, a, b0, b2 = (g.alloc_batch(lay, 2) for lay in (L.INTERIOR,) + (L.HALO,) * 3)
        for q, f in enumerate(_fields(g, 2, True)):
            g.upload(src[q], f, L.INTERIOR)
        for out, sweeps in ((a, -1), (b0, 0), (b2, 2)):
            g.ppe_batch(src, out, sweeps)
        n = slice(1, g.nyc + 1)
        rate = min(0.1, np.finfo(np.float32).eps * g.nyc ** 2)
        for q in range(2):
            x, y0, y2 = (g.download(h[q], L.HALO)[1:-2, n, 1:-2] for h in (a, b0, b2))
            e0, e2 = (np.abs(x - y).max() / np.abs(x).max() for y in (y0, y2))
            assert e0 <= rate
            assert e2 <= rate ** 2 * e0 + 1e-12


@pytest.mark.parametrize("grid", LONG + [(16, 3, 8), (64, 33, 16)],
                         ids=lambda v: "x".join(map(str, v)))
def test_mean_mode(grid):
    """The (0, 0) mode alone: a source that depends on y only, small integers, so that
    the FP32 transforms (lengths of powers of two) are exact.  Its line is solved in
    FP64 and rounded to FP32 once: 2^-24 of the largest value, where an FP32
    elimination would lose eps ny^2; a sweep squares that.  Besides, FP64 rounding of
    the line, whose condition number is about ny^2."""
    from channel3d_amd import lib as L
    nx, ny, nz = grid
    with _channel(*grid) as g:
        src, a, b = (g.alloc_batch(lay, 2) for lay in (L.INTERIOR,) + (L.HALO,) * 2)
        rng = np.random.default_rng(ny)
        for q in range(2):
            f = rng.integers(-1000, 1000, ny).astype(float)
            g.upload(src[q], np.broadcast_to(f[None, :, None], grid), L.INTERIOR)
        g.ppe_batch(src, a, -1)
        rounding = np.finfo(float).eps * ny ** 2
        for sweeps, once in ((0, 2.0 ** -24), (1, 2.0 ** -48), (2, 0.0)):
            g.ppe_batch(src, b, sweeps)
            for q in range(2):
                x, y = (g.download(h[q], L.HALO)[1:-2, 1:ny + 1, 1:-2] for h in (a, b))
                assert np.abs(x).max() > 0
                assert np.abs(x - y).max() <= (once + rounding) * np.abs(x).max()


@pytest.mark.parametrize("grid", GRIDS, ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("comp", [0, 1])
def test_velocity_refinement(grid, comp):
    from channel3d_amd import lib as L
    with _channel(*grid) as g:
        rhs, a, b = (g.alloc_batch(L.INTERIOR, 2) for _ in range(3))
        for q, f in enumerate(_fields(g, 2, False)):
            g.upload(rhs[q], f, L.INTERIOR)
        g.helmholtz_batch(comp, 1, rhs, a, -1)
        g.helmholtz_batch(comp, 1, rhs, b, 1)
        for q in range(2):
            x, y = g.download(a[q], L.INTERIOR), g.download(b[q], L.INTERIOR)
            assert np.abs(x - y).max() <= 1e-11 * np.abs(x).max()  # (20 eps)^2, rounding
