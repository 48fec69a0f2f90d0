"""The pressure solve's wall-normal sweep with its forward values in LDS, which
small grids take (one or two wavefronts per CU), against the one-lane sweep with
checkpoints, bit for bit: the same operations.  Rows at the edges of the 16-row
segments and of the rows that half a CU's LDS holds (FP64 104, FP32 208) and a
CU's (208, 416), line counts at the edges of a wavefront and on both sides of the
form's own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (nx, ny, nz): nx / 2 + 1 times nz wavenumber pairs
GRIDS = [(16, 3, 8), (24, 16, 20), (18, 17, 16), (64, 33, 64), (32, 104, 48), (32, 105, 48),
         (16, 208, 24), (16, 209, 24), (16, 416, 16), (16, 417, 16), (120, 24, 128),
         (120, 104, 256), (128, 24, 256), (120, 150, 128)]


@pytest.mark.parametrize("grid", GRIDS, ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
@pytest.mark.parametrize("nt", ["0", "1"])
def test_lds_sweep_bitwise(monkeypatch, grid, fp32, nt):
    from channel3d_amd import Channel, lib as L
    nx, ny, nz = grid
    case = dict(nxc=nx, nyc=ny, nzc=nz, xlx=6.0, yly=2.0, zlz=3.0, xnu=1e-4, dt=0.002,
                gamma=1.2, ubulk=1.0)
    monkeypatch.setenv("C3D_NT", nt)
    f = np.random.default_rng(ny).standard_normal(grid)
    out = []
    for lanes in ("1", None):
        if lanes:
            monkeypatch.setenv("C3D_TRIDIAG_LANES", lanes)
        else:
            monkeypatch.delenv("C3D_TRIDIAG_LANES")
        with Channel(case, precision=L.FP32 if fp32 else L.FP64) as g:
            g.upload(L.ARR1, f - f.mean())
            g.ppe(L.ARR1, L.HALOARR)
            out.append(g.download(L.HALOARR)[1:-2, 1:ny + 1, 1:-2])
    assert np.isfinite(out[0]).all() and np.abs(out[0]).max() > 0
    assert np.array_equal(out[0], out[1])
