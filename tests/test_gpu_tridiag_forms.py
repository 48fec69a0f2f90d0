"""The pressure solve's wall-normal sweep in the form that large grids take (a
lane per real or imaginary part, 24-row FP64 and 32-row FP32 segments,
256-thread workgroups) against the one-lane sweep with 16-row segments, bit for
bit: the same operations, cut elsewhere.  129 x 256 wavenumber pairs just pass
the line count of that form; the rows run over the edges of both segmentings."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny", [3, 16, 24, 25, 32, 33, 49, 73])
@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
def test_large_grid_sweep_bitwise(monkeypatch, ny, fp32):
    from channel3d_amd import Channel, lib as L
    case = dict(nxc=256, nyc=ny, nzc=256, xlx=6.0, yly=2.0, zlz=3.0, xnu=1e-4, dt=0.002,
                gamma=1.2, ubulk=1.0)
    f = np.random.default_rng(ny).standard_normal((256, ny, 256))
    out = []
    for lanes in ("1", "2"):
        monkeypatch.setenv("C3D_TRIDIAG_LANES", lanes)
        with Channel(case, precision=L.FP32 if fp32 else L.FP64) as g:
            g.upload(L.ARR1, f - f.mean())
            g.ppe(L.ARR1, L.HALOARR)
            out.append(g.download(L.HALOARR)[1:-2, 1:ny + 1, 1:-2])
    assert np.isfinite(out[0]).all() and np.abs(out[0]).max() > 0
    assert np.array_equal(out[0], out[1])
