"""The fused elastic Born steps on tiles (kernels_eborn_tile.hip) at their edges
against the per-cell kernels: windows narrower and lower than a tile, of
exactly a tile's rows and columns (of both widths) and one more, several
windows, few steps, the strain history and the reversed background, and a batch
large enough for the wide tiles.

The two share their arithmetic down to each contraction, so records and
gradients are equal bit for bit."""
import numpy as np
import pytest

from cases import DT, DX, DZ, elastic_model, uneven_shots, wavelet
from ds2d_amd import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bg_mode", [1, 2])
@pytest.mark.parametrize("allnx,allnz,pml,widths,nt", [
    (3, 2, 4, [3], 60), (16, 48, 4, [16], 60), (17, 49, 4, [17, 9], 61), (15, 47, 4, [15, 1], 60),
    (33, 97, 4, [33, 31], 60), (75, 61, 20, [75, 40, 33], 61), (40, 30, 20, [40], 1), (40, 30, 20, [40], 2),
    (201, 140, 20, [201] * 120 + [77] * 60, 5)])
def test_tiles_equal_the_per_cell_kernels(allnx, allnz, pml, widths, nt, bg_mode):
    vp, vs, rho = elastic_model(allnx, allnz, 5)
    wav = wavelet(nt, f0=40.0)
    shots = uneven_shots(allnx, pml, widths, [allnx - w for w in widths], boundary=1)
    for sh in shots:
        sh.isz = pml + min(2, allnz - 1)
    rng = np.random.default_rng(3)
    pp = (0.05 * rng.standard_normal((allnx, allnz))).astype(np.float32)
    ps = (0.03 * rng.standard_normal((allnx, allnz))).astype(np.float32)
    n = sum(s.ntr for s in shots) * nt
    rz, rx = (rng.standard_normal(n).astype(np.float32) for _ in range(2))
    out = []
    for fused in (True, False):
        s = Solver(dx=DX, dz=DZ, dt=DT, nt=nt, allnx=allnx, allnz=allnz, pml=pml, nx_max=allnx, wavelet=wav,
                   bg_mode=bg_mode)
        s.set_model(vp, vs, rho)
        s.set_fused_born(fused)
        fz, fx, _ = s.eborn_forward(shots, pp, ps)
        gpp, gps, _ = s.eborn_adjoint(shots, rz, rx)
        out.append([fz, fx, gpp, gps])
        if nt > 2:  # no gradient before
            ipp, ips, hist, _ = s.elsrtm_cg(shots, rz, rx, 1)
            out[-1] += [ipp, ips, np.asarray(hist)]
        s.close()
    assert np.abs(out[0][0]).max() > 0 or nt < 3
    for a, b in zip(*out):
        assert np.array_equal(a, b)
