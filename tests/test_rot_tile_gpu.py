"""The fused rotation step on tiles (kernels_rot_tile.hip) at its edges against
the per-cell kernels, damped and random-boundary windows in one batch: windows
narrower and lower than a tile, of exactly a tile's rows and columns (of both
widths) and one more, few steps, and a batch large enough for the wide tiles.

The two sum the same increments in another order (the tile kernel keeps vx, vz
and theta, omega as totals); over 120 steps their rounding may differ by a few
units in the last place a step, so records are held to a relative L2 of
120 * 2^-23 (1.4e-5)."""
import numpy as np
import pytest

from cases import DT, DX, DZ, elastic_model, uneven_shots, wavelet
from ds2d_amd import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("allnx,allnz,pml,widths,nt", [
    (3, 2, 4, [3], 120), (16, 48, 4, [16, 16], 120), (17, 49, 4, [17, 9], 121), (15, 47, 4, [15, 1], 120),
    (49, 97, 4, [49, 48, 47], 120), (75, 61, 20, [75, 40, 33], 121), (40, 30, 20, [40, 12], 1),
    (40, 30, 20, [40, 12], 2), (201, 140, 20, [201] * 120 + [77] * 100, 12)])
def test_tiles_match_the_per_cell_kernels(allnx, allnz, pml, widths, nt):
    vp, vs, rho = elastic_model(allnx, allnz, 5)
    wav = wavelet(nt, f0=40.0)
    shots = uneven_shots(allnx, pml, widths, [allnx - w for w in widths], boundary=0)
    for i, sh in enumerate(shots):
        sh.isz, sh.boundary = pml + min(2, allnz - 1), i % 2
    out = []
    for fused in (True, False):
        s = Solver(dx=DX, dz=DZ, dt=DT, nt=nt, allnx=allnx, allnz=allnz, pml=pml, nx_max=allnx, wavelet=wav)
        s.set_model(vp, vs, rho)
        s.set_fused_rotation(fused)
        out.append(s.rot_forward(shots)[:2])
        s.close()
    for a, b in zip(*out):
        assert np.abs(b).max() > 0 or nt == 1  # the wavelet starts from zero
        assert np.linalg.norm(a - b) <= 120 * 2.0 ** -23 * np.linalg.norm(b)
