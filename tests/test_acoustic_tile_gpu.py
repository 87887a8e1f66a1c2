"""The fused acoustic steps on tiles (kernels_acoustic_tile.hip) at their edges
against the per-cell kernels: windows narrower and lower than a tile, of
exactly a tile's rows and columns and one more, several windows, one step.

The two run the same expressions on the same FP32 state; over 120 steps their
rounding may differ by a few units in the last place a step, so records and
gradients are held to a relative L2 of 120 * 2^-23 (1.4e-5)."""
import numpy as np
import pytest

import oracle_lib as orc
from cases import DT, DX, DZ, elastic_model, uneven_shots, wavelet
from ds2d_amd import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("allnx,allnz,pml,widths,nt", [
    (3, 2, 4, [3], 120), (16, 48, 4, [16], 120), (17, 49, 4, [17, 9], 120), (15, 47, 4, [15], 121),
    (75, 61, 20, [75, 40, 33], 120), (40, 30, 20, [40], 1), (40, 30, 20, [40], 2)])
def test_tiles_match_the_per_cell_kernels(allnx, allnz, pml, widths, nt):
    vp, _, rho = elastic_model(allnx, allnz, 5)
    wav = wavelet(nt, f0=40.0)
    shots = uneven_shots(allnx, pml, widths, [allnx - w for w in widths], boundary=1)
    for sh in shots:
        sh.isz = pml + min(2, allnz - 1)
    rng = np.random.default_rng(3)
    refl = (0.05 * rng.standard_normal((allnx, allnz))).astype(np.float32)
    res = rng.standard_normal(sum(s.ntr for s in shots) * nt).astype(np.float32)
    out = []
    for fused in (0, -1):
        s = Solver(dx=DX, dz=DZ, dt=DT, nt=nt, allnx=allnx, allnz=allnz, pml=pml, nx_max=allnx, wavelet=wav,
                   physics=1, bg_mode=1)
        s.set_model(vp, None, rho)
        s.set_fused(fused)
        g, _ = s.born_adjoint(shots, res)
        # an image from a start of refl: the first residual is d - L refl
        img, hist, _ = s.lsrtm_cg(shots, res, 1, image0=refl)
        out.append((g, img, hist))
        s.close()
    (g0, i0, h0), (g1, i1, h1) = out
    tol = 120 * 2.0 ** -23
    assert np.abs(g0).max() > 0 and orc.rel_l2(g1, g0) <= tol
    assert orc.rel_l2(i1 - refl, i0 - refl) <= tol and np.allclose(h1, h0, rtol=tol)
