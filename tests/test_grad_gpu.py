"""The launches of the reference gradient (kernels_grad.hip) where they can go
wrong: windows whose edge bands overlap or that end inside a block, one batch
with a PML and a random-boundary window, and several traces on one column.  Tolerance: relative L2 <= 1e-5 against FP64 (FP32 records and
images), as for the other tests of these entry points."""
import numpy as np
import pytest

import oracle_lib as orc
from cases import DT, DX, DZ, elastic_model, uneven_shots, wavelet
from ds2d_amd import Solver
from ds2d_amd.lib import ShotSpec

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _osh(spec, allnx, allnz, pml, nt):
    return orc.make_shot(spec, allnx, allnz, pml, nt, DX, DZ, DT, rho_const=2000.0)


def _images(allnx, allnz):
    rng = np.random.default_rng(22)
    return [(0.05 * rng.standard_normal((allnx, allnz))).astype(np.float32) for _ in range(2)]


@pytest.mark.parametrize("allnx,allnz,pml,widths,boundaries,nt", [
    (6, 5, 4, [6], [0], 160), (5, 61, 8, [5], [0], 160), (67, 5, 20, [67], [1], 160),
    (69, 30, 20, [33, 69], [0, 1], 200)])
def test_gradient_matches_oracle(allnx, allnz, pml, widths, boundaries, nt):
    vp, vs, _ = elastic_model(allnx, allnz, 21)
    wav = wavelet(nt, f0=40.0)
    pp, ps = _images(allnx, allnz)
    shots = uneven_shots(allnx, pml, widths, [allnx - w for w in widths])
    for sh, b in zip(shots, boundaries):
        sh.boundary = b
        sh.isz = pml + min(2, allnz - 1)
    obs = [orc.elastic_forward(_osh(sh, allnx, allnz, pml, nt), vp * np.float32(1.03), vs, None, wav, prec="f")
           for sh in shots]
    s = Solver(dx=DX, dz=DZ, dt=DT, nt=nt, allnx=allnx, allnz=allnz, pml=pml, nx_max=allnx, wavelet=wav,
               rho_const=2000.0)
    s.set_model(vp, vs, None)
    s.set_image(pp, ps)
    mf = s.batch_gradient(shots, np.concatenate([o[0] for o in obs]), np.concatenate([o[1] for o in obs]), 1)
    g = s.take_gradients()
    s.close()
    og, omf = np.zeros(7 * allnx * allnz), 0.0
    for sh, (z, x) in zip(shots, obs):
        og, m1 = orc.elsrtm_shot(_osh(sh, allnx, allnz, pml, nt), vp, vs, None, wav, pp, ps, z, x, 1, sh.ngx_min,
                                 grads7=og)
        omf += m1
    for k, name in enumerate(["pp", "ps", "illum", "b_pp", "b_ps", "b2_pp", "b2_ps"]):
        e = orc.rel_l2(g[k], og.reshape(7, allnx, allnz)[k])
        print(f"{name}: {e:.2e}")
        assert e <= TOL, name
    assert abs(mf - omf) <= TOL * max(1.0, abs(omf))


@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("allnx,allnz", [(8, 56), (16, 57), (17, 55), (9, 112)])
def test_gradient_at_the_edges_of_tiles(allnx, allnz, boundary):
    """Update regions of exactly one and two tiles of 8 x 56 cells, one cell more and one less."""
    test_gradient_matches_oracle(allnx, allnz, 4, [allnx], [boundary], 160)


def test_background_beside_the_window(monkeypatch):
    """The rows above and below the physical window, of which the background's Born source of b
    (images 3 and 4) sees the velocities a step late.  4e-6: rounding of the FP32 fields of 2 * 400
    steps, sqrt(800) * 2^-24 = 1.7e-6, and twice that; stale velocities there give 6.9e-6 and 1.0e-5."""
    monkeypatch.setitem(globals(), "TOL", 4e-6)
    test_gradient_matches_oracle(60, 30, 20, [60], [0], 400)


def test_born_records_of_traces_on_one_column():
    allnx, allnz, pml, nt = 40, 30, 20, 150
    vp, vs, _ = elastic_model(allnx, allnz, 21)
    wav = wavelet(nt, f0=40.0)
    cols = pml + np.array([7, 20, 7, 33, 7], np.int32)
    shots = [ShotSpec(0, allnx, pml + 20, pml + 2, pml, c, boundary=0) for c in (cols, np.unique(cols))]
    s = Solver(dx=DX, dz=DZ, dt=DT, nt=nt, allnx=allnx, allnz=allnz, pml=pml, nx_max=allnx, wavelet=wav,
               rho_const=2000.0)
    s.set_model(vp, vs, None)
    s.set_image(*_images(allnx, allnz))
    for order in (1, 2):
        (az, ax), (bz, bx) = (s.born([sh], order) for sh in shots)
        at = np.searchsorted(np.unique(cols), cols)
        assert np.abs(bz).max() > 0
        assert np.array_equal(az.reshape(-1, nt), bz.reshape(-1, nt)[at])
        assert np.array_equal(ax.reshape(-1, nt), bx.reshape(-1, nt)[at])
    s.close()
