"""Two elastic steps per launch (kernels_fused2.hip) where waves change between
the damped and the undamped code: chunks that start in a damping strip, in the
middle or end in the other strip, strips wider and narrower than the march's
lead, windows of several row blocks, random-boundary windows in the same batch.

Compared with one step per launch, the same scheme in another order of sums:
over nt steps the rounding may differ by a few units in the last place a step,
so records are held to a relative L2 of nt * 2^-23."""
import numpy as np
import pytest

import oracle_lib as orc
from cases import DT, DX, DZ, elastic_model, uneven_shots, wavelet
from ds2d_amd import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("allnx,allnz,pml,widths,chunk,nt", [
    (150, 60, 8, [150, 61], 40, 120), (150, 60, 8, [150, 97], 64, 121), (120, 40, 20, [120, 33], 200, 120),
    (90, 40, 4, [90, 5], 16, 120), (60, 560, 12, [60, 44], 30, 120), (70, 40, 40, [70], 64, 120)])
def test_two_steps_match_one(allnx, allnz, pml, widths, chunk, nt):
    vp, vs, rho = elastic_model(allnx, allnz, 5)
    wav = wavelet(nt, f0=40.0)
    shots = uneven_shots(allnx, pml, widths, [allnx - w for w in widths], boundary=0)
    for i, sh in enumerate(shots):
        sh.isz, sh.boundary = pml + 2, i % 2
    out = []
    for block in (2, 1):
        s = Solver(dx=DX, dz=DZ, dt=DT, nt=nt, allnx=allnx, allnz=allnz, pml=pml, nx_max=allnx, wavelet=wav)
        s.set_model(vp, vs, rho)
        s.set_chunk(chunk, 512, 2)
        s.set_chunk_plan(False)
        s.set_time_block(block)
        z, x, st = s.batch_forward(shots, mode=2)
        assert st["stencil_launches"] == (nt // 2 if block == 2 else nt)
        out.append((z, x))
        s.close()
    for a, b in zip(*out):
        assert np.abs(b).max() > 0
        assert orc.rel_l2(a, b) <= nt * 2.0 ** -23
