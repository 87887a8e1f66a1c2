"""Routes of the fused elastic forward (mode 2) on a batch that is small enough
for the tiles of two steps: without a tile width it takes them, and a width
given with set_chunk takes the one-step march.  `blocked_bytes`, which only a
launch of two steps reports, tells them apart.  Either is captured in a graph
with the eager run's bits, replays after eager work in between included, and
agrees with the FP64 oracle to 1e-5, as every FP32 forward kernel."""
import numpy as np
import pytest

import oracle_lib as orc
from cases import DT, DX, DZ, elastic_model, uneven_shots, wavelet
from ds2d_amd import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("chunk", [None, (64, 256, 2), (32, 256, 4), (64, 512, 4), (64, 704, 4)])
def test_eager_graph_and_oracle(chunk, boundary):
    allnx, allnz, pml, nt = 96, 40, 20, 125
    vp, vs, rho = elastic_model(allnx, allnz, 16)
    wav = wavelet(nt, f0=40.0)
    shots = uneven_shots(allnx, pml, widths=[50, 96], starts=[10, 0], boundary=boundary)
    s = Solver(dx=DX, dz=DZ, dt=DT, nt=nt, allnx=allnx, allnz=allnz, pml=pml, nx_max=allnx, wavelet=wav)
    s.set_model(vp, vs, rho)
    if chunk:
        s.set_chunk(*chunk)
    z, x, st = s.batch_forward(shots)
    assert (st["blocked_bytes"] > 0) == (chunk is None)
    for _ in range(3):
        s.set_graph(False)
        s.batch_forward(shots[:1], mode=1)  # unrelated eager work in between
        s.set_graph(True)
        gz, gx, st = s.batch_forward(shots)
        assert (st["blocked_bytes"] > 0) == (chunk is None)
        assert np.array_equal(gz, z) and np.array_equal(gx, x)
    s.close()
    at = 0
    for sh in shots:
        n = sh.ntr * nt
        oz, ox = orc.elastic_forward(orc.make_shot(sh, allnx, allnz, pml, nt, DX, DZ, DT), vp, vs, rho, wav)
        e = orc.rel_l2(z[at:at + n], oz), orc.rel_l2(x[at:at + n], ox)
        print(f"chunk {chunk} boundary {boundary}: {e[0]:.1e} {e[1]:.1e}")
        assert np.abs(oz).max() > 0 and max(e) <= 1e-5
        at += n
