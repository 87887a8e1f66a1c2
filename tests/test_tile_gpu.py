"""The tiles of two elastic steps per launch (k_tile_steps) against the FP64 oracle.

The batch sizes pick each tile width in turn (10, 16, 24 and 28 owned
columns); the windows end inside a tile in both directions and an odd number
of steps ends on a single-step launch.  Tolerance: the 1e-5 relative L2 that
every FP32 forward kernel of the library is held to against the oracle."""
import numpy as np
import pytest

import oracle_lib as orc
from cases import DT, DX, DZ, elastic_model, uneven_shots, wavelet
from ds2d_amd import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("allnx,allnz,nshots,nt", [(9, 9, 1, 3), (61, 43, 1, 121), (247, 101, 2, 41), (251, 97, 4, 41),
                                                   (251, 101, 8, 21)])
def test_tile_steps_match_oracle(allnx, allnz, nshots, nt, boundary):
    pml = 20
    vp, vs, rho = elastic_model(allnx, allnz, 11)
    wav = wavelet(nt, f0=60.0)
    widths = [max(1, allnx - 3 * i) for i in range(nshots)]
    shots = uneven_shots(allnx, pml, widths, [allnx - w for w in widths], boundary=boundary)
    s = Solver(dx=DX, dz=DZ, dt=DT, nt=nt, allnx=allnx, allnz=allnz, pml=pml, nx_max=allnx, wavelet=wav)
    s.set_model(vp, vs, rho)
    rz, rx, st = s.batch_forward(shots)
    assert s.time_block() == 1 and st["blocked_bytes"] > 0  # the tiles ran
    at = 0
    for sh in shots[:3]:
        oz, ox = orc.elastic_forward(orc.make_shot(sh, allnx, allnz, pml, nt, DX, DZ, DT), vp, vs, rho, wav)
        n = sh.ntr * nt
        assert orc.rel_l2(rz[at:at + n], oz) <= 1e-5 and orc.rel_l2(rx[at:at + n], ox) <= 1e-5
        at += n
    # the same records from a graph of the loop, and again from its replay on a warm handle
    s.set_graph(True)
    for _ in range(2):
        gz, gx, _ = s.batch_forward(shots)
        assert np.array_equal(gz, rz) and np.array_equal(gx, rx)
    s.close()
