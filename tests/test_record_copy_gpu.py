"""Records of a batch too large for one plain copy (record_copy.hpp): they
arrive whole, in pieces that do not divide them, and equal those of the same
shots a few at a time, bit for bit; the buffer may be used before and one
component may be left out."""
import ctypes as C

import numpy as np
import pytest

from cases import DT, DX, DZ, elastic_model, uneven_shots, wavelet
from ds2d_amd import Solver
from ds2d_amd import lib as L

pytestmark = pytest.mark.gpu


def test_large_records_equal_small_batches():
    allnx, allnz, pml, nt, n = 75, 30, 8, 1003, 18
    vp, vs, rho = elastic_model(allnx, allnz, 5)
    widths = [75 - (i % 5) for i in range(n)]
    shots = uneven_shots(allnx, pml, widths, [allnx - w for w in widths], boundary=0)
    assert 2 * sum(s.ntr for s in shots) * nt * 4 > 9 << 20  # two components, above 8 MB
    s = Solver(dx=DX, dz=DZ, dt=DT, nt=nt, allnx=allnx, allnz=allnz, pml=pml, nx_max=allnx, wavelet=wavelet(nt))
    s.set_model(vp, vs, rho)
    s.set_chunk(64, 256, 2)
    z, x, _ = s.batch_forward(shots, mode=2)
    parts = [s.batch_forward(shots[i:i + 3], mode=2)[:2] for i in range(0, n, 3)]
    assert np.abs(z).max() > 0
    assert np.array_equal(z, np.concatenate([p[0] for p in parts]))
    assert np.array_equal(x, np.concatenate([p[1] for p in parts]))
    only = np.full(z.size + 3, 7, np.float32)  # a used buffer, x left out
    p = only[1:].ctypes.data_as(C.POINTER(C.c_float))
    assert s.lib.ds2d_batch_forward(s.h, n, L._shots_array(shots), p, None, 2, None) == 0
    assert np.array_equal(only[1:-2], z) and only[0] == 7 and np.all(only[-2:] == 7)
    s.close()
