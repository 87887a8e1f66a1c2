"""Records above and below the size that goes through pinned pieces
(record_copy.hpp) into buffers on the device: the bits that host memory gets."""
import ctypes as C

import numpy as np
import pytest

from cases import DT, DX, DZ, elastic_model, uneven_shots, wavelet
from ds2d_amd import Solver
from ds2d_amd import lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nshots", [1, 18])
def test_records_into_device_memory(nshots):
    allnx, allnz, pml, nt = 75, 30, 8, 1003
    vp, vs, rho = elastic_model(allnx, allnz, 5)
    shots = uneven_shots(allnx, pml, [75] * nshots, [0] * nshots)
    s = Solver(dx=DX, dz=DZ, dt=DT, nt=nt, allnx=allnx, allnz=allnz, pml=pml, nx_max=allnx, wavelet=wavelet(nt))
    s.set_model(vp, vs, rho)
    want = s.batch_forward(shots)[:2]
    hip = C.CDLL("libamdhip64.so.7")
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    hip.hipFree.argtypes = [C.c_void_p]
    buf = [C.c_void_p(), C.c_void_p()]
    for b in buf:
        assert hip.hipMalloc(C.byref(b), want[0].nbytes) == 0
    z, x = (C.cast(b, C.POINTER(C.c_float)) for b in buf)
    assert s.lib.ds2d_batch_forward(s.h, nshots, L._shots_array(shots), z, x, 2, None) == 0, s.lib.ds2d_last_error()
    for b, w in zip(buf, want):
        got = np.empty_like(w)
        assert hip.hipMemcpy(got.ctypes.data, b, got.nbytes, 2) == 0
        assert np.abs(w).max() > 0 and np.array_equal(got, w)
        hip.hipFree(b)
    s.close()
