"""Device memory of the calls that hold the most of it, a padded cell.

A batch that fits a card has to go on fitting it, so what a call takes is held
to what its wavefields, media and histories need:
  gradient        two FP64 and three FP32 split wavefields (15 arrays each),
                  9 medium arrays, and 8 floats of products or velocity copies
  acoustic Born   16 FP32 and 3 FP64 arrays, 9 medium arrays, and the history
plus images and records.  64 MB on top: some 30 allocations, each rounded up
to 2 MB.  What the library keeps by itself is there before the measurement,
from a small call of the same kind."""
import ctypes as C

import numpy as np
import pytest

from cases import DT, DX, DZ, wavelet
from ds2d_amd import Solver
from ds2d_amd.lib import ShotSpec, load

pytestmark = pytest.mark.gpu

PML, NT = 20, 2
SLACK = 64 << 20


def _free():
    load()
    hip = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipDeviceSynchronize() == 0 and hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _used(call, nx, nz, physics, boundary):
    """Bytes that the first call on a handle takes; the handle's own buffers are there before."""
    s = Solver(dx=DX, dz=DZ, dt=DT, nt=NT, allnx=nx, allnz=nz, pml=PML, nx_max=nx, wavelet=wavelet(NT),
               physics=physics, rho_const=2000.0, bg_mode=1)
    vp = np.full((nx, nz), 2500.0, np.float32)
    s.set_model(vp, None if physics else vp / 2, None)
    shot = ShotSpec(0, nx, PML + nx // 2, PML + 2, PML, PML + np.arange(0, nx, 50, dtype=np.int32), boundary=boundary)
    before = _free()
    call(s, shot, np.ones(shot.ntr * NT, np.float32))
    used = before - _free()
    s.close()
    return used


@pytest.mark.parametrize("boundary", [0, 1])
def test_gradient(boundary):
    def call(s, shot, d):
        s.batch_gradient([shot], d, d, 1)

    nx, nz = 4000, 1960
    _used(call, 60, 40, 0, boundary)
    used = _used(call, nx, nz, 0, boundary)
    cells = (nx + 2 * PML) * (nz + 2 * PML)
    bound = cells * (2 * 15 * 8 + 3 * 15 * 4 + 9 * 4 + 8 * 4) + 7 * 4 * nx * nz + SLACK
    print(f"{used / cells:.1f} B a cell, at most {bound / cells:.1f}")
    assert used <= bound


def test_acoustic_adjoint():
    def call(s, shot, d):
        s.born_adjoint([shot], d)

    nx, nz = 4000, 1960
    _used(call, 60, 40, 1, 1)
    used = _used(call, nx, nz, 1, 1)
    cells = (nx + 2 * PML) * (nz + 2 * PML)
    bound = cells * (16 * 4 + 3 * 8 + 9 * 4) + 4 * nx * nz * (NT + 2) + SLACK
    print(f"{used / cells:.1f} B a cell, at most {bound / cells:.1f}")
    assert used <= bound
