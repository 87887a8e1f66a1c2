"""Addresses of the gradient's kernels (ds2d_amd/csrc/slot_address.hpp), compiled
on the host: the cell of every window that has a place in memory, those of more
than 2^32 bytes too, where a 32-bit offset from the window's start wraps (FP64
fields from 2^29 cells on, FP32 fields from 2^30)."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r'''
#define __host__
#define __device__
#include "slot_address.hpp"
template <typename T>
static unsigned long long place(unsigned long long base, long long off, int ix, int nz, int z) {
    return (unsigned long long)&ds2d::column_cell((T*)base, ds2d::column_start(off, ix, nz), z);
}
extern "C" unsigned long long place4(unsigned long long base, long long off, int ix, int nz, int z) {
    return place<float>(base, off, ix, nz, z);
}
extern "C" unsigned long long place8(unsigned long long base, long long off, int ix, int nz, int z) {
    return place<double>(base, off, ix, nz, z);
}
'''


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("address")
    (d / "shim.cpp").write_text(SHIM)
    so = d / "libaddress.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "ds2d_amd", "csrc"),
                    str(d / "shim.cpp"), "-o", str(so)], check=True)
    return C.CDLL(str(so))


@pytest.mark.parametrize("size", [4, 8])
@pytest.mark.parametrize("off,nxp,nzp", [(0, 9, 9), (64, 291, 141), (1 << 20, 16384, 32768), (3 << 29, 16385, 32768),
                                         (0, 46341, 46341), (0, 70001, 65537)])
def test_cells(lib, size, off, nxp, nzp):
    f = getattr(lib, f"place{size}")
    f.restype = C.c_ulonglong
    f.argtypes = [C.c_ulonglong, C.c_longlong, C.c_int, C.c_int, C.c_int]
    base = 0x7F0000000000
    for ix in (0, 4, nxp // 2, nxp - 5, nxp - 1):
        for z in (0, 4, nzp // 2, nzp - 1):
            assert f(base, off, ix, nzp, z) == base + size * (off + ix * nzp + z), (ix, z)
