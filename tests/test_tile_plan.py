"""The choice of tile of the two-step launches (ds2d_amd/csrc/tile_plan.hpp,
compiled on the host) and each tile's kernel against the FP64 oracle: one batch
for every tile that the plan can pick, so that a table of costs that drops one
of them does not drop its test.  Tolerance of the kernels: the 1e-5 relative L2
that every FP32 forward kernel of the library is held to."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import oracle_lib as orc
from cases import DT, DX, DZ, elastic_model, uneven_shots, wavelet
from ds2d_amd import Solver

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PML, CUS = 20, 256

# columns and rows of the model, windows -> owned columns of the tile
BATCHES = [((61, 43), 1, 10), ((247, 101), 2, 16), ((251, 97), 4, 24), ((251, 101), 26, 28)]

SHIM = r'''
#include "tile_plan.hpp"
extern "C" int plan(const int* nxp, int n, int nzp, int ncu, int* cols, long long* rounds) {
    const ds2d::TilePlan p = ds2d::plan_tiles(std::vector<int>(nxp, nxp + n), nzp, ncu);
    *cols = p.cols;
    *rounds = p.rounds;
    return p.kind;
}
extern "C" int kinds() { return ds2d::TILE_KINDS; }
'''


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    d = tmp_path_factory.mktemp("tiles")
    (d / "shim.cpp").write_text(SHIM)
    so = d / "libtiles.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "ds2d_amd", "csrc"),
                    str(d / "shim.cpp"), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))

    def run(nxp, nzp):
        cols, rounds = C.c_int(), C.c_longlong()
        w = (C.c_int * len(nxp))(*nxp)
        kind = lib.plan(w, len(nxp), nzp, CUS, C.byref(cols), C.byref(rounds))
        return kind, cols.value, rounds.value
    run.kinds = lib.kinds()
    return run


def _widths(allnx, nshots):
    return [max(1, allnx - 3 * i) for i in range(nshots)]


def test_batches_take_every_tile(planner):
    got = [planner([w + 2 * PML for w in _widths(nx, n)], nz + 2 * PML) for (nx, nz), n, _ in BATCHES]
    assert [c for _, c, _ in got] == [c for _, _, c in BATCHES]
    assert sorted(k for k, _, _ in got) == list(range(planner.kinds))
    # untuned batches take tiles up to eight rounds of one workgroup a CU
    assert all(1 <= r <= 8 for _, _, r in got)


@pytest.mark.parametrize("nxp,nzp", [((9,), 9), ((18, 19, 34), 40), ((291,) * 26, 141), ((8, 100), 41), ((1240,) * 16, 640)])
def test_rounds_hold_every_tile(planner, nxp, nzp):
    kind, cols, rounds = planner(nxp, nzp)
    tiles = sum(-(-(w - 8) // cols) * -(-(nzp - 8) // 32) for w in nxp)
    assert (rounds - 1) * CUS < tiles <= rounds * CUS


@pytest.mark.gpu
@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("size,nshots,cols", BATCHES)
def test_tiles_match_oracle(size, nshots, cols, boundary):
    (allnx, allnz), nt = size, 61
    vp, vs, rho = elastic_model(allnx, allnz, 11)
    wav = wavelet(nt, f0=60.0)
    widths = _widths(allnx, nshots)
    shots = uneven_shots(allnx, PML, widths, [allnx - w for w in widths], boundary=boundary)
    s = Solver(dx=DX, dz=DZ, dt=DT, nt=nt, allnx=allnx, allnz=allnz, pml=PML, nx_max=allnx, wavelet=wav)
    s.set_model(vp, vs, rho)
    rz, rx, st = s.batch_forward(shots)
    s.close()
    assert st["blocked_bytes"] > 0  # the tiles ran
    at = np.cumsum([0] + [sh.ntr * nt for sh in shots])
    for i in sorted({0, nshots // 2, nshots - 1}):
        oz, ox = orc.elastic_forward(orc.make_shot(shots[i], allnx, allnz, PML, nt, DX, DZ, DT), vp, vs, rho, wav)
        e = [orc.rel_l2(r[at[i]:at[i + 1]], o) for r, o in ((rz, oz), (rx, ox))]
        print(f"{cols} columns, shot {i}: {e[0]:.1e} {e[1]:.1e}")
        assert np.abs(oz).max() > 0 and max(e) <= 1e-5
