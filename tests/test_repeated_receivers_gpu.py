"""Several traces on one receiver column.

A forward pass writes each of them: the same bits as a run that has every
column once, whatever kernels take the step and whatever an earlier call left
in the record buffer.  An adjoint pass injects the sum of their residuals:
with whole-numbered residuals, whose sums are exact, the same bits as one
trace a column that carries the sum."""
import numpy as np
import pytest

from cases import DT, DX, DZ, elastic_model, wavelet
from ds2d_amd import Solver
from ds2d_amd.lib import ShotSpec

pytestmark = pytest.mark.gpu

NX, NZ, PML, NT = 50, 30, 8, 90
COLS = [PML + np.array(c, np.int32) for c in ([7, 20, 7, 33, 7, 0, 0], [4, 12, 49, 12])]


def _shots(cols, boundary):
    return [ShotSpec(0, NX, PML + 20 + 3 * i, PML + 2, PML, c, shot_id=i, boundary=boundary)
            for i, c in enumerate(cols)]


def _pair(boundary):
    """The shots with repeated columns, with each once, and the places of the former's traces in the latter's."""
    once = [np.unique(c) for c in COLS]
    place, base = [], 0
    for c, u in zip(COLS, once):
        place.append(base + np.searchsorted(u, c))
        base += u.size
    return _shots(COLS, boundary), _shots(once, boundary), np.concatenate(place)


def _solver(physics=0, bg_mode=0):
    s = Solver(dx=DX, dz=DZ, dt=DT, nt=NT, allnx=NX, allnz=NZ, pml=PML, nx_max=NX, wavelet=wavelet(NT, f0=40.0),
               physics=physics, bg_mode=bg_mode)
    vp, vs, rho = elastic_model(NX, NZ, 8)
    s.set_model(vp, None if physics else vs, rho)
    return s


def _check_records(run, boundary):
    twice, once, place = _pair(boundary)
    out = [run(sh) for sh in (once, twice)]
    for a, b in zip(*out):
        assert np.abs(a).max() > 0
        assert np.array_equal(b.reshape(-1, NT), a.reshape(-1, NT)[place])


@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("step", ["tiles", "march", "two-step march", "two kernels", "reference layout"])
def test_elastic_records(step, boundary):
    s = _solver()
    mode = {"two kernels": 1, "reference layout": 0}.get(step, 2)
    if step == "march":
        s.set_chunk(64, 256, 2)
    if step == "two-step march":
        s.set_chunk(64, 704, 2)
        s.set_time_block(2)
    _check_records(lambda sh: s.batch_forward(sh, mode=mode)[:2], boundary)
    s.close()


@pytest.mark.parametrize("fused", [False, True])
def test_rotation_records(fused):
    s = _solver()
    s.set_fused_rotation(fused)
    _check_records(lambda sh: s.rot_forward(sh)[:2], 0)
    s.close()


def test_acoustic_born_records():
    s = _solver(physics=1)
    refl = (0.05 * np.random.default_rng(2).standard_normal((NX, NZ))).astype(np.float32)
    _check_records(lambda sh: s.born_forward(sh, refl)[:2], 1)
    s.close()


@pytest.mark.parametrize("fused", [False, True])
def test_elastic_born_records(fused):
    s = _solver()
    s.set_fused_born(fused)
    pp, ps = (0.05 * np.random.default_rng(2).standard_normal((2, NX, NZ))).astype(np.float32)
    _check_records(lambda sh: s.eborn_forward(sh, pp, ps)[:2], 1)
    s.close()


def _residuals(seed):
    """Residuals of the repeated traces and their sums a column: whole numbers up to 9."""
    _, once, place = _pair(1)
    r = np.random.default_rng(seed).integers(-9, 10, (place.size, NT)).astype(np.float32)
    total = np.zeros((sum(sh.ntr for sh in once), NT), np.float32)
    np.add.at(total, place, r)
    return r.ravel(), total.ravel()


# the shots of one launch, and one after another
@pytest.mark.parametrize("batch", [0, 1])
@pytest.mark.parametrize("bg_mode", [1, 2])
@pytest.mark.parametrize("fused", [0, -1])
def test_acoustic_adjoint(fused, bg_mode, batch):
    twice, once, _ = _pair(1)
    r, total = _residuals(5)
    s = _solver(physics=1, bg_mode=bg_mode)
    s.set_fused(fused)
    s.set_batch(batch)
    a, b = s.born_adjoint(once, total)[0], s.born_adjoint(twice, r)[0]
    assert np.abs(a).max() > 0 and np.array_equal(a, b)
    s.close()


@pytest.mark.parametrize("batch", [0, 1])
@pytest.mark.parametrize("bg_mode", [1, 2])
@pytest.mark.parametrize("fused", [False, True])
def test_elastic_adjoint(fused, bg_mode, batch):
    twice, once, _ = _pair(1)
    (rz, tz), (rx, tx) = _residuals(6), _residuals(7)
    s = _solver(bg_mode=bg_mode)
    s.set_fused_born(fused)
    s.set_batch(batch)
    a, b = s.eborn_adjoint(once, tz, tx)[:2], s.eborn_adjoint(twice, rz, rx)[:2]
    for i in range(2):
        assert np.abs(a[i]).max() > 0 and np.array_equal(a[i], b[i])
    s.close()


def test_least_squares_migration_of_repeated_traces():
    """The solvers' maps are each other's adjoints with repeated columns too: the first step's residual is what
    CGLS gives for the Born records and adjoint images of the single calls."""
    twice, _, _ = _pair(1)
    s = _solver(physics=1)
    refl = (0.05 * np.random.default_rng(2).standard_normal((NX, NZ))).astype(np.float32)
    d = s.born_forward(twice, refl)[1]
    img, resid, _ = s.lsrtm_cg(twice, d, 1)
    g = s.born_adjoint(twice, d)[0]
    q = s.born_forward(twice, g)[1]
    g, q, d = (a.astype(np.float64) for a in (g, q, d))
    step = (g * g).sum() / (q * q).sum()
    want = np.linalg.norm(d - step * q) / np.linalg.norm(d)
    # FP32 passes of NT steps: NT * 2^-23 of the gradient and of the records
    assert np.abs(resid[1] - want) <= 2 * NT * 2.0 ** -23 * max(1.0, want)
    assert np.linalg.norm(img - step * g) <= 2 * NT * 2.0 ** -23 * np.linalg.norm(step * g)
    s.close()


def test_rotation_rtm():
    """The receiver side adds every trace's sample."""
    twice, once, _ = _pair(1)
    (rz, tz), (rx, tx) = _residuals(6), _residuals(7)
    s = _solver()
    a, b = s.rot_rtm(once, tz, tx), s.rot_rtm(twice, rz, rx)
    for i in range(2):
        assert np.abs(a[i]).max() > 0 and np.array_equal(a[i], b[i])
    s.close()


@pytest.mark.parametrize("boundary", [0, 1])
def test_decomposed_rtm(boundary):
    """The receiver side assigns the samples, of several on a cell the last trace's, as one after another would."""
    twice, once, place = _pair(boundary)
    r = np.random.default_rng(4).standard_normal((place.size, NT)).astype(np.float32)
    last = np.zeros((sum(sh.ntr for sh in once), NT), np.float32)
    for t, p in enumerate(place):
        last[p] = r[t]
    s = _solver()
    a, b = s.decomp_rtm(once, 0, last.ravel()), s.decomp_rtm(twice, 0, r.ravel())
    assert np.abs(a).max() > 0 and np.array_equal(a, b)
    s.close()
