"""Performance cases of the DS2D hot path: what a user of the framework has it do, through its public entry points.

A case is a dict of plain values.  `kind` names the entry point that one pass
calls (see `run`); the rest are sizes and options.  The models, images and
records of a case are made from its seed with numpy alone: faulted layered
models with Gardner density, 9x9-smoothed migration models, reflectivities of
the layers that smoothing removed, and records of hyperbolic reflection
events.  The window layout of a batch depends on the case only, so every seed
has the same amount of work.

`exact` restates every propagator in 64 bits with plain torch: the staggered
derivatives are banded matrices, so an x derivative is D @ f and a z
derivative f @ D^T, and the adjoints of the plain Born maps come from
autograd.
"""
import math

import numpy as np
import torch

# Cells around the window that the eight-point stencils read but never update.
NOP = 4
F0 = 15.0          # Ricker peak frequency (Hz) of every workload
PML_RR = 1e-3      # reflection coefficient of the damping profile
RB_AMP, RB_SEED = 0.3, 1234   # random boundary of the library's defaults


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def _case(kind, nx, nz, shots, nt, **kw):
    c = dict(kind=kind, nx=nx, nz=nz, wmin=nx, wmax=nx, shots=shots, nt=nt, pml=20, boundary=0, dx=10.0, dt=0.0008)
    c.update(kw)
    return c


def listed():
    cases = [
        # One shot of a small model, untuned: a quick look at a model or a unit of a larger program;
        # every time step is shorter than a launch.
        dict(name="shot_forward_small", **_case("shot_forward", 101, 61, 1, 400)),
        # Plain elastic modelling of one shot on the 251x101 model, tile tuned once beforehand.
        dict(name="forward_251x101", **_case("forward", 251, 101, 1, 1000)),
        # The headline batch: 128 windows of 400-1200 columns on the 2000x600 model, tuned once.
        dict(name="forward_2000x600_128", **_case("forward", 2000, 600, 128, 200, wmin=400, wmax=1200, dx=12.5,
                                                   dt=0.001)),
        # The reference program's LSRTM gradient of a batch of shots (its main loop's work per iteration).
        dict(name="gradient_251x101_8", **_case("gradient", 251, 101, 8, 700)),
        # The same gradient shot by shot, as the reference's workers take it, with the random boundary.
        dict(name="shot_gradient_small", **_case("shot_gradient", 101, 61, 1, 400, boundary=1)),
        # Acoustic least-squares migration: 26 shots on 251x101, a few CG iterations.
        dict(name="lsrtm_cg_251x101_26", **_case("lsrtm_cg", 251, 101, 26, 500, pml=40, boundary=1, dt=0.0006,
                                                 niter=3)),
        # Reverse-time migration of 16 shots on 512x256 (one image of the learned preconditioner's training set).
        dict(name="born_adjoint_512x256_16", **_case("born_adjoint", 512, 256, 16, 300, pml=40, boundary=1)),
        # Elastic PP/PS Born modelling of uneven windows of the 4000x1000 model.
        dict(name="eborn_forward_4000x1000_16", **_case("eborn_forward", 4000, 1000, 16, 150, wmin=400, wmax=1200,
                                                        pml=40, boundary=1)),
        # Its adjoint with the background rebuilt by reversal, as surveys too long for a resident history run it.
        dict(name="eborn_adjoint_4000x1000_8", **_case("eborn_adjoint", 4000, 1000, 8, 150, wmin=400, wmax=1200,
                                                       pml=40, boundary=1, bg_mode=2)),
        # Elastic PP/PS least-squares migration on 512x256 with the resident history.
        dict(name="elsrtm_cg_512x256_8", **_case("elsrtm_cg", 512, 256, 8, 200, pml=40, boundary=1, niter=1)),
        # P/S-decoupled modelling of uneven windows.
        dict(name="rot_forward_2000x600_16", **_case("rot_forward", 2000, 600, 16, 200, wmin=400, wmax=1200, dx=12.5,
                                                     dt=0.001)),
        # One training gradient of the learned preconditioner at its training shape.
        dict(name="unet_gradient_512x256_8", kind="unet_gradient", nx=512, nz=256, batch=8, levels=4, base=32),
    ]
    return cases


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# cell-steps of one pass that a drawn case of a kind may cost
_MOST = {"shot_forward": 1e8, "forward": 1e10, "gradient": 2.4e8, "shot_gradient": 3e7, "lsrtm_cg": 8e8,
         "born_adjoint": 1.5e9, "eborn_forward": 2.5e9, "eborn_adjoint": 1.2e9, "elsrtm_cg": 6e8, "rot_forward": 2e9}


def draw(rng):
    kind = rng.choice(list(_MOST) + ["unet_gradient"])
    if kind == "unet_gradient":
        levels = rng.choice([3, 4])
        q = 2 ** (levels - 1)
        return dict(kind=kind, nx=q * _log(rng, 64 // q, 512 // q), nz=q * _log(rng, 48 // q, 256 // q),
                    batch=rng.randint(1, 8), levels=levels, base=32)
    single = kind in ("shot_forward", "shot_gradient")
    large = kind in ("forward", "eborn_forward", "eborn_adjoint", "rot_forward")
    nx = _log(rng, 80, 300 if single else 1200 if large else 520)
    nz = _log(rng, 50, 200 if single else 1000 if large else 260)
    shots = 1 if single else _log(rng, 1, 32)
    # the plain Born maps and their solvers need the random boundary
    either = kind in ("shot_forward", "forward", "gradient", "shot_gradient", "rot_forward")
    boundary = rng.choice([0, 0, 1]) if either else 1
    pml = 20 if boundary == 0 else rng.choice([20, 40])
    # the correlation residual of the gradient needs a signal on every trace
    nt = _log(rng, 350, 700) if kind.endswith("gradient") else _log(rng, 100, 400 if large else 600)
    cells = (nx + 2 * pml) * (nz + 2 * pml)
    shots = max(1, min(shots, int(_MOST[kind] / (cells * nt))))
    c = _case(kind, nx, nz, shots, nt, pml=pml, boundary=boundary)
    if not single and nx > 200:
        c["wmin"] = rng.randint(nx // 3, nx)
    if kind in ("lsrtm_cg", "elsrtm_cg"):
        c["niter"] = rng.randint(1, 2)
    if kind in ("eborn_adjoint", "born_adjoint"):
        c["bg_mode"] = rng.choice([0, 2])
    return c


# ---------------------------------------------------------------------------
# Inputs from the seed
# ---------------------------------------------------------------------------

def _ricker(nt, dt):
    """Ricker wavelet with its peak at sample 1 / (f0 dt)."""
    t = (np.arange(nt) - int(1.0 / (F0 * dt))) * dt
    a = (math.pi * F0 * t) ** 2
    return (np.exp(-a) * (1.0 - 2.0 * a)).astype(np.float32)


def _layers(rng, nx, nz):
    """Layered velocities of 2000-5500 m/s cut by one dipping fault."""
    edges = np.sort(rng.uniform(0.05, 0.95, int(rng.integers(8, 16)))) * nz
    vel = 2000.0 + 3500.0 * np.sort(rng.uniform(0.0, 1.0, edges.size + 1))
    z = np.arange(nz)[None, :].astype(np.float64)
    x = np.arange(nx)[:, None].astype(np.float64)
    fault = rng.uniform(0.3, 0.7) * nx + z / math.tan(math.radians(rng.uniform(60.0, 80.0)))
    depth = z - np.where(x > fault, int(rng.integers(3, 11)), 0)
    return vel[np.searchsorted(edges, depth, side="right")]


def _smooth(v):
    """9x9 Gaussian smoothing (sigma 2) with replicated edges."""
    k = np.exp(-0.5 * (np.arange(-4, 5) / 2.0) ** 2)
    k /= k.sum()
    p = np.pad(v, 4, mode="edge")
    a = sum(k[i] * p[i:i + v.shape[0]] for i in range(9))
    return sum(k[j] * a[:, j:j + v.shape[1]] for j in range(9))


def _windows(case):
    """Plain shot windows: start column, width, source column, receivers on every column of the window
    (gradients: on those that the slowest wave reaches within the record, as far traces hold no signal
    to correlate)."""
    rng = np.random.default_rng(case["nx"] + 7 * case["shots"])
    gradient = case["kind"] in ("gradient", "shot_gradient")
    reach = int((case["nt"] * case["dt"] - 0.1) * 2000.0 / case["dx"]) if gradient else case["nx"]
    out = []
    for i in range(case["shots"]):
        w = int(rng.integers(case["wmin"], case["wmax"] + 1))
        x0 = int(rng.integers(0, case["nx"] - w + 1))
        sx = w // 2 if w < case["nx"] else min(w - 1, int((i + 0.5) * w / case["shots"]))
        col = np.arange(w, dtype=np.int32)
        rec = col[np.abs(col - sx) <= reach] + np.int32(case["pml"])
        out.append(dict(x0=x0, nx=w, isx=case["pml"] + sx, isz=case["pml"] + 2, igz=case["pml"] + case["gz"],
                        rec=rec, shot_id=i))
    return out


def _events(rng, case, windows):
    """Records of hyperbolic reflections: [shot][trace][it], flat."""
    nt, dt = case["nt"], case["dt"]
    t = (np.arange(nt, dtype=np.float32) * np.float32(dt))[None, :]
    out = []
    for w in windows:
        off = (w["rec"] - w["isx"])[:, None].astype(np.float32) * np.float32(case["dx"])
        rec = np.zeros((w["rec"].size, nt), np.float32)
        for _ in range(4):
            t0, v = rng.uniform(0.1, 0.9) * nt * dt, rng.uniform(2000.0, 5000.0)
            te = np.sqrt(np.float32(t0 * t0) + (off / np.float32(v)) ** 2)
            a = (np.float32(math.pi * F0) * (t - te)) ** 2
            rec += np.float32(rng.uniform(-1.0, 1.0)) * np.exp(-a) * (1 - 2 * a)
        out.append(rec.ravel())
    return np.concatenate(out)


def _inputs(case, seed):
    """The arrays of a case, in the library's layout ([ix][iz] models, [trace][it] records)."""
    rng = np.random.default_rng([int(seed), case["nx"], case["nz"]])
    nx, nz = case["nx"], case["nz"]
    if case["kind"] == "unet_gradient":
        # an RTM image and a multi-iteration image, both of unit RMS
        def images():
            a = np.stack([np.diff(_layers(rng, nx, nz + 1), axis=1) for _ in range(case["batch"])])
            a = a + 20.0 * rng.standard_normal(a.shape)
            return (a / np.sqrt((a * a).mean(axis=(1, 2), keepdims=True))).astype(np.float32)
        theta = []
        for cin, cout, taps in _unet_layers(case):
            lim = math.sqrt(6.0 / (cin * taps))
            theta += [rng.uniform(-lim, lim, taps * cout * cin), 0.01 * rng.standard_normal(cout)]
        return dict(x=images(), t=images(), theta=np.concatenate(theta).astype(np.float32))
    case = dict(case, gz=1 if case["kind"].startswith("e") else 0)
    vp = _layers(rng, nx, nz)
    vs = vp / 1.73 * (1.0 + 0.1 * np.cos(np.arange(nz) / nz * rng.uniform(3.0, 9.0)))[None, :]
    d = dict(windows=_windows(case), wav=_ricker(case["nt"], case["dt"]))
    if case["kind"] not in ("shot_forward", "forward", "rot_forward"):
        vpm, vsm = _smooth(vp), _smooth(vs)
        d["pp"] = ((vp - vpm) / vpm).astype(np.float32)
        d["ps"] = ((vs - vsm) / vsm).astype(np.float32)
        vp, vs = vpm, vsm
    d["vp"], d["vs"] = vp.astype(np.float32), vs.astype(np.float32)
    d["rho"] = (310.0 * vp ** 0.25).astype(np.float32)
    if case["kind"] in ("gradient", "shot_gradient", "eborn_adjoint", "elsrtm_cg", "lsrtm_cg", "born_adjoint"):
        d["z"] = _events(rng, case, d["windows"])
        if case["kind"] not in ("lsrtm_cg", "born_adjoint"):
            d["x"] = _events(rng, case, d["windows"])
    return d


# ---------------------------------------------------------------------------
# One pass through the public entry points
# ---------------------------------------------------------------------------

def prepare(case, seed):
    from ds2d_amd.lib import ShotSpec, Solver, Unet
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "unet_gradient":
        u = Unet(levels=case["levels"], base=case["base"], max_batch=case["batch"], max_h=case["nx"],
                 max_w=case["nz"])
        u.set_params(d["theta"])
        return dict(kind=kind, unet=u, **d)
    acoustic = kind in ("lsrtm_cg", "born_adjoint")
    gradient = kind in ("gradient", "shot_gradient")
    s = Solver(dx=case["dx"], dz=case["dx"], dt=case["dt"], nt=case["nt"], allnx=case["nx"], allnz=case["nz"],
               pml=case["pml"], nx_max=case["wmax"], wavelet=d["wav"], physics=1 if acoustic else 0, pml_rr=PML_RR,
               rho_const=2000.0 if gradient else 0.0, rb_amp=RB_AMP, rb_seed=RB_SEED,
               bg_mode=case.get("bg_mode", 0))
    s.set_model(d["vp"], None if acoustic else d["vs"], None if gradient else d["rho"])
    if gradient:
        s.set_image(d["pp"], d["ps"])
    shots = [ShotSpec(w["x0"], w["nx"], w["isx"], w["isz"], w["igz"], w["rec"], shot_id=w["shot_id"],
                      boundary=case["boundary"]) for w in d["windows"]]
    if kind == "forward":
        s.autotune(shots, nsteps=min(40, case["nt"]))
    return dict(kind=kind, solver=s, shots=shots, niter=case.get("niter", 0), **d)


def run(state):
    kind = state["kind"]
    if kind == "unet_gradient":
        return state["unet"].loss_grad(state["x"], state["t"])
    s, shots = state["solver"], state["shots"]
    if kind == "shot_forward":
        s.set_shot(shots[0])
        return s.forward()
    if kind == "forward":
        return s.batch_forward(shots)[:2]
    if kind == "gradient":
        misfit = s.batch_gradient(shots, state["z"], state["x"], 1)
        return misfit, s.take_gradients()
    if kind == "shot_gradient":
        s.set_shot(shots[0], state["z"], state["x"])
        misfit = s.shot_gradient(1)
        return misfit, s.take_gradients()
    if kind == "lsrtm_cg":
        image, resid, _ = s.lsrtm_cg(shots, state["z"], state["niter"])
        return image, resid.tolist()
    if kind == "born_adjoint":
        return s.born_adjoint(shots, state["z"])[0]
    if kind == "eborn_forward":
        return s.eborn_forward(shots, state["pp"], state["ps"])[:2]
    if kind == "eborn_adjoint":
        return s.eborn_adjoint(shots, state["z"], state["x"])[:2]
    if kind == "elsrtm_cg":
        pp, ps, resid, _ = s.elsrtm_cg(shots, state["z"], state["x"], state["niter"])
        return pp, ps, resid.tolist()
    if kind == "rot_forward":
        return s.rot_forward(shots)[:2]
    raise ValueError(kind)


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

# floating-point operations of one cell and time step: derivatives (23 each: eight-point, odd symmetric), updates
_FLOPS = {"shot_forward": 8 * 23 + 30, "forward": 8 * 23 + 30, "rot_forward": 8 * 23 + 24,
          "gradient": 44 * 23 + 300, "shot_gradient": 44 * 23 + 300,   # 7 wavefields and 4 Born sources
          "eborn_forward": 16 * 23 + 90, "eborn_adjoint": 24 * 23 + 90, "elsrtm_cg": 8 * 23 + 40,
          "lsrtm_cg": 4 * 23 + 12, "born_adjoint": 12 * 23 + 30}


def _unet_layers(case):
    """(input channels, output channels, taps) of the network's layers, in parameter order."""
    ch = [case["base"] << k for k in range(case["levels"])]
    out = []
    for k in range(case["levels"]):
        out += [(ch[k - 1] if k else 1, ch[k], 9), (ch[k], ch[k], 9)]
    for k in range(case["levels"] - 2, -1, -1):
        out += [(ch[k] + ch[k + 1], ch[k], 9), (ch[k], ch[k], 9)]
    return out + [(ch[0], 1, 1)]


def work(case):
    if case["kind"] == "unet_gradient":
        pix = case["batch"] * case["nx"] * case["nz"]
        layers = _unet_layers(case)
        level = [k for k in range(case["levels"]) for _ in (0, 1)]
        level += [k for k in range(case["levels"] - 2, -1, -1) for _ in (0, 1)] + [0]
        # forward, data gradient and weight gradient: 2 operations a multiply-add each (the first layer has no data gradient)
        flops = sum((4 if i == 0 else 6) * ci * co * taps * pix / 4 ** k
                    for i, ((ci, co, taps), k) in enumerate(zip(layers, level)))
        theta = sum(ci * co * taps + co for ci, co, taps in layers)
        return dict(bytes=4.0 * (2 * pix + 2 * theta), flops=flops)
    kind = case["kind"]
    windows = _windows(dict(case, gz=0))
    cells = sum((w["nx"] + 2 * case["pml"]) * (case["nz"] + 2 * case["pml"]) for w in windows)
    rec = sum(w["rec"].size for w in windows) * case["nt"]
    model = case["nx"] * case["nz"]
    # Born and adjoint passes of the CG solvers: background, first residual, first gradient, two a step
    passes = 3 + 2 * case["niter"] if kind in ("lsrtm_cg", "elsrtm_cg") else 1
    arrays, records = {"gradient": (2 + 2 + 7, 2), "shot_gradient": (2 + 2 + 7, 2), "lsrtm_cg": (2 + 1, 1),
                       "born_adjoint": (2 + 1, 1), "eborn_forward": (3 + 2, 2), "eborn_adjoint": (3 + 2, 2),
                       "elsrtm_cg": (3 + 2, 2), "rot_forward": (2, 2)}.get(kind, (3, 2))
    return dict(bytes=4.0 * (arrays * model + records * rec), flops=float(_FLOPS[kind]) * cells * case["nt"] * passes)


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_device(), torch.float64)


class _Grid:
    """Staggered derivatives, medium and damping of one or several equal shot windows ([shot][x][z])."""

    def __init__(self, case, d, group):
        f32 = lambda v: float(np.float32(v))  # noqa: E731  (the library holds the geometry in 32 bits)
        self.dx, self.dt, self.pml = f32(case["dx"]), f32(case["dt"]), case["pml"]
        self.a = self.dt / self.dx
        self.group, self.d, self.nt, self.nz = group, d, case["nt"], case["nz"]
        p = case["pml"]
        self.nx = group[0]["nx"]
        nxp, nzp = self.nx + 2 * p, case["nz"] + 2 * p
        self.shape = (len(group), nxp, nzp)
        fx, bx = self._matrices(nxp)
        fz, bz = self._matrices(nzp)
        self.fx, self.bx, self.fz, self.bz = fx, bx, fz.t().contiguous(), bz.t().contiguous()
        # cells that are updated, and the physical window
        self.u = torch.zeros(nxp, nzp, dtype=torch.float64, device=_device())
        self.u[NOP:nxp - NOP, NOP:nzp - NOP] = 1.0
        self.core = torch.zeros_like(self.u)
        self.core[p:nxp - p, p:nzp - p] = 1.0
        vp, vs, rho, ex, ez = zip(*[self._medium(case, d, w) for w in group])
        self.vp, self.vs, self.rho = (torch.stack([_t(m) for m in v]) for v in (vp, vs, rho))
        self.mu = self.rho * self.vs ** 2
        self.lam = self.rho * (self.vp ** 2 - 2 * self.vs ** 2)
        # split damping: x' = (d1 x + increment) / d2
        ex, ez = torch.stack([_t(e) for e in ex]), torch.stack([_t(e) for e in ez])
        self.x1, self.x2 = 1 - self.dt * ex / 2, 1 / (1 + self.dt * ex / 2)
        self.z1, self.z2 = 1 - self.dt * ez / 2, 1 / (1 + self.dt * ez / 2)
        at = lambda k: torch.tensor([w[k] for w in group], device=_device())  # noqa: E731
        self.s, self.isx, self.isz = torch.arange(len(group), device=_device()), at("isx"), at("isz")
        self.rec = torch.arange(p, nxp - p, device=_device())
        self.ntr = torch.tensor([float(w["rec"].size) for w in group], device=_device(), dtype=torch.float64)
        self.igz = group[0]["igz"]
        self.wav = _t(d["wav"])

    @staticmethod
    def _matrices(n):
        """Forward and backward half-point derivatives (eighth order, unit spacing)."""
        f = np.zeros((n, n))
        for i, c in enumerate((1225.0 / 1024.0, -245.0 / 3072.0, 49.0 / 5120.0, -5.0 / 7168.0), 1):
            for r in range(NOP, n - NOP):
                f[r, r + i] += c
                f[r, r - i + 1] -= c
        b = np.zeros_like(f)
        b[NOP:n - NOP, :-1] = f[NOP:n - NOP, 1:]
        return _t(f), _t(b)

    @staticmethod
    def _medium(case, d, w):
        p, nx, nz = case["pml"], w["nx"], case["nz"]
        pad = lambda m: np.pad(m[w["x0"]:w["x0"] + nx], p, mode="edge")  # noqa: E731
        acoustic = case["kind"] in ("lsrtm_cg", "born_adjoint")
        gradient = case["kind"] in ("gradient", "shot_gradient")
        vp, vs = pad(d["vp"]), pad(d["vs"])
        vs = np.zeros_like(vp) if acoustic else vs
        rho = np.full_like(vp, 2000.0) if gradient else pad(d["rho"])
        ix, iz = np.meshgrid(np.arange(nx + 2 * p), np.arange(nz + 2 * p), indexing="ij")
        ex, ez = np.zeros(vp.shape), np.zeros(vp.shape)
        if case["boundary"]:
            frame = (ix < p) | (ix >= nx + p) | (iz < p) | (iz >= nz + p)
            fac = (1.0 + float(np.float32(RB_AMP)) * _hash(w["shot_id"], ix, iz)).astype(np.float32)
            ratio = vs / vp
            vp = np.where(frame, vp * fac, vp)
            vs = np.where(frame, ratio * vp, vs)
        else:
            base = math.log10(1.0 / float(np.float32(PML_RR))) * 5.0 * vp.astype(np.float64) / (2.0 * p)
            for e, i, n in ((ex, ix, nx + 2 * p), (ez, iz, nz + 2 * p)):
                depth = np.where(i < p, p - i, np.where(i > n - p, i - (n - p), 0)) / p
                e[:] = base * depth ** 4
        return vp, vs, rho, ex, ez

    def image(self, m, pad):
        """Image windows: replicated beyond the physical window (pad) or zero there."""
        p = self.pml
        return torch.stack([torch.nn.functional.pad(m[None, None, w["x0"]:w["x0"] + self.nx], (p,) * 4,
                                                    mode="replicate" if pad else "constant")[0, 0]
                            for w in self.group])

    def zeros(self, n):
        return [torch.zeros(self.shape, dtype=torch.float64, device=_device()) for _ in range(n)]

    def fdx(self, f): return self.fx @ f  # noqa: E704
    def bdx(self, f): return self.bx @ f  # noqa: E704
    def fdz(self, f): return f @ self.fz  # noqa: E704
    def bdz(self, f): return f @ self.bz  # noqa: E704

    def source(self, f, it):
        f[self.s, self.isx, self.isz] += self.wav[it]

    def record(self, f):
        return f[:, self.rec, self.igz]

    def traces(self, rows):
        """A list over time of [shot][trace] -> [shot][trace][it]."""
        return torch.stack(rows, dim=-1)

    def shots(self, flat):
        """The records of the group's shots on all columns, [shot][column][it] (zero where no receiver is)."""
        out = torch.zeros(len(self.group), self.nx, self.nt, dtype=torch.float64, device=_device())
        for o, w in zip(out, self.group):
            n = w["rec"].size * self.nt
            o[w["rec"] - self.pml] = flat[w["at"]:w["at"] + n].view(-1, self.nt)
        return out


def _hash(shot, ix, iz):
    """Uniform in [-1, 1) from the SplitMix64 hash of (seed, shot, cell)."""
    m = (1 << 64) - 1
    key = (np.uint64((RB_SEED * 0x100000001B3) & m) ^ np.uint64((shot << 42) & m) ^ (ix.astype(np.uint64) << np.uint64(21))
           ^ iz.astype(np.uint64))
    x = key + np.uint64(0x9E3779B97F4A7C15)
    x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    x = x ^ (x >> np.uint64(31))
    return 2.0 * ((x >> np.uint64(40)).astype(np.float64) / 16777216.0) - 1.0


class _Split:
    """Elastic wavefield with damped x and z parts of every component."""

    def __init__(self, g):
        self.vx, self.vz, self.xx, self.zz, self.xz = g.zeros(5)
        (self.vx1, self.vx2, self.vz1, self.vz2, self.xx1, self.xx2, self.zz1, self.zz2, self.xz1,
         self.xz2) = g.zeros(10)

    def velocity(self, g, sign=1.0, where=None):
        w = g.u if where is None else where
        c = sign * g.a * w / g.rho
        self._velocity(g, c * g.fdx(self.xx), c * g.bdz(self.xz), c * g.bdx(self.xz), c * g.fdz(self.zz), where)

    def _velocity(self, g, ax, az, bx, bz, where=None):
        for name, part, inc, k1, k2 in (("vx", 1, ax, g.x1, g.x2), ("vx", 2, az, g.z1, g.z2),
                                        ("vz", 1, bx, g.x1, g.x2), ("vz", 2, bz, g.z1, g.z2)):
            self._step(g, "%s%d" % (name, part), inc, k1, k2, where)
        self._sum(g, "vx", self.vx1 + self.vx2, where)
        self._sum(g, "vz", self.vz1 + self.vz2, where)

    def _step(self, g, name, inc, k1, k2, where):
        old = getattr(self, name)
        new = (k1 * old + inc) * k2
        setattr(self, name, new if where is None else torch.where(where > 0, new, old))

    def _sum(self, g, name, new, where):
        # the cells outside the update keep what they hold
        w = g.u if where is None else where
        setattr(self, name, torch.where(w > 0, new, getattr(self, name)))

    def strain(self, g):
        return g.bdx(self.vx), g.bdz(self.vz), g.fdz(self.vx), g.fdx(self.vz)

    def stress(self, g, sign=1.0, where=None):
        w = g.u if where is None else where
        dxx, dzz, dzx, dxz = self.strain(g)
        c = sign * g.a * w
        l2m = g.lam + 2 * g.mu
        for name, inc, k1, k2 in (("xx1", c * l2m * dxx, g.x1, g.x2), ("xx2", c * g.lam * dzz, g.z1, g.z2),
                                  ("zz1", c * g.lam * dxx, g.x1, g.x2), ("zz2", c * l2m * dzz, g.z1, g.z2),
                                  ("xz1", c * g.mu * dxz, g.x1, g.x2), ("xz2", c * g.mu * dzx, g.z1, g.z2)):
            self._step(g, name, inc, k1, k2, where)
        for k in ("xx", "zz", "xz"):
            self._sum(g, k, getattr(self, k + "1") + getattr(self, k + "2"), where)
        return dxx / g.dx, dzz / g.dx, dzx / g.dx, dxz / g.dx


def _forward(g):
    f, rz, rx = _Split(g), [], []
    for it in range(g.nt):
        g.source(f.xx, it)
        g.source(f.zz, it)
        f.velocity(g)
        f.stress(g)
        rz.append(g.record(f.vz))
        rx.append(g.record(f.vx))
    return g.traces(rz), g.traces(rx)


def _rot_forward(g):
    """Dilatation / rotation scheme: velocity parts driven by vp^2 grad(theta) and vs^2 curl(omega)."""
    th1, th2, om1, om2, px, pz, sx, sz, th, om = g.zeros(10)
    rz, rx = [], []
    for it in range(g.nt):
        g.source(th, it)
        p2, s2 = g.a * g.u * g.vp ** 2, g.a * g.u * g.vs ** 2
        px = (g.x1 * px + p2 * g.bdx(th)) * g.x2
        pz = (g.z1 * pz + p2 * g.bdz(th)) * g.z2
        sx = (g.x1 * sx + s2 * g.fdz(om)) * g.x2
        sz = (g.z1 * sz - s2 * g.fdx(om)) * g.z2
        vx, vz = px + sx, pz + sz
        c = g.a * g.u
        th1 = (g.x1 * th1 + c * g.fdx(vx)) * g.x2
        th2 = (g.z1 * th2 + c * g.fdz(vz)) * g.z2
        om1 = (g.x1 * om1 - c * g.bdx(vz)) * g.x2
        om2 = (g.z1 * om2 + c * g.bdz(vx)) * g.z2
        th, om = th1 + th2, om1 + om2
        rz.append(g.record(vz))
        rx.append(g.record(vx))
    return g.traces(rz), g.traces(rx)


def _born_source(g, e, b, dmp, dms):
    """Born source of the images on the physical window, into the stresses of b."""
    exx, ezz, ezx, exz = (v / g.dx for v in e)
    l2m, w = g.lam + 2 * g.mu, g.core
    p = -l2m * dmp
    q = p + 2 * g.mu * dms
    b.xx = b.xx + w * 2 * (p * exx + q * ezz)
    b.zz = b.zz + w * 2 * (q * exx + p * ezz)
    b.xz = b.xz - w * 2 * g.mu * dms * (exz + ezx)


def _adjoint_velocity(g, f):
    """Receiver-side velocity: moduli inside the derivatives, stepped backwards."""
    l2m, c = g.lam + 2 * g.mu, -g.a * g.u / g.rho
    f._velocity(g, c * (g.fdx(l2m * f.xx) + g.fdx(g.lam * f.zz)), c * g.bdz(g.mu * f.xz), c * g.bdx(g.mu * f.xz),
                c * (g.fdz(l2m * f.zz) + g.fdz(g.lam * f.xx)))


def _adjoint_stress(g, f):
    dxx, dzz, dzx, dxz = f.strain(g)
    c = -g.a * g.u
    for name, inc, k1, k2 in (("xx1", c * dxx, g.x1, g.x2), ("zz2", c * dzz, g.z1, g.z2),
                              ("xz1", c * dxz, g.x1, g.x2), ("xz2", c * dzx, g.z1, g.z2)):
        f._step(g, name, inc, k1, k2, None)
    f._sum(g, "xx", f.xx1, None)
    f._sum(g, "zz", f.zz2, None)
    f._sum(g, "xz", f.xz1 + f.xz2, None)


def _adjoint_source(g, s, f, dmp, dms):
    """Receiver-side Born source: into the velocities of f on the physical window, backwards."""
    cp = -2 * (g.lam + 2 * g.mu) * dmp
    cx = cp + 4 * g.mu * dms
    cs = -2 * g.mu * dms
    w = -g.core / (g.rho * g.dx)
    # the reference weights both taps of the x derivative of txz with the modulus of the upper one
    odd = torch.zeros_like(s.xz)
    c8 = (1225.0 / 1024.0, -245.0 / 3072.0, 49.0 / 5120.0, -5.0 / 7168.0)
    n = s.xz.shape[1]
    for i, c in enumerate(c8, 1):
        hi = slice(NOP + i - 1, n - NOP + i - 1)
        lo = slice(NOP - i, n - NOP - i)
        odd[:, NOP:n - NOP] += c * cs[:, hi] * (s.xz[:, hi] - s.xz[:, lo])
    f.vx = f.vx + w * (g.fdx(cp * s.xx) + g.fdx(cx * s.zz) + g.bdz(cs * s.xz))
    f.vz = f.vz + w * (g.fdz(cp * s.zz) + g.fdz(cx * s.xx) + odd)


def _gradient(g, case):
    """The reference program's gradient of a group of shots: (misfit, seven window images)."""
    d, p = g.d, g.pml
    dmp, dms = g.image(_t(d["pp"]), True), g.image(_t(d["ps"]), True)
    bg, b, b2, bk, bb = (_Split(g) for _ in range(5))
    rows, kept = ([], []), []
    n, m = g.shape[1:]
    ix, iz = torch.arange(n, device=_device())[:, None], torch.arange(m, device=_device())[None, :]
    inx, inz = (ix >= p) & (ix < n - p), (iz >= p) & (iz < m - p)
    band = (inx & ((iz >= p - NOP) & (iz < p + NOP) | (iz >= m - p - NOP) & (iz < m - p + NOP))
            | inz & ((ix >= p - NOP) & (ix < p + NOP) | (ix >= n - p - NOP) & (ix < n - p + NOP)))
    pml = case["boundary"] == 0
    for it in range(g.nt):
        g.source(bg.xx, it)
        g.source(bg.zz, it)
        bg.velocity(g)
        bg.stress(g)
        _born_source(g, bg.strain(g), b, dmp, dms)
        b.velocity(g)
        b.stress(g)
        _born_source(g, b.strain(g), b2, dmp, dms)
        b2.velocity(g)
        b2.stress(g)
        rows[0].append(g.record(b.vz) + g.record(b2.vz))
        rows[1].append(g.record(b.vx) + g.record(b2.vx))
        if pml:
            kept.append((bg.vx, bg.vz, b.vx, b.vz))
    misfit, res = 0.0, []
    for syn, obs in ((g.traces(rows[0]), g.shots(_t(d["z"]))), (g.traces(rows[1]), g.shots(_t(d["x"])))):
        ss, oo, so = (syn * syn).sum(-1), (obs * obs).sum(-1), (syn * obs).sum(-1)
        live = (ss > 0) & (oo > 0)
        a = torch.where(live, 1 / torch.sqrt(torch.where(live, ss * oo, 1.0)), 0.0)
        misfit -= float(((so * a).sum(-1) / (2 * g.ntr)).sum())
        res.append(a[..., None] * (torch.where(live, so / torch.where(live, ss, 1.0), 0.0)[..., None] * syn - obs))
    out = [torch.zeros(g.shape, dtype=torch.float64, device=_device()) for _ in range(7)]
    kp, ks = -2 * g.vp ** 2 * g.rho, -2 * g.vs ** 2 * g.rho

    def image(e, f, pp, ps):
        exx, ezz, ezx, exz = e
        out[pp] += kp * (exx + ezz) * (f.xx + f.zz)
        out[ps] += ks * (-2 * (exx * f.zz + ezz * f.xx) + (ezx + exz) * f.xz)

    for it in range(g.nt - 1, -1, -1):
        if pml:
            bg.vx, bg.vz, b.vx, b.vz = (torch.where(band, k, f) for k, f in
                                        zip(kept.pop(), (bg.vx, bg.vz, b.vx, b.vz)))
        eg = bg.stress(g, -1.0, g.core)
        bg.velocity(g, -1.0, g.core)
        eb = b.stress(g, -1.0, g.core)
        _born_source(g, bg.strain(g), b, dmp, dms)
        b.velocity(g, -1.0, g.core)
        bk.vz = bk.vz.clone()
        bk.vx = bk.vx.clone()
        bk.vz[:, g.rec, g.igz] += res[0][..., it]
        bk.vx[:, g.rec, g.igz] += res[1][..., it]
        _adjoint_stress(g, bk)
        _adjoint_velocity(g, bk)
        _adjoint_velocity(g, bb)
        _adjoint_source(g, bk, bb, dmp, dms)
        _adjoint_stress(g, bb)
        image(eg, bk, 0, 1)
        image(eb, bk, 3, 4)
        image(eg, bb, 5, 6)
        out[2] += bg.vx ** 2 + bg.vz ** 2
    return misfit, [o[:, p:-p, p:-p] for o in out]


class _Acoustic:
    """Linear acoustic Born map of a group: background increments kept per step."""

    def __init__(self, g):
        self.g = g
        self.b, self.k = g.a * g.u / g.rho, g.a * g.u * g.rho * g.vp ** 2
        vx, vz, p = g.zeros(3)
        self.dp = []
        for it in range(g.nt):
            q = p.clone()
            g.source(q, it)
            vx, vz = vx + self.b * g.fdx(q), vz + self.b * g.fdz(q)
            self.dp.append(self.k * (g.bdx(vx) + g.bdz(vz)))
            p = p + self.dp[-1]

    def __call__(self, refl):
        g, m = self.g, 2 * self.g.image(refl, False)
        vx, vz, p = g.zeros(3)
        rows = []
        for it in range(g.nt):
            vx, vz = vx + self.b * g.fdx(p), vz + self.b * g.fdz(p)
            p = p + self.k * (g.bdx(vx) + g.bdz(vz)) + m * self.dp[it]
            rows.append(g.record(p))
        return [g.traces(rows)]


class _Elastic:
    """Linear elastic PP/PS Born map of a group: background strains kept per step."""

    def __init__(self, g):
        self.g, self.e = g, []
        f = g.zeros(5)
        for it in range(g.nt):
            q = [f[0], f[1], f[2].clone(), f[3].clone(), f[4]]
            g.source(q[2], it)
            g.source(q[3], it)
            v = self._velocity(q)
            e = self._strain(v)
            f = v + self._stress(f[2:], e)
            self.e.append([k * g.core for k in (e[0], e[1], e[2] + e[3])])

    def _velocity(self, f):
        g = self.g
        c = g.a * g.u / g.rho
        return [f[0] + c * (g.fdx(f[2]) + g.bdz(f[4])), f[1] + c * (g.bdx(f[4]) + g.fdz(f[3]))]

    def _strain(self, v):
        g = self.g
        return g.bdx(v[0]), g.bdz(v[1]), g.fdz(v[0]), g.fdx(v[1])

    def _stress(self, s, e):
        g = self.g
        c, l2m = g.a * g.u, g.lam + 2 * g.mu
        return [s[0] + c * (l2m * e[0] + g.lam * e[1]), s[1] + c * (g.lam * e[0] + l2m * e[1]),
                s[2] + c * g.mu * (e[2] + e[3])]

    def __call__(self, pp, ps):
        g = self.g
        p = -2 * (g.lam + 2 * g.mu) / g.dx * g.image(pp, False)
        s = -2 * g.mu / g.dx * g.image(ps, False)
        q = p - 2 * s
        f, rz, rx = g.zeros(5), [], []
        for it in range(g.nt):
            v = self._velocity(f)
            f = v + self._stress(f[2:], self._strain(v))
            exx, ezz, exz = self.e[it]
            f = v + [f[2] + p * exx + q * ezz, f[3] + q * exx + p * ezz, f[4] + s * exz]
            rz.append(g.record(f[1]))
            rx.append(g.record(f[0]))
        return [g.traces(rz), g.traces(rx)]


class _Map:
    """A Born map over all groups: images -> flat records, and its transpose."""

    def __init__(self, case, d, kind):
        self.maps = [kind(g) for g in _groups(case, d)]
        self.rec = sum(w["rec"].size for w in d["windows"]) * case["nt"]

    def __call__(self, *images):
        out = None
        for m in self.maps:
            got = m(*images)
            out = out or [torch.zeros(self.rec, dtype=torch.float64, device=_device()) for _ in got]
            for o, r in zip(out, got):
                for k, w in enumerate(m.g.group):
                    o[w["at"]:w["at"] + r[k].numel()] = r[k].reshape(-1)
        return out

    def transpose(self, shape, n, res):
        total = [torch.zeros(shape, dtype=torch.float64, device=_device()) for _ in range(n)]
        for m in self.maps:
            x = [torch.zeros_like(t).requires_grad_() for t in total]
            got = m(*x)
            for t, v in zip(total, torch.autograd.grad(got, x, [m.g.shots(r) for r in res])):
                t += v
        return total


def _groups(case, d):
    """The windows of a batch, those of one width together."""
    at = 0
    for w in d["windows"]:
        w["at"] = at
        at += w["rec"].size * case["nt"]
    width = {}
    for w in d["windows"]:
        width.setdefault(w["nx"], []).append(w)
    return (_Grid(case, d, ws) for ws in width.values())


def _cgls(born, shape, n, data, niter):
    dot = lambda a, b: float(sum((x * y).sum() for x, y in zip(a, b)))  # noqa: E731
    x = [torch.zeros(shape, dtype=torch.float64, device=_device()) for _ in range(n)]
    r = [v.clone() for v in data]
    dd = dot(r, r)
    resid = [1.0]
    s = born.transpose(shape, n, r)
    p, gamma = s, dot(s, s)
    for _ in range(niter):
        q = born(*p)
        alpha = gamma / dot(q, q)
        x = [a + alpha * b for a, b in zip(x, p)]
        r = [a - alpha * b for a, b in zip(r, q)]
        resid.append(math.sqrt(dot(r, r) / dd))
        s = born.transpose(shape, n, r)
        gamma, old = dot(s, s), gamma
        p = [a + gamma / old * b for a, b in zip(s, p)]
    return x, resid


def _unet_gradient(case, d):
    theta = _t(d["theta"]).requires_grad_()
    parts, at = [], 0
    for cin, cout, taps in _unet_layers(case):
        w = theta[at:at + taps * cout * cin].view(taps, cout, cin)
        at += w.numel()
        parts.append((w, theta[at:at + cout]))
        at += cout
    layers = iter(parts)

    def conv(x):
        w, b = next(layers)
        h, v = x.shape[1:3]
        p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
        y = sum(p[:, k // 3:k // 3 + h, k % 3:k % 3 + v] @ w[k].t() for k in range(9))
        return torch.relu(y + b)

    def up(x):
        return x.repeat_interleave(2, 1).repeat_interleave(2, 2)

    x, skips = _t(d["x"])[..., None], []
    for k in range(case["levels"]):
        if k:
            n, h, v, c = x.shape
            x = x.view(n, h // 2, 2, v // 2, 2, c).mean((2, 4))
        x = conv(conv(x))
        skips.append(x)
    for k in range(case["levels"] - 2, -1, -1):
        x = conv(conv(torch.cat([skips[k], up(x)], -1)))
    w, b = next(layers)
    loss = ((x @ w[0].t() + b)[..., 0] - _t(d["t"])).square().mean()
    return float(loss.detach()), torch.autograd.grad(loss, theta)[0]


def exact(case, seed):
    kind, d = case["kind"], _inputs(case, seed)
    shape = (case["nx"], case["nz"])
    if kind == "unet_gradient":
        loss, g = _unet_gradient(case, d)
        return loss, g.cpu()
    if kind in ("shot_forward", "forward", "rot_forward"):
        n = sum(w["rec"].size for w in d["windows"]) * case["nt"]
        rz, rx = np.zeros(n), np.zeros(n)
        for g in _groups(case, d):
            for out, r in zip((rz, rx), (_rot_forward if kind == "rot_forward" else _forward)(g)):
                for k, w in enumerate(g.group):
                    out[w["at"]:w["at"] + r[k].numel()] = r[k].reshape(-1).cpu().numpy()
        return rz, rx
    if kind in ("gradient", "shot_gradient"):
        misfit, images = 0.0, [np.zeros(shape) for _ in range(7)]
        for g in _groups(case, d):
            m, win = _gradient(g, case)
            misfit += m
            for im, v in zip(images, win):
                for k, w in enumerate(g.group):
                    im[w["x0"]:w["x0"] + w["nx"]] += v[k].cpu().numpy()
        return misfit, images
    data = [_t(d[k]) for k in ("z", "x") if k in d]
    if kind == "born_adjoint":
        return _Map(case, d, _Acoustic).transpose(shape, 1, data)[0].cpu()
    if kind == "lsrtm_cg":
        x, resid = _cgls(_Map(case, d, _Acoustic), shape, 1, data, case["niter"])
        return x[0].cpu(), resid
    if kind == "eborn_forward":
        return tuple(r.cpu() for r in _Map(case, d, _Elastic)(_t(d["pp"]), _t(d["ps"])))
    if kind == "eborn_adjoint":
        return tuple(r.cpu() for r in _Map(case, d, _Elastic).transpose(shape, 2, data))
    if kind == "elsrtm_cg":
        x, resid = _cgls(_Map(case, d, _Elastic), shape, 2, data, case["niter"])
        return x[0].cpu(), x[1].cpu(), resid
    raise ValueError(kind)
