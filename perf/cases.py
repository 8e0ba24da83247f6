"""The work that programs have this framework do, as timed cases.

Families (``"do"``):

  dropin      one step of a sample-style script: physics and integrator
              classes, ``RK2mid.do_advance``
  step        one RK2 step of ``_hip.Plan.step`` (plain 2D and 3D grids, and
              batched 2D ensembles), state resident on the GPU
  transforms  the backward transforms of several fields and the forward
              transforms of the results (the per-operation path, analysis
              and pair generation)
  closure     steps of a coarse run corrected by the learned closure
  infer       the closure network's inference pass on a batch of images
  train       forward and backward of the closure network on a batch

Grid extents are 2^a 3^b 5^c (even along x), as the plans take them.  Every
input is made on the GPU from the seed.  ``exact`` repeats a case with
torch's transforms in double precision, in convective form, on the full
half-spectrum layout.
"""

import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "dedalus-1.0_amd"))

TWO_PI = 2.0 * math.pi
NU, KAPPA, ETA, RHO0 = 1e-3, 2e-3, 1.5e-3, 1.0


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # a sample script on a small grid (the 64^2 Taylor-Green setup): host
        # work, launches and latency
        dict(name="dropin_hydro2d_64", do="dropin", physics="hydro", ny=64, nx=64),
        # one 2D convection run, integrated over many small steps
        dict(name="step_boussinesq2d_512", do="step", physics="boussinesq", nz=0, ny=512, nx=512,
             batch=0, f32=False, integrator="RK2mid"),
        # 2D MHD on a box that is no power of two, trapezoidal integrator
        dict(name="step_mhd2d_360x450", do="step", physics="mhd", nz=0, ny=360, nx=450, batch=0,
             f32=False, integrator="RK2trap"),
        # one size class of an FP32 ensemble
        dict(name="step_ensemble_256x128", do="step", physics="hydro", nz=0, ny=128, nx=128,
             batch=256, f32=True, integrator="RK2mid"),
        # 3D turbulence, FP32 and FP64
        dict(name="step_hydro3d_128_f32", do="step", physics="hydro", nz=128, ny=128, nx=128,
             batch=0, f32=True, integrator="RK2mid"),
        dict(name="step_hydro3d_192", do="step", physics="hydro", nz=192, ny=192, nx=192,
             batch=0, f32=False, integrator="RK2mid"),
        # 3D convection in a flat box with unequal, ragged extents
        dict(name="step_boussinesq3d_75x96x120", do="step", physics="boussinesq", nz=75, ny=96,
             nx=120, batch=0, f32=False, integrator="RK2mid"),
        # the largest run: 3D MHD turbulence
        dict(name="step_mhd3d_256", do="step", physics="mhd", nz=256, ny=256, nx=256, batch=0,
             f32=False, integrator="RK2mid"),
        # the fields of a 3D velocity to x space and back
        dict(name="transforms_3x160x144x180", do="transforms", nz=160, ny=144, nx=180, batch=0,
             nf=3, f32=False),
        # ten coarse steps with the learned closure, as a run replays them
        dict(name="closure_64_ten_steps", do="closure", members=0),
        # the network on a batch of coarse states
        dict(name="infer_256x64", do="infer", members=256, h=64, w=64),
        # one training batch (the pipeline's batch size)
        dict(name="train_32x64", do="train", members=32, h=64, w=64),
    ]


def _smooth(lo, hi, even):
    out = []
    for n in range(lo, hi + 1):
        m = n
        for p in (2, 3, 5):
            while m % p == 0:
                m //= p
        if m == 1 and not (even and n % 2):
            out.append(n)
    return out


def _extent(rng, lo, hi, even=False):
    """An admissible extent, its logarithm spread evenly over [lo, hi]."""
    x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(_smooth(lo, hi, even), key=lambda n: abs(n - x))


def draw(rng):
    kind = rng.choice(["step2d", "step2d", "step2d", "step3d", "step3d", "step3d", "ensemble",
                       "ensemble", "transforms", "transforms", "dropin", "infer", "train"])
    phys = rng.choice(["hydro", "boussinesq", "mhd"])
    integ = rng.choice(["RK2mid", "RK2trap"])
    f32 = rng.random() < 0.3
    if kind == "dropin":
        return dict(do="dropin", physics=phys, ny=_extent(rng, 30, 512), nx=_extent(rng, 30, 512, True))
    if kind == "step2d":
        return dict(do="step", physics=phys, nz=0, ny=_extent(rng, 30, 640), nx=_extent(rng, 30, 640, True),
                    batch=0, f32=f32, integrator=integ)
    if kind == "ensemble":
        ny, nx = _extent(rng, 30, 256), _extent(rng, 30, 256, True)
        most = max(2, min(300, int(4e6 / (ny * nx))))
        return dict(do="step", physics=phys, nz=0, ny=ny, nx=nx, f32=rng.random() < 0.7,
                    batch=int(round(math.exp(rng.uniform(math.log(2), math.log(most))))), integrator=integ)
    if kind == "step3d":
        nz, ny, nx = (_extent(rng, 24, 256, even) for even in (False, False, True))
        return dict(do="step", physics=phys, nz=nz, ny=ny, nx=nx, batch=0, f32=f32, integrator=integ)
    if kind == "transforms":
        nf = rng.randint(1, 6)
        if rng.random() < 0.4:
            return dict(do="transforms", nz=0, ny=_extent(rng, 30, 640), nx=_extent(rng, 30, 640, True),
                        batch=0, nf=nf, f32=f32)
        nz, ny, nx = (_extent(rng, 24, 256, even) for even in (False, False, True))
        return dict(do="transforms", nz=nz, ny=ny, nx=nx, batch=0, nf=nf, f32=f32)
    h, w = rng.choice([32, 64, 96, 128]), rng.choice([32, 64, 128])
    if kind == "infer":
        m = int(round(math.exp(rng.uniform(0.0, math.log(256)))))
        return dict(do="infer", members=min(m, 256 * 4096 // (h * w)), h=h, w=w)
    return dict(do="train", members=min(rng.randint(4, 64), 64 * 4096 // (h * w)), h=h, w=w)


# ---------------------------------------------------------------------------
# grids, layouts and inputs (nothing of the framework: shared by exact)
# ---------------------------------------------------------------------------

def _kept(n):
    """Largest |index| of the 2/3 rule |k| < (2/3) k_Nyquist on n points of a 2 pi box."""
    kny = math.pi * n / TWO_PI
    thr = 2.0 / 3.0 * kny
    c = 0
    while c + 1 <= n // 2 and ((c + 1) * (1.0 / n)) * 2.0 * kny < thr:
        c += 1
    return c


class _Grid:
    """Wavenumbers and the 2/3 mask of a half-spectrum grid (2D with a leading
    member axis, or 3D), and the compact layout (Ky, Kz or members, padded kx)."""

    def __init__(self, case):
        self.nz, self.ny, self.nx = case.get("nz", 0), case["ny"], case["nx"]
        self.three = self.nz > 0
        self.nd = 3 if self.three else 2
        self.lead = self.nz if self.three else max(1, case.get("batch", 0))
        self.dims = (-3, -2, -1) if self.three else (-2, -1)
        self.shape = (self.lead, self.ny, self.nx)          # x space
        self.size = (self.nz, self.ny, self.nx) if self.three else (self.ny, self.nx)
        dev = torch.device("cuda")

        def full(n):
            m = torch.arange(n, device=dev, dtype=torch.float64)
            return torch.where(m < (n - 1) // 2 + 1, m, m - n)

        kx = torch.arange(self.nx // 2 + 1, device=dev, dtype=torch.float64)
        ky = full(self.ny)
        kz = full(self.nz) if self.three else torch.zeros(1, device=dev, dtype=torch.float64)
        self.cx, self.cy = _kept(self.nx), _kept(self.ny)
        self.cz = _kept(self.nz) if self.three else 0
        keep = (kx <= self.cx).view(1, 1, -1) & (ky.abs() <= self.cy).view(1, -1, 1)
        if self.three:
            keep = keep & (kz.abs() <= self.cz).view(-1, 1, 1)
        self.keep = keep
        self.k = [kx.view(1, 1, -1), ky.view(1, -1, 1), kz.view(-1, 1, 1)]
        self.k2 = self.k[0] ** 2 + self.k[1] ** 2 + self.k[2] ** 2
        self.k2n = torch.where(self.k2 == 0, torch.ones_like(self.k2), self.k2)
        self.kxp = (self.cx + 1 + 7) // 8 * 8

        def rows(n, c):
            return torch.cat([torch.arange(c + 1, device=dev), torch.arange(n - c, n, device=dev)])

        self.ry = rows(self.ny, self.cy)
        self.rz = rows(self.nz, self.cz) if self.three else torch.arange(self.lead, device=dev)
        self.npts = self.lead * self.ny * self.nx
        self.nkc = self.ry.numel() * self.rz.numel() * self.kxp

    def pack(self, a, dtype):
        """Half-spectrum array (lead, ky, kx) -> compact array."""
        s = a.index_select(0, self.rz).index_select(1, self.ry)[:, :, :self.cx + 1].transpose(0, 1)
        out = torch.zeros((self.ry.numel(), self.rz.numel(), self.kxp), dtype=dtype, device=a.device)
        out[:, :, :self.cx + 1] = s.to(dtype)
        return out.reshape(-1)

    def unpack(self, c):
        s = c.reshape(self.ry.numel(), self.rz.numel(), self.kxp).to(torch.complex128)
        out = torch.zeros((self.lead, self.ny, self.nx // 2 + 1), dtype=torch.complex128, device=c.device)
        out[self.rz.view(-1, 1), self.ry.view(1, -1), :self.cx + 1] = s[:, :, :self.cx + 1].transpose(0, 1)
        return out

    def fwd(self, x):
        return torch.fft.rfftn(x, dim=self.dims, norm="forward") * self.keep

    def bwd(self, k):
        return torch.fft.irfftn(k, s=self.size, dim=self.dims, norm="forward")

    def d(self, k, axis):
        return 1j * self.k[axis] * k

    def project(self, f):
        kf = sum(self.k[i] * f[i] for i in range(self.nd))
        return [f[i] - self.k[i] * (kf / self.k2n) for i in range(self.nd)]


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 13)
    return g


def _random_scalar(grid, gen, rms):
    """A smooth random field: white noise with a Gaussian envelope in k."""
    x = torch.randn(grid.shape, generator=gen, device="cuda", dtype=torch.float64)
    k0 = max(2.0, min(grid.cx, grid.cy, grid.cz if grid.three else grid.cy) / 4.0)
    a = torch.fft.rfftn(x, dim=grid.dims, norm="forward") * grid.keep * torch.exp(-grid.k2 / (k0 * k0))
    a = torch.where(grid.k2 == 0, torch.zeros_like(a), a)
    return a * (rms / grid.bwd(a).square().mean().sqrt())


def _random_vector(grid, gen, rms):
    """A solenoidal vector field."""
    v = grid.project([_random_scalar(grid, gen, 1.0) for _ in range(grid.nd)])
    s = sum(grid.bwd(a).square().mean() for a in v).sqrt()
    return [a * (rms / s) for a in v]


def _random_state(case, grid, seed):
    """Compact state arrays of a physics, in the plan's precision."""
    gen = _gen(seed)
    dt = torch.complex64 if case.get("f32") else torch.complex128
    f = _random_vector(grid, gen, 1.0)
    if case["physics"] == "boussinesq":
        f.append(_random_scalar(grid, gen, 0.1))
    elif case["physics"] == "mhd":
        f += _random_vector(grid, gen, 0.5)
    return [grid.pack(a, dt) for a in f]


def _dt(case):
    """A time step well inside the advective stability limit at |u| = 4."""
    return 0.06 / max(case["nx"], case["ny"], case.get("nz", 0))


def _nstate(case, nd):
    return {"hydro": nd, "boussinesq": nd + 1, "mhd": 2 * nd}[case["physics"]]


def _random_weights(seed, chans):
    """Weights and biases of a network in training: He-scaled weights, small biases."""
    gen = torch.Generator().manual_seed(int(seed) * 31 + 5)
    ws, bs = [], []
    for ci, co in zip(chans[:-1], chans[1:]):
        ws.append(torch.randn(co, ci, 3, 3, generator=gen) * math.sqrt(2.0 / (9 * ci)))
        bs.append(torch.randn(co, generator=gen) * 0.1)
    return ws, bs


CHANS = (3, 32, 32, 32, 32, 2)


def _images(case, seed, channels):
    gen = _gen(seed)
    return torch.randn((case["members"], case["h"], case["w"], channels), generator=gen, device="cuda")


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------

_STREAM = None


def _stream():
    """The stream that a program runs its plans on."""
    global _STREAM
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
    return _STREAM


class _View:
    """A device buffer of the framework as an array that torch can wrap."""

    def __init__(self, buf, n, keep=None):
        self.buf, self.keep = buf, keep
        self.__cuda_array_interface__ = dict(shape=(int(n), 2), typestr="<f8", data=(int(buf), False),
                                             version=3, strides=None)


def _view(buf, n):
    return torch.as_tensor(_View(buf, n), device="cuda")


def _ptrs(ts):
    return [t.data_ptr() for t in ts]


def _params(case, nd):
    from dedalus import _hip
    phys = {"hydro": _hip.HYDRO, "boussinesq": _hip.BOUSSINESQ, "mhd": _hip.MHD}[case["physics"]]
    return _hip.make_params(phys, nu=NU, kappa=KAPPA, eta=ETA, rho0=RHO0, bdir=nd - 1)


def _plan(case, grid):
    from dedalus import _hip
    length = (TWO_PI,) * grid.nd
    prec = _hip.F32 if case.get("f32") else _hip.F64
    batch = case.get("batch", 0)
    plan = _hip.Plan(grid.size, length, prec, batch=batch) if batch else _hip.Plan(grid.size, length, prec)
    plan.set_stream(_stream().cuda_stream)
    return plan


def prepare(case, seed):
    return _PREPARE[case["do"]](case, seed)


def _prepare_step(case, seed):
    grid = _Grid(case)
    y = _random_state(case, grid, seed)
    stage, d1 = ([torch.zeros_like(a) for a in y] for _ in range(2))
    return dict(case=case, plan=_plan(case, grid), prm=_params(case, grid.nd), y=y, stage=stage, d1=d1,
                dt=_dt(case))


def _prepare_dropin(case, seed):
    import logging
    from dedalus.config import decfg
    decfg.set("utils", "loglevel", "warning")
    logging.getLogger("Dedalus").setLevel(logging.WARNING)
    import dedalus.mods as m
    cls = {"hydro": m.IncompressibleHydro, "boussinesq": m.BoussinesqHydro,
           "mhd": m.IncompressibleMHD}[case["physics"]]
    grid = _Grid(case)
    rhs = cls((case["ny"], case["nx"]), m.FourierRepresentation)
    p = {"nu": NU}
    if case["physics"] == "boussinesq":
        p.update(kappa=KAPPA, boussinesq_direction="y", g=1., alpha_t=1., beta=1.)
    elif case["physics"] == "mhd":
        p.update(eta=ETA, rho0=RHO0)
    rhs.parameters.update(p)
    data = rhs.create_fields(0.)
    comps = [c for _, field in data for _, c in field]
    for c, a in zip(comps, _random_state(case, grid, seed)):
        # a script sets k space in the reference's (kx, ky) layout
        c["kspace"] = grid.unpack(a)[0].transpose(0, 1).contiguous().cpu().numpy()
    ti = m.RK2mid(rhs)
    return dict(case=case, rhs=rhs, data=data, ti=ti, comps=comps, dt=_dt(case), nkc=grid.nkc)


def _prepare_transforms(case, seed):
    grid = _Grid(case)
    gen = _gen(seed)
    dt = torch.complex64 if case["f32"] else torch.complex128
    kc = [grid.pack(_random_scalar(grid, gen, 1.0), dt) for _ in range(case["nf"])]
    rt = torch.float32 if case["f32"] else torch.float64
    return dict(case=case, plan=_plan(case, grid), kc=kc, out=[torch.zeros_like(a) for a in kc],
                x=[torch.empty(grid.npts, dtype=rt, device="cuda") for _ in kc])


def _net(seed):
    from dedalus.closure import ClosureNet
    net = ClosureNet(cin=CHANS[0], cout=CHANS[-1], width=32, depth=5, seed=0)
    with torch.no_grad():
        for p, v in zip(list(net.weights) + list(net.biases), sum(_random_weights(seed, CHANS), [])):
            p.copy_(v)
    return net.cuda()


def _prepare_infer(case, seed):
    from dedalus.closure.net import Inference
    net = _net(seed)
    inf = Inference(net, case["members"], case["h"], case["w"])
    inf.x[:, :3] = _images(case, seed, 3).reshape(-1, 3).to(torch.bfloat16)
    return dict(case=case, inf=inf, net=net)


def _prepare_train(case, seed):
    return dict(case=case, net=_net(seed), x=_images(case, seed, 3), y=_images(case, seed + 1, 2))


_PIPE = None


def _prepare_closure(case, seed):
    """A coarse 64^2 run of the 512^2 -> 64^2 configuration (the pipeline is a
    program's one setup object) with its own network and state."""
    global _PIPE
    from dedalus.closure import pipeline as P
    if _PIPE is None:
        _PIPE = P.Pipeline(dict(P.CLOSURE_512_64), stream=_stream())
    net = _net(seed)
    # a tendency of rms about 0.01: weak enough for thousands of steps
    scales = (np.array([0.7, 0.7, 4.0]), np.array([0.01, 0.01]))
    run_ = _PIPE.coarse_run(net, scales, batch=case["members"] or None)
    grid = _Grid(dict(ny=64, nx=64, batch=case["members"]))
    u = [grid.pack(a, torch.complex128) for a in _random_vector(grid, _gen(seed), 1.0)]
    torch.cuda.synchronize()
    run_.capture(steps_per_graph=10)
    state = [_view(b, grid.nkc) for b in run_.state]
    for v, a in zip(state, u):
        v.copy_(torch.view_as_real(a))
    torch.cuda.synchronize()
    return dict(case=case, run=run_, state=state, net=net)


_PREPARE = dict(step=_prepare_step, dropin=_prepare_dropin, transforms=_prepare_transforms,
                infer=_prepare_infer, train=_prepare_train, closure=_prepare_closure)


# ---------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------

def run(state):
    return _RUN[state["case"]["do"]](state)


def _run_step(s):
    from dedalus import _hip
    mid = s["case"]["integrator"] == "RK2mid"
    s["plan"].step(_hip.RK2MID if mid else _hip.RK2TRAP, s["prm"], _ptrs(s["y"]),
                   _ptrs(s["stage"]) if mid else None, _ptrs(s["d1"]), None, 1, s["dt"])
    return dict(y=s["y"], d1=s["d1"], stage=s["stage"] if mid else [])


def _run_dropin(s):
    s["ti"].do_advance(s["data"], s["dt"])
    return [_view(c._kdev(), s["nkc"]) for c in s["comps"]]


def _run_transforms(s):
    s["plan"].bwd_many(_ptrs(s["kc"]), _ptrs(s["x"]))
    s["plan"].fwd_many(_ptrs(s["x"]), _ptrs(s["out"]))
    return dict(x=s["x"], kc=s["out"])


def _run_infer(s):
    return s["inf"].run()


def _run_train(s):
    net = s["net"]
    net.zero_grad(set_to_none=True)
    out = net(s["x"])
    loss = ((out - s["y"]) ** 2).mean()
    loss.backward()
    return dict(out=out.detach(), loss=loss.detach(), gw=[p.grad for p in net.weights],
                gb=[p.grad for p in net.biases])


def _run_closure(s):
    s["run"].advance(10)
    return s["state"]


_RUN = dict(step=_run_step, dropin=_run_dropin, transforms=_run_transforms, infer=_run_infer,
            train=_run_train, closure=_run_closure)


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------

def _fft_flops(case, grid):
    """Operations of one real transform of the grid (all members)."""
    per = grid.ny * grid.nx * (grid.nz if grid.three else 1)
    return 2.5 * grid.npts * math.log2(per)


def work(case):
    if case["do"] in ("step", "dropin", "transforms"):
        grid = _Grid(case)
        cb = 8 if case.get("f32") else 16
        valid = grid.ry.numel() * grid.rz.numel() * (grid.cx + 1) * cb
        if case["do"] == "transforms":
            real = grid.npts * cb / 2
            return dict(bytes=2 * case["nf"] * (valid + real), flops=2 * case["nf"] * _fft_flops(case, grid))
        ns = _nstate(case, grid.nd)
        # the state read and written; the first stage's derivative (and the
        # midpoint state) written
        arrays = ns * (4 if case.get("integrator", "RK2mid") == "RK2mid" else 3)
        # fewest transforms of a right-hand side (rotational form)
        nt = {("hydro", 2): 5, ("hydro", 3): 9, ("boussinesq", 2): 8, ("boussinesq", 3): 13,
              ("mhd", 2): 9, ("mhd", 3): 18}[case["physics"], grid.nd]
        return dict(bytes=arrays * valid, flops=2 * nt * _fft_flops(case, grid))
    mac = sum(2 * 9 * a * b for a, b in zip(CHANS[:-1], CHANS[1:]))
    wb = sum(4 * (9 * a * b + b) for a, b in zip(CHANS[:-1], CHANS[1:]))
    if case["do"] == "closure":
        npix = max(1, case["members"]) * 64 * 64
        grid = _Grid(dict(ny=64, nx=64, batch=case["members"]))
        valid = grid.ry.numel() * grid.rz.numel() * (grid.cx + 1) * 16
        return dict(bytes=10 * (4 * valid + wb), flops=10 * (mac * npix + 10 * _fft_flops(case, grid)))
    npix = case["members"] * case["h"] * case["w"]
    if case["do"] == "infer":
        # bf16 input and fp32 output, as the buffers hold them (16 channels)
        return dict(bytes=npix * (2 * 16 + 4 * 16) + wb // 2, flops=mac * npix)
    return dict(bytes=npix * 4 * (CHANS[0] + 2 * CHANS[-1]) + 2 * wb, flops=(3 * mac - 2 * 9 * 3 * 32) * npix)


# ---------------------------------------------------------------------------
# exact
# ---------------------------------------------------------------------------

def _rhs(case, g, y):
    """The right-hand side in the physics' own (convective) form."""
    nd = g.nd
    u = y[:nd]
    ux = [g.bwd(a) for a in u]

    def advect(a):
        return g.fwd(sum(ux[j] * g.bwd(g.d(a, j)) for j in range(nd)))

    def curl(v):
        if nd == 3:
            return [g.d(v[2], 1) - g.d(v[1], 2), g.d(v[0], 2) - g.d(v[2], 0), g.d(v[1], 0) - g.d(v[0], 1)]
        return [g.d(v[1], 0) - g.d(v[0], 1)]

    f = [-advect(a) for a in u]
    if case["physics"] == "boussinesq":
        f[nd - 1] = f[nd - 1] + y[nd]
        return g.project(f) + [-advect(y[nd]) - u[nd - 1]]
    if case["physics"] == "mhd":
        b = y[nd:]
        bx, jx = [g.bwd(a) for a in b], [g.bwd(a) for a in curl(b)]
        s = 1.0 / (4.0 * math.pi * RHO0)
        if nd == 3:
            def cross(p, q):
                return [p[1] * q[2] - p[2] * q[1], p[2] * q[0] - p[0] * q[2], p[0] * q[1] - p[1] * q[0]]
            lor = cross(jx, bx)
            ind = curl([g.fwd(e) for e in cross(ux, bx)])
        else:
            lor = [-jx[0] * bx[1], jx[0] * bx[0]]
            e = g.fwd(ux[0] * bx[1] - ux[1] * bx[0])
            ind = [g.d(e, 1), -g.d(e, 0)]
        return g.project([a + s * g.fwd(p) for a, p in zip(f, lor)]) + ind
    return g.project(f)


def _phis(z):
    """exp(z), (e^z - 1) / z and (e^z - 1 - z) / z^2 for z <= 0."""
    small = z.abs() < 0.5
    zs, zl = torch.where(small, z, torch.zeros_like(z)), torch.where(small, -torch.ones_like(z), z)
    p2 = torch.zeros_like(z)
    for j in range(18, 1, -1):
        p2 = p2 * zs + 1.0 / math.factorial(j)
    p1l = torch.expm1(zl) / zl
    p1 = torch.where(small, 1.0 + zs * p2, p1l)
    return torch.exp(z), p1, torch.where(small, p2, (p1l - 1.0) / zl)


def _exact_step(case, seed):
    g = _Grid(case)
    y = [g.unpack(a) for a in _random_state(case, g, seed)]
    dt, nd = _dt(case), g.nd
    ns = _nstate(case, nd)
    coef = [NU] * ns
    if case["physics"] == "boussinesq":
        coef[nd] = KAPPA
    elif case["physics"] == "mhd":
        coef[nd:] = [ETA] * nd

    def sweep(h):
        done = {}
        for c in coef:
            if c not in done:
                done[c] = _phis(-c * g.k2 * h)
        return [done[c] for c in coef]

    d1 = _rhs(case, g, y)
    dtype = torch.complex128
    if case.get("integrator", "RK2mid") == "RK2mid":
        stage = [p0 * a + p1 * (dt / 2) * f for a, f, (p0, p1, _) in zip(y, d1, sweep(dt / 2))]
        d2 = _rhs(case, g, stage)
        new = [p0 * a + 2.0 * p2 * dt * (f2 - f1) + p1 * dt * f1
               for a, f1, f2, (p0, p1, p2) in zip(y, d1, d2, sweep(dt))]
        ends = [g.pack(a, dtype) for a in stage]
    else:
        a1 = [p0 * a + p1 * dt * f for a, f, (p0, p1, _) in zip(y, d1, sweep(dt))]
        d2 = _rhs(case, g, a1)
        new = [a + p2 * dt * (f2 - f1) for a, f1, f2, (_, _, p2) in zip(a1, d1, d2, sweep(dt))]
        ends = []
    out = [g.pack(a, dtype) for a in new]
    if case["do"] == "dropin":
        return [torch.view_as_real(a) for a in out]
    return dict(y=out, d1=[g.pack(a, dtype) for a in d1], stage=ends)


def _exact_transforms(case, seed):
    g, gen = _Grid(case), _gen(seed)
    dt = torch.complex64 if case["f32"] else torch.complex128
    xs, ks = [], []
    for _ in range(case["nf"]):
        x = g.bwd(g.unpack(g.pack(_random_scalar(g, gen, 1.0), dt)))
        xs.append(x.reshape(-1))
        ks.append(g.pack(g.fwd(x), torch.complex128))
    return dict(x=xs, kc=ks)


def _exact_net(x, ws, bs):
    """The unrounded network: periodic 3x3 convolutions as nine shifted products, tanh GELU."""
    for l, (w, b) in enumerate(zip(ws, bs)):
        z = b
        for t in range(9):
            z = z + torch.roll(x, (1 - t // 3, 1 - t % 3), (1, 2)) @ w[:, :, t // 3, t % 3].t()
        x = torch.nn.functional.gelu(z, approximate="tanh") if l < len(ws) - 1 else z
    return x


def _exact_infer(case, seed):
    x = _images(case, seed, 3).to(torch.bfloat16).double()
    ws, bs = ([p.cuda().double() for p in v] for v in _random_weights(seed, CHANS))
    out = torch.cat([_exact_net(c, ws, bs) for c in x.split(16)])
    full = torch.zeros((out.numel() // CHANS[-1], 16), dtype=torch.float64, device="cuda")
    full[:, :CHANS[-1]] = out.reshape(-1, CHANS[-1])
    return full


def _exact_train(case, seed):
    x, y = _images(case, seed, 3).double(), _images(case, seed + 1, 2).double()
    ws, bs = ([p.cuda().double().requires_grad_() for p in v] for v in _random_weights(seed, CHANS))
    outs, loss = [], 0.0
    for xc, yc in zip(x.split(8), y.split(8)):
        o = _exact_net(xc, ws, bs)
        part = ((o - yc) ** 2).sum() / y.numel()
        part.backward()
        outs.append(o.detach())
        loss = loss + part.detach()
    return dict(out=torch.cat(outs), loss=loss, gw=[w.grad for w in ws], gb=[b.grad for b in bs])


def exact(case, seed):
    if case["do"] == "closure":
        return None      # rounded activations inside a run of ten steps
    return dict(step=_exact_step, dropin=_exact_step, transforms=_exact_transforms, infer=_exact_infer,
                train=_exact_train)[case["do"]](case, seed)
