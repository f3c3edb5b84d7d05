"""The work that programs have this framework do, as measurable cases.

A case is a dict of plain values; `prepare` makes what a program has in hand
before the call (grid, simulation or solver, seeded fields on the device),
`run` is one pass through the public entry points, `work` states the bytes
and operations that a pass cannot do without, `tolerance` the error that
another correct implementation at the same precision may show, and `exact`
the pass's outputs from plain torch in 64 bits.

Fields are torch tensors indexed [z, y, x] over the storage (halo included),
which is the framework's column-major (x, y, z) layout.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "aeolus.jl_amd"))

import aeolus_hip as hip  # noqa: E402
from aeolus_hip import _lib as L  # noqa: E402
from aeolus_hip import anelastic as AN  # noqa: E402
from aeolus_hip import cutcell as CC  # noqa: E402
from aeolus_hip import learned  # noqa: E402
from aeolus_hip import terrain as TF  # noqa: E402
from aeolus_hip import workloads as W  # noqa: E402

HALO = 3
FORMS = {  # the two forms of the terrain core's step
    "fp64": dict(flux_precision="f64", vcycle="f64", smoother="rbgs", warm_start=False),
    "fast": dict(flux_precision="f32", vcycle="f32", smoother="jacobi", warm_start="extrapolate"),
}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one RK3 step of a small triply periodic Taylor-Green flow: latency and launches
        dict(name="tgv-32", kind="boussinesq", flow="tgv", nx=32, ny=32, nz=32, prec="f64", les=False),
        # a modest LES in all its options (Coriolis, sponge, Smagorinsky) on a ragged stretched grid
        dict(name="les-90x72x50", kind="boussinesq", flow="cbl", nx=90, ny=72, nz=50, prec="f64", les=True),
        # the dry convective boundary layer at its usual size, in both state precisions
        dict(name="cbl-256x256x128", kind="boussinesq", flow="cbl", nx=256, ny=256, nz=128, prec="f64", les=False),
        dict(name="cbl-256x256x128-f32", kind="boussinesq", flow="cbl", nx=256, ny=256, nz=128, prec="f32", les=False),
        # anelastic flow over terrain: a test-sized run, a mid-sized one in the fast form, the full size
        dict(name="terrain-96x96x48", kind="terrain", form="fp64", nx=96, ny=96, nz=48),
        dict(name="terrain-320x256x160-fast", kind="terrain", form="fast", nx=320, ny=256, nz=160),
        dict(name="terrain-512x512x256", kind="terrain", form="fp64", nx=512, ny=512, nz=256),
        # the sound-proof core on a regular grid, one RK3 step
        dict(name="anelastic-192x160x96", kind="anelastic", nx=192, ny=160, nz=96, prec="f64"),
        # the pressure of a flow around buildings: one MG-preconditioned CG solve and its gradient
        dict(name="cutcell-256x256x96", kind="cutcell", nx=256, ny=256, nz=96, vcycle="f32"),
        # a positive tracer's limited advection, and a scalar by the seventh-order scheme on an odd grid
        dict(name="tracer-256x256x128", kind="tracer", nx=256, ny=256, nz=128, scheme="weno_z5", prec="f64"),
        dict(name="scalar-187x141x75-f32", kind="scalar", nx=187, ny=141, nz=75, scheme="weno_z7", prec="f32"),
        # training the learned preconditioner: loss and gradients of one sample (forward and backward)
        dict(name="unet-128x128x64", kind="unet", nx=128, ny=128, nz=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth(n, even=False):
    """The product of 2, 3 and 5 nearest to n (times 2 with `even`): the transforms' sizes."""
    def ok(m):
        m = m // 2 if even and m % 2 == 0 else (0 if even else m)
        if m < 2:
            return False
        for q in (2, 3, 5):
            while m % q == 0:
                m //= q
        return m == 1
    return next(m for d in range(n) for m in (n + d, n - d) if m > 3 and ok(m))


def draw(rng):
    kind = rng.choice(["boussinesq", "boussinesq", "terrain", "terrain", "anelastic", "cutcell", "tracer", "scalar",
                       "unet"])
    prec = rng.choice(["f64", "f32"])
    if kind in ("boussinesq", "anelastic"):
        c = dict(kind=kind, nx=_smooth(_log_int(rng, 24, 256), even=True), ny=_smooth(_log_int(rng, 20, 256)),
                 nz=_log_int(rng, 16, 128), prec=prec)
        if kind == "boussinesq":
            c.update(flow=rng.choice(["tgv", "cbl"]), les=rng.random() < 0.4)
            if c["flow"] == "tgv":
                c.update(nz=_smooth(c["nz"]), les=False)
        return c
    if kind == "terrain":
        return dict(kind=kind, form=rng.choice(["fp64", "fast"]), nx=8 * _log_int(rng, 6, 40),
                    ny=8 * _log_int(rng, 6, 36), nz=8 * _log_int(rng, 4, 20))
    if kind == "cutcell":
        return dict(kind=kind, nx=8 * _log_int(rng, 6, 32), ny=8 * _log_int(rng, 6, 32), nz=8 * _log_int(rng, 6, 12),
                    vcycle=rng.choice(["f32", "f64"]))
    if kind in ("tracer", "scalar"):
        schemes = ["weno_z5", "weno_z7"] if kind == "tracer" else ["weno_z5", "weno_z7", "upwind", "centered"]
        return dict(kind=kind, nx=_log_int(rng, 24, 280), ny=_log_int(rng, 20, 256), nz=_log_int(rng, 12, 128),
                    scheme=rng.choice(schemes), prec=prec)
    return dict(kind=kind, nx=4 * _log_int(rng, 6, 36), ny=4 * _log_int(rng, 6, 36), nz=4 * _log_int(rng, 4, 18))


def _cells(c):
    return c["nx"] * c["ny"] * c["nz"]


def work(case):
    n, b = _cells(case), 4 if case.get("prec") == "f32" else 8
    kind = case["kind"]
    if kind in ("boussinesq", "anelastic", "terrain"):
        # u, v, w, theta in; they and p out. Three substages of 12 reconstructed
        # faces a cell (about 75 operations each; 8 for the centred ones of the
        # sound-proof core), the other terms and a transform solve
        faces = 12 * (8 if kind == "anelastic" else 75)
        return dict(bytes=9.0 * b * n, flops=3.0 * n * (faces + 100 + 10 * math.log2(case["nx"] * case["ny"])))
    if kind == "cutcell":
        # the source and the three apertures in; p and its gradient out; about ten smoothings' worth of operations
        return dict(bytes=8.0 * n * 8, flops=200.0 * n)
    if kind in ("tracer", "scalar"):
        # u, v, w, phi (and the accumulated tendency) in, the tendency out; three faces a cell
        per = {"weno_z5": 75, "weno_z7": 150, "upwind": 2, "centered": 3}[case["scheme"]]
        return dict(bytes=(5.0 if kind == "tracer" else 6.0) * b * n, flops=n * (3.0 * per + (60 if kind == "tracer" else 6)))
    # the network: the source, mask and target in; 2 operations a weight and voxel, forward and twice backward
    per = sum(27 * ci * co / 8 ** lev for ci, co, lev in ((2, 16, 0), (16, 16, 0), (16, 32, 1), (32, 32, 1), (32, 64, 2),
                                                          (64, 64, 2), (96, 32, 1), (32, 32, 1), (48, 16, 0), (16, 16, 0)))
    return dict(bytes=24.0 * n, flops=6.0 * per * n)


def tolerance(case):
    """About four times a pass's distance from `exact` (over the listed and drawn cases)."""
    kind = case["kind"]
    if kind == "terrain":
        # projections to a relative residual of 1e-8 (p is the furthest off); the fast form's tendencies are in 32 bits
        return {"rel": 5e-7, "max": 5e-5} if case["form"] == "fp64" else {"rel": 1e-4, "max": 1e-2}
    if kind == "cutcell":
        return {"rel": 1e-8, "max": 2e-6}  # a solve to a relative residual of 1e-8
    if kind == "unet":
        return {"rel": 3e-2, "max": 0.9}  # weights and activations in bf16, sums in 32 bits
    return {"rel": 1e-12, "max": 1e-9} if case["prec"] == "f64" else {"rel": 5e-6, "max": 5e-3}


# ---------------------------------------------------------------------------
# inputs (torch, from the seed alone; shared by prepare and exact)
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _uniform(shape, gen, lo=-1.0, hi=1.0):
    return torch.rand(shape, generator=gen, device="cuda", dtype=torch.float64) * (hi - lo) + lo


def _hartley(n):
    """The orthonormal Hartley basis (symmetric): the eigenvectors of periodic differences."""
    k = torch.arange(n, device="cuda", dtype=torch.float64)
    t = (2 * math.pi / n) * torch.remainder(k[:, None] * k[None, :], n)
    return (torch.cos(t) + torch.sin(t)) / math.sqrt(n)


def _transform(a, axes):
    """a [z, y, x] in the Hartley basis of the axes; its own inverse."""
    nz, ny, nx = a.shape
    if 2 in axes:
        a = (a.reshape(nz * ny, nx) @ _hartley(nx)).reshape(nz, ny, nx)
    if 1 in axes:
        a = (a.transpose(1, 2).reshape(nz * nx, ny) @ _hartley(ny)).reshape(nz, nx, ny).transpose(1, 2).contiguous()
    if 0 in axes:
        a = (_hartley(nz) @ a.reshape(nz, ny * nx)).reshape(nz, ny, nx)
    return a


def _turbulence(nz, ny, nx, gen):
    """A periodic random field [z, y, x] with a k^-5/3 energy spectrum, zero mean, unit RMS."""
    k2 = 0.0
    for n, ax in ((nz, 0), (ny, 1), (nx, 2)):
        q = torch.arange(n, device="cuda", dtype=torch.float64)
        q = torch.minimum(q, n - q) / n
        k2 = k2 + (q * q).reshape([-1 if a == ax else 1 for a in range(3)])
    k2[0, 0, 0] = 1.0
    amp = k2 ** (-11.0 / 12.0)
    amp[0, 0, 0] = 0.0
    a = _transform(amp * torch.randn((nz, ny, nx), generator=gen, device="cuda", dtype=torch.float64), (0, 1, 2))
    return a / a.square().mean().sqrt()


def _storage(c, H):
    return (c["nz"] + 2 * H, c["ny"] + 2 * H, c["nx"] + 2 * H)


def _inner(a, H):
    return a[H:-H, H:-H, H:-H]


def _halo(scheme):
    return 4 if scheme == "weno_z7" else HALO


def _boussinesq_setup(c):
    """(extent, interior z faces or None, physics keywords, dt)."""
    if c["flow"] == "tgv":
        s = 2 * math.pi / c["nx"]
        return (s * c["nx"], s * c["ny"], s * c["nz"]), None, dict(nu=1.0 / 1600, theta0=0.0, bcs=("periodic",) * 3), 0.1 * s
    dz1, r = 10.0, 1.02
    Lz = dz1 * (r ** c["nz"] - 1) / (r - 1)
    zf, dz = [0.0], Lz * (r - 1) / (r ** c["nz"] - 1)
    for _ in range(c["nz"]):
        zf.append(zf[-1] + dz)
        dz *= r
    zf[-1] = Lz
    phys = dict(nu=0.0, theta0=300.0, g_accel=9.81, flux_bot=0.1, flux_top=0.0, bcs=("periodic", "periodic", "wall"),
                theta_bcs=("periodic", "periodic", "noflux"))
    if c["les"]:
        phys.update(f_coriolis=1e-4, sponge_alpha_max=0.02, sponge_z_start=0.75 * Lz, C_s=0.17, Pr_t=1 / 3)
    return (20.0 * c["nx"], 20.0 * c["ny"], Lz), np.array(zf), phys, 0.5


def _boussinesq_state(c, seed):
    nx, ny, nz, H = c["nx"], c["ny"], c["nz"], HALO
    gen = _gen(seed)
    f = [torch.zeros(_storage(c, H), device="cuda", dtype=torch.float64) for _ in range(4)]
    u, v, w, th = (_inner(a, H) for a in f)
    extent, zf, _, _ = _boussinesq_setup(c)
    if c["flow"] == "tgv":
        x, y, z = (torch.arange(n, device="cuda", dtype=torch.float64) * (2 * math.pi / n) for n in (nx, ny, nz))
        hx, hy, hz = math.pi / nx, math.pi / ny, math.pi / nz
        z = z[:, None, None] + hz
        u.copy_(torch.sin(x)[None, None] * torch.cos(y + hy)[None, :, None] * torch.cos(z))
        v.copy_(-torch.cos(x + hx)[None, None] * torch.sin(y)[None, :, None] * torch.cos(z))
        for a in (u, v, w):
            a += 0.05 * _turbulence(nz, ny, nx, gen)
        th.copy_(300.0 + 0.1 * _turbulence(nz, ny, nx, gen))
    else:
        zfc = torch.tensor(zf, device="cuda")
        zc = 0.5 * (zfc[1:] + zfc[:-1])
        taper = torch.sin(math.pi * zfc[:-1] / extent[2])[:, None, None]  # w vanishes at the walls
        for a, s in ((u, 0.7), (v, 0.7), (w, 0.5 * taper)):
            a.copy_(s * _turbulence(nz, ny, nx, gen))
        th.copy_((300.0 + 0.003 * torch.clamp(zc - 1000.0, min=0.0))[:, None, None] + 0.1 * _turbulence(nz, ny, nx, gen))
    return f


def _terrain_setup(c):
    return 50.0, 10000.0, 2.5  # dx, lid, dt


def _terrain_state(c, seed):
    """(terrain (ny, nx), [u, v, w, theta] over the storage): three hills, a 10 m/s westerly with weak gusts."""
    nx, ny, nz, H = c["nx"], c["ny"], c["nz"], HALO
    dx, lid, _ = _terrain_setup(c)
    rng = np.random.default_rng(seed)
    Lx, Ly = nx * dx, ny * dx
    scale = min(1.0, min(nx, ny) / 128.0)  # narrower hills in a small domain
    x, y = (np.arange(nx) + 0.5) * dx, (np.arange(ny) + 0.5) * dx
    h = np.zeros((ny, nx))
    for _ in range(3):
        A, wd = rng.uniform(100.0, 400.0), rng.uniform(800.0, 2000.0) * scale
        x0, y0 = rng.uniform(0, Lx), rng.uniform(0, Ly)
        ddx, ddy = (x - x0 + Lx / 2) % Lx - Lx / 2, (y - y0 + Ly / 2) % Ly - Ly / 2
        h += A * scale * np.exp(-(ddx[None, :] ** 2 + ddy[:, None] ** 2) / (2 * wd * wd))
    gen = _gen(seed)
    plane = torch.tensor(np.pad(h, H, mode="wrap"), device="cuda")
    zc = (torch.arange(nz + 2 * H, device="cuda", dtype=torch.float64) - H + 0.5) * (lid / nz)
    th = 300.0 + 0.003 * (plane + zc[:, None, None] * ((lid - plane) / lid))
    f = [torch.zeros(_storage(c, H), device="cuda", dtype=torch.float64) for _ in range(3)]
    _inner(f[0], H).copy_(10.0 + 0.3 * _turbulence(nz, ny, nx, gen))
    _inner(f[1], H).copy_(0.3 * _turbulence(nz, ny, nx, gen))
    _inner(th, H)[:10] += _uniform((min(10, nz), ny, nx), gen, -0.1, 0.1)
    return h, f + [th]


def _anelastic_setup(c):
    dz = 10000.0 / c["nz"]
    return (100.0 * c["nx"], 100.0 * c["ny"], 10000.0), dz, dict(nu=5.0, flux_bot=0.02, f_coriolis=1e-4), 1.0


def _anelastic_state(c, seed):
    nx, ny, nz, H = c["nx"], c["ny"], c["nz"], HALO
    gen = _gen(seed)
    f = [torch.zeros(_storage(c, H), device="cuda", dtype=torch.float64) for _ in range(4)]
    zw = torch.sin(math.pi * torch.arange(nz, device="cuda", dtype=torch.float64) / nz)[:, None, None]
    for a, s in ((f[0], 1.0), (f[1], 1.0), (f[2], zw)):
        _inner(a, H).copy_(s * _turbulence(nz, ny, nx, gen))
    _inner(f[3], H).copy_(300.0 + 0.2 * _turbulence(nz, ny, nx, gen))
    return f


def _cutcell_heights(c, seed):
    n = max(4, c["nx"] * c["ny"] // 4096)
    h = W.buildings_heightmap((c["nx"], c["ny"]), (2.0, 2.0), n=n, seed=seed, height=(10.0, min(80.0, c["nz"] * 1.6)))
    return np.pad(h, 1, mode="wrap")  # the storage plane: the geometry is as periodic as the flow


def _cutcell_source(c, seed, ax, ay, az, fluid):
    """The aperture-weighted flux balance of a seeded turbulent velocity over the fluid [z, y, x]; ax, ay, az over
    the storage with a halo of 1."""
    gen = _gen(seed)
    b = 0.0
    for a, ax_ in ((ax, 2), (ay, 1), (az, 0)):
        flux = a[1:, 1:, 1:].clone()
        vel = _turbulence(c["nz"], c["ny"], c["nx"], gen)
        lead = [slice(0, n) for n in (c["nz"], c["ny"], c["nx"])]
        hi = list(lead)
        hi[ax_] = slice(1, flux.shape[ax_])
        vel_hi = torch.roll(vel, -1, ax_)
        if ax_ == 0:
            vel_hi[-1] = 0.0
            vel[0] = 0.0
        b = b + (flux[tuple(hi)] * vel_hi - flux[tuple(lead)] * vel) / 2.0
    b = torch.where(fluid, b, torch.zeros_like(b))
    return torch.where(fluid, b - b.sum() / fluid.sum(), b)


def _advection_state(c, seed):
    H = _halo(c["scheme"])
    gen = _gen(seed)
    f = []
    for k in range(4):
        a = _turbulence(c["nz"], c["ny"], c["nx"], gen)
        if k == 3:  # patches of tracer with sharp edges, zero outside them
            a = torch.clamp(a, min=0.0)
        if c["prec"] == "f32":
            a = a.float().double()
        f.append(torch.nn.functional.pad(a[None, None], (H,) * 6, mode="circular")[0, 0])
    return f


SPEC = [(2, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (96, 32), (32, 32), (48, 16), (16, 16)]


def _unet_params(seed):
    rng = np.random.default_rng(seed)
    out = []
    for ci, co in SPEC:
        out += [rng.standard_normal(27 * ci * co) * math.sqrt(2.0 / (27 * ci)), 0.05 * rng.standard_normal(co)]
    out += [rng.standard_normal(16) * 0.25, np.zeros(1)]
    return np.concatenate(out).astype(np.float32)


def _unet_inputs(c, seed):
    gen = _gen(seed)
    n = (c["nz"], c["ny"], c["nx"])
    heights = W.buildings_heightmap((c["nx"], c["ny"]), (2.0, 2.0), n=16, seed=seed, height=(10.0, c["nz"] * 1.2))
    z = (torch.arange(c["nz"], device="cuda") + 0.5) * 2.0
    mask = (z[:, None, None] > torch.tensor(np.ascontiguousarray(heights.T), device="cuda")).double()
    return _turbulence(*n, gen) * mask, mask, _turbulence(*n, gen) * mask


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
class _Mem:
    """A DeviceArray's memory for torch, indexed [z, y, x]."""

    def __init__(self, a):
        self.a = a
        self.__cuda_array_interface__ = dict(shape=a.shape[::-1], typestr="<f8" if a.precision == L.F64 else "<f4",
                                             data=(a.ptr, False), version=3, strides=None)


def _view(a):
    return torch.as_tensor(_Mem(a), device="cuda")


def _device(x, precision=L.F64):
    """A DeviceArray holding the torch tensor x [z, y, x]."""
    a = hip.DeviceArray(tuple(x.shape)[::-1], precision)
    hip.sync()
    _view(a).copy_(x)
    return a


def _fill(sim, fields):
    hip.sync()
    for a, x in zip((sim.u, sim.v, sim.w, sim.theta), fields):
        _view(a).copy_(x)
    torch.cuda.synchronize()


def _fields(sim):
    return {n: _view(getattr(sim, n)) for n in ("u", "v", "w", "theta", "p")}


def prepare(case, seed):
    hip.init(0)
    kind, prec = case["kind"], L.F32 if case.get("prec") == "f32" else L.F64
    N = (case["nx"], case["ny"], case["nz"])
    st = dict(kind=kind)
    if kind == "boussinesq":
        extent, zf, phys, dt = _boussinesq_setup(case)
        grid = hip.Grid(N, extent, halo=HALO, zf=zf)
        sim = hip.BoussinesqSimulation(grid, scheme="weno_z5", precision=prec, **phys)
        _fill(sim, _boussinesq_state(case, seed))
        st.update(sim=sim, dt=dt, out=_fields(sim))
    elif kind == "terrain":
        dx, lid, dt = _terrain_setup(case)
        h, fields = _terrain_state(case, seed)
        grid = hip.Grid(N, (N[0] * dx, N[1] * dx, lid), halo=HALO)
        sim = TF.AnelasticTerrainSimulation(TF.TerrainFollowingGrid(grid, h.T, lid=lid), tol=1e-8, maxit=200,
                                            **W.TERRAIN_PHYS, **FORMS[case["form"]])
        _fill(sim, fields)
        sim.fill_halos()
        sim.project()
        # this core's halos are its scratch (filled from the interior before they are read)
        st.update(sim=sim, dt=dt, out={n: _inner(a, HALO) for n, a in _fields(sim).items()})
    elif kind == "anelastic":
        extent, dz, kw, dt = _anelastic_setup(case)
        grid = hip.Grid(N, extent, halo=HALO)
        sim = AN.AnelasticSimulation(grid, AN.isentropic_reference(N[2], dz, HALO), precision=prec, **kw)
        _fill(sim, _anelastic_state(case, seed))
        st.update(sim=sim, dt=dt, out=_fields(sim))
    elif kind == "cutcell":
        grid = hip.Grid(N, tuple(2.0 * n for n in N), halo=1)
        geom = CC.CutCellGeometry(grid, _cutcell_heights(case, seed))
        solver = hip.MGPreconditionedCG(N, (2.0,) * 3, coeff=geom.coefficients(), tol=1e-8, maxit=500, nu1=2, nu2=2,
                                        vcycle=case["vcycle"], smoother="jacobi" if case["vcycle"] == "f32" else "rbgs")
        b = _cutcell_source(case, seed, _view(geom.ax), _view(geom.ay), _view(geom.az),
                            _inner(_view(geom.vol_eff), 1) > 0)
        st.update(grid=grid, geom=geom, solver=solver, b=_device(torch.nn.functional.pad(b, (1,) * 6)),
                  p=grid.field(), g=[grid.field() for _ in range(3)])
        st["out"] = [_view(a) for a in st["g"]]
    elif kind in ("tracer", "scalar"):
        H = _halo(case["scheme"])
        grid = hip.Grid(N, tuple(float(n) for n in N), halo=H)
        f = [_device(a, prec) for a in _advection_state(case, seed)]
        tend = grid.field(prec)
        st.update(grid=grid, f=f, tend=tend, scheme=case["scheme"], out=_view(tend))
        if kind == "tracer":
            st["ws"] = hip.FluxLimiterWorkspace(grid, prec)
        else:
            st["adv"] = hip.advection_scheme(case["scheme"], grid)
    else:
        net = learned.UNet(N, in_channels=2, seed=0)
        net.set_params(_unet_params(seed))
        src, mask, target = (_device(a) for a in _unet_inputs(case, seed))
        st.update(net=net, src=src, mask=mask, target=target)
    torch.cuda.synchronize()
    hip.sync()
    return st


def run(state):
    kind = state["kind"]
    if kind in ("boussinesq", "terrain", "anelastic"):
        state["sim"].step_rk3(state["dt"])
    elif kind == "cutcell":
        g = state["grid"]
        hip.solve(state["p"], state["b"], state["solver"], 1)
        hip.fill_halos(g, state["p"], L.CELL, ("periodic", "periodic", "noflux"))
        CC.gradient(*state["g"], state["p"], state["geom"])
    elif kind == "tracer":
        hip.advect_positive(state["grid"], state["tend"], *state["f"], 0.05, scheme=state["scheme"],
                            workspace=state["ws"], accumulate=False)
    elif kind == "scalar":
        state["adv"](state["tend"], *state["f"])
    else:
        loss, grad = state["net"].gradients(state["src"], state["target"], state["mask"])
        return loss, grad
    return state["out"]


# ---------------------------------------------------------------------------
# exact: the same in plain torch, 64 bits. Storage tensors [z, y, x]; `sh`
# reads a neighbour (the outermost layers it wraps are never used)
# ---------------------------------------------------------------------------
def sh(a, dz=0, dy=0, dx=0):
    return torch.roll(a, (-dz, -dy, -dx), (0, 1, 2)) if a.dim() == 3 else torch.roll(a, (-dy, -dx), (0, 1))


def _ax(a, ax, d):
    return sh(a, *[d if q == ax else 0 for q in range(3)])


def _b3(a1, a2):
    return a1 * a1 + (13.0 / 3.0) * (a2 * a2)


def _weno_z5(t):
    v1, v2, v3, v4, v5 = t
    eps = np.finfo(np.float64).eps ** 2
    q0, q1, q2 = (2 * v1 - 7 * v2 + 11 * v3) / 6, (-v2 + 5 * v3 + 2 * v4) / 6, (2 * v3 + 5 * v4 - v5) / 6
    b0 = _b3((v1 - 4 * v2 + 3 * v3) / 2, (v1 - 2 * v2 + v3) / 2)
    b1 = _b3((v4 - v2) / 2, (v2 - 2 * v3 + v4) / 2)
    b2 = _b3((-3 * v3 + 4 * v4 - v5) / 2, (v3 - 2 * v4 + v5) / 2)
    tau = (b0 - b2).abs()
    a0, a1, a2 = (g * (1 + (tau / (b + eps)) ** 2) for g, b in ((0.1, b0), (0.6, b1), (0.3, b2)))
    return (a0 * q0 + a1 * q1 + a2 * q2) / (a0 + a1 + a2)


def _weno_z7(t):
    v1, v2, v3, v4, v5, v6, v7 = t
    eps = np.finfo(np.float64).eps ** 2
    q = ((-3 * v1 + 13 * v2 - 23 * v3 + 25 * v4) / 12, (v2 - 5 * v3 + 13 * v4 + 3 * v5) / 12,
         (-v3 + 7 * v4 + 7 * v5 - v6) / 12, (3 * v4 + 13 * v5 - 5 * v6 + v7) / 12)
    # Jiang-Shu smoothness indicators of the cubics (Balsara and Shu, J. Comput. Phys. 160 (2000) 405), over 240
    b = ((v1 * (547 * v1 - 3882 * v2 + 4642 * v3 - 1854 * v4) + v2 * (7043 * v2 - 17246 * v3 + 7042 * v4)
          + v3 * (11003 * v3 - 9402 * v4) + 2107 * v4 * v4) / 240,
         (v2 * (267 * v2 - 1642 * v3 + 1602 * v4 - 494 * v5) + v3 * (2843 * v3 - 5966 * v4 + 1922 * v5)
          + v4 * (3443 * v4 - 2522 * v5) + 547 * v5 * v5) / 240,
         (v3 * (547 * v3 - 2522 * v4 + 1922 * v5 - 494 * v6) + v4 * (3443 * v4 - 5966 * v5 + 1602 * v6)
          + v5 * (2843 * v5 - 1642 * v6) + 267 * v6 * v6) / 240,
         (v4 * (2107 * v4 - 9402 * v5 + 7042 * v6 - 1854 * v7) + v5 * (11003 * v5 - 17246 * v6 + 4642 * v7)
          + v6 * (7043 * v6 - 3882 * v7) + 547 * v7 * v7) / 240)
    tau = (b[0] - b[1] - b[2] + b[3]).abs()
    a = [g / 35 * (1 + (tau / (bb + eps)) ** 2) for g, bb in zip((1, 12, 18, 4), b)]
    return sum(x * y for x, y in zip(a, q)) / sum(a)


def _face(f, ax, vel, scheme="weno_z5"):
    """The upwinded value of f at the lower face of every cell along ax."""
    if scheme == "centered":
        return (_ax(f, ax, -1) + f) / 2
    n = {"upwind": 1, "weno_z5": 5, "weno_z7": 7}[scheme]
    up, h = vel >= 0, n // 2
    t = [torch.where(up, _ax(f, ax, m - h - 1), _ax(f, ax, h - m)) for m in range(n)]
    return t[0] if n == 1 else (_weno_z5 if n == 5 else _weno_z7)(t)


def _diff(F, ax):
    return _ax(F, ax, 1) - F


def _col(v):
    return torch.as_tensor(v, device="cuda", dtype=torch.float64)[:, None, None]


def _periodic(a, H, axes):
    for ax in axes:
        n = a.shape[ax] - 2 * H
        a.narrow(ax, 0, H).copy_(a.narrow(ax, n, H).clone())
        a.narrow(ax, H + n, H).copy_(a.narrow(ax, H, H).clone())


def _fill_halo(a, H, z="mirror"):
    """Periodic x and y, then z: "periodic", "mirror" or "wall" (a z-face field, zero on both walls)."""
    _periodic(a, H, (2, 1))
    n = a.shape[0] - 2 * H
    if z == "periodic":
        _periodic(a, H, (0,))
    elif z == "mirror":
        for h in range(1, H + 1):
            a[H - h] = a[H + h - 1]
            a[H + n - 1 + h] = a[H + n - h]
    else:
        a[H] = 0.0
        a[H + n] = 0.0
        for h in range(1, H + 1):
            a[H - h] = -a[H + h]
            if H + n + h < a.shape[0]:
                a[H + n + h] = -a[H + n - h]


def _thomas(lower, diag, upper, b):
    """Tridiagonal solves along z; lower, upper per level, diag and b [z, ...]."""
    nz = b.shape[0]
    cp, x = [None] * nz, [None] * nz
    for k in range(nz):
        den = diag[k] - (lower[k] * cp[k - 1] if k else 0.0)
        cp[k] = upper[k] / den
        x[k] = (b[k] - (lower[k] * x[k - 1] if k else 0.0)) / den
    for k in range(nz - 2, -1, -1):
        x[k] = x[k] - cp[k] * x[k + 1]
    return torch.stack(x)


def _eigen(n, d, ax):
    k = torch.arange(n, device="cuda", dtype=torch.float64)
    return (4 / d ** 2 * torch.sin(math.pi * k / n) ** 2).reshape([-1 if a == ax else 1 for a in range(3)])


def _column_solve(b, dx, dy, lower, upper, hweight, measure, icoup, gauge):
    """Periodic x-y transforms, a tridiagonal solve a column, the mean mode by its fluxes."""
    nz, ny, nx = b.shape
    lam = (_eigen(nx, dx, 2) + _eigen(ny, dy, 1))[0]
    hat = _transform(b, (1, 2))
    mean = hat[:, 0, 0].cpu().numpy().copy()
    lam[0, 0] = 1.0
    diag = [-(lower[k] + upper[k]) - lam * hweight[k] for k in range(nz)]
    x = _thomas(lower, diag, upper, hat)
    mean = mean - (mean * measure).sum() / measure.sum()
    F = np.concatenate([[0.0], np.cumsum(mean * measure)[:-1]])
    ph = np.cumsum(F * icoup[:nz])
    x[:, 0, 0] = torch.as_tensor(ph - (ph * gauge).sum() / gauge.sum(), device=b.device)
    return _transform(x, (1, 2))


def _stretched_solve(dx, dy, dzc, dzf):
    nz = len(dzc)
    lower = np.array([1 / (dzc[k] * dzf[k]) if k else 0.0 for k in range(nz)])
    upper = np.array([1 / (dzc[k] * dzf[k + 1]) if k < nz - 1 else 0.0 for k in range(nz)])
    return lambda b: _column_solve(b, dx, dy, lower, upper, np.ones(nz), dzc, dzf, dzc)


def _periodic_solve(dx, dy, dz):
    def solve(b):
        lam = -(_eigen(b.shape[0], dz, 0) + _eigen(b.shape[1], dy, 1) + _eigen(b.shape[2], dx, 2))
        lam[0, 0, 0] = 1.0
        hat = _transform(b, (0, 1, 2)) / lam
        hat[0, 0, 0] = 0.0
        return _transform(hat, (0, 1, 2))
    return solve


def _smagorinsky(u, v, w, th, m, H, C_s, Pr_t, z):
    """The eddy terms of u, v, w, theta (m: the grid's metrics)."""
    ix, iy = 1 / m["dx"], 1 / m["dy"]
    off = _col(2 / (m["dzf"][:-1] + m["dzf"][1:]))
    coef = _col((C_s * (m["dx"] * m["dy"] * m["dzc"]) ** (1.0 / 3)) ** 2)
    iz, izf = _col(1 / m["dzc"]), _col(1 / m["dzf"][:-1])
    sx, sy, sz = (_ax(u, 2, 1) - u) * ix, (_ax(v, 1, 1) - v) * iy, (_ax(w, 0, 1) - w) * iz

    def cross(f, own, ax, q):  # a velocity averaged to the centre along its own axis, differenced across along ax
        c = f + _ax(f, own, 1)
        return (_ax(c, ax, 1) - _ax(c, ax, -1)) * (0.25 * q)
    s12 = 0.5 * (cross(u, 2, 1, iy) + cross(v, 1, 2, ix))
    s13 = 0.5 * (cross(u, 2, 0, off) + cross(w, 0, 2, ix))
    s23 = 0.5 * (cross(v, 1, 0, off) + cross(w, 0, 1, iy))
    nu = coef * torch.sqrt(2 * (sx * sx + sy * sy + sz * sz) + 4 * (s12 * s12 + s13 * s13 + s23 * s23))
    _fill_halo(nu, H, "periodic" if z == "periodic" else "mirror")

    def term(f, own):  # d_j(nu d_j f) for f on the lower faces of axis `own` (None: at centres)
        t = 0.0
        for ax, q in ((2, ix), (1, iy), (0, None)):
            if ax == own:  # fluxes at cell centres: nu of the cell below
                qi, qo = (_col(1 / m["dzc"]), izf) if ax == 0 else (q, q)
                t = t + (nu * (_ax(f, ax, 1) - f) * qi - _ax(nu, ax, -1) * (f - _ax(f, ax, -1)) * (sh(qi, -1) if ax == 0 else qi)) * qo
                continue
            e = 0.5 * (_ax(nu, ax, -1) + nu) if own is None else 0.25 * (nu + _ax(nu, ax, -1) + _ax(nu, own, -1) + _ax(_ax(nu, ax, -1), own, -1))
            F = e * (f - _ax(f, ax, -1)) * (izf if ax == 0 else q)
            t = t + _diff(F, ax) * (iz if ax == 0 else q)
        return t
    return term(u, 2), term(v, 1), term(w, 0), term(th, None) / Pr_t


def _exact_boussinesq(c, seed):
    H, nz = HALO, c["nz"]
    extent, zf, phys, dt = _boussinesq_setup(c)
    u, v, w, th = _boussinesq_state(c, seed)
    if c["prec"] == "f32":
        u, v, w, th = (a.float().double() for a in (u, v, w, th))
    dx, dy, dz = extent[0] / c["nx"], extent[1] / c["ny"], extent[2] / nz
    n = nz + 2 * H
    if zf is None:
        dzc, dzf = np.full(n, dz), np.full(n + 1, dz)
    else:
        z = np.zeros(n + 1)
        z[H:H + nz + 1] = zf
        for k in range(H - 1, -1, -1):
            z[k] = 2 * z[k + 1] - z[k + 2]
        for k in range(H + nz + 1, n + 1):
            z[k] = 2 * z[k - 1] - z[k - 2]
        dzc, zc = np.diff(z), (z[1:] + z[:-1]) / 2
        dzf = np.concatenate([[dzc[0]], np.diff(zc), [dzc[-1]]])
    m = dict(dx=dx, dy=dy, dzc=dzc, dzf=dzf)
    prev = np.roll(dzc, 1)
    whi, ahi = _col(prev / (prev + dzc)), _col(dzc / (prev + dzc))  # weights of the upper level at a z face
    iz, izf, ix, iy = _col(1 / dzc), _col(1 / dzf[:-1]), 1 / dx, 1 / dy
    zw, zs = ("periodic", "periodic") if c["flow"] == "tgv" else ("wall", "mirror")
    I = (slice(H, H + nz), slice(H, -H), slice(H, -H))
    solve = _periodic_solve(dx, dy, dz) if c["flow"] == "tgv" else _stretched_solve(dx, dy, dzc[H:H + nz], dzf[H:H + nz + 1])

    def fill(uvw):
        for a, k in zip(uvw, (zs, zs, zw)):
            _fill_halo(a, H, k)

    def adv(f, U, V, Wv, q):
        return (_diff(U * _face(f, 2, U), 2) * ix + _diff(V * _face(f, 1, V), 1) * iy) + _diff(Wv * _face(f, 0, Wv), 0) * q

    def lap(f, own_z):
        g = (sh(f, 0, 0, 1) - 2 * f + sh(f, 0, 0, -1)) * ix * ix + (sh(f, 0, 1) - 2 * f + sh(f, 0, -1)) * iy * iy
        return g + (sh(f, 1) - 2 * f + sh(f, -1)) / dz ** 2  # viscosity is used on uniform levels only

    p = torch.zeros_like(u)
    start = None
    for stage, (ca, cb) in enumerate(((0.0, 1.0), (0.75, 0.25), (1.0 / 3, 2.0 / 3))):
        fill((u, v, w))
        _fill_halo(th, H, zs)
        if stage == 0:
            start = [a.clone() for a in (u, v, w, th)]
        mx, my = (lambda a: (sh(a, 0, 0, -1) + a) / 2), (lambda a: (sh(a, 0, -1) + a) / 2)
        zm = lambda a: (1 - ahi) * sh(a, -1) + ahi * a  # noqa: E731
        t = [-adv(u, mx(u), mx(v), mx(w), iz), -adv(v, my(u), my(v), my(w), iz),
             -adv(w, zm(u), zm(v), (sh(w, -1) + w) / 2, izf), -adv(th, u, v, w, iz)]
        if phys["nu"]:
            t = [a + phys["nu"] * lap(f, None) for a, f in zip(t, (u, v, w, th))]
        if phys.get("C_s"):
            t = [a + e for a, e in zip(t, _smagorinsky(u, v, w, th, m, H, phys["C_s"], phys["Pr_t"], zs))]
        if phys["theta0"]:
            t[2] = t[2] + phys["g_accel"] / phys["theta0"] * ((1 - whi) * sh(th, -1) + whi * th - phys["theta0"])
        f = phys.get("f_coriolis", 0.0)
        if f:
            t[0] = t[0] + f * 0.5 * (mx(v) + sh(mx(v), 0, 1))
            t[1] = t[1] - f * 0.5 * (my(u) + sh(my(u), 0, 0, 1))
        if phys.get("flux_bot"):
            t[3][H] += phys["flux_bot"] / dzc[H]
        if phys.get("sponge_alpha_max"):
            zi = z[H:H + nz + 1]
            for q, (a, lev) in enumerate(((u, (zi[1:] + zi[:-1]) / 2), (v, (zi[1:] + zi[:-1]) / 2), (w, zi[:-1]))):
                zs0 = phys["sponge_z_start"]
                r = np.where(lev >= zs0, phys["sponge_alpha_max"] * np.sin(0.5 * math.pi * (lev - zs0) / (zf[-1] - zs0)) ** 2, 0.0)
                t[q][H:H + nz] -= _col(r) * a[H:H + nz]
        th_old, new = th, []
        for a, tt in zip((u, v, w), t):
            a = a.clone()
            a[I] += dt * tt[I]
            new.append(a)
        u, v, w = new
        fill((u, v, w))
        div = (_diff(u, 2) * ix + _diff(v, 1) * iy + _diff(w, 0) * iz)[I]
        phi = torch.zeros_like(u)
        phi[I] = solve(div.contiguous())
        _fill_halo(phi, H, zs)
        for a, ax, q in ((u, 2, ix), (v, 1, iy), (w, 0, izf)):
            a[I] -= ((phi - _ax(phi, ax, -1)) * q)[I]
        th = th_old.clone()
        th[I] += dt * t[3][I]
        if stage:
            u, v, w, th = (ca * s + cb * a for s, a in zip(start, (u, v, w, th)))
        p[I] = phi[I] / dt
    return dict(u=u, v=v, w=w, theta=th, p=p)


def _exact_anelastic(c, seed):
    H, nz = HALO, c["nz"]
    extent, dz, kw, dt = _anelastic_setup(c)
    f = _anelastic_state(c, seed)
    if c["prec"] == "f32":
        f = [a.float().double() for a in f]
    dx, dy = extent[0] / c["nx"], extent[1] / c["ny"]
    # an isentropic column in the discrete hydrostatic balance (log-mean face densities)
    R, cp, p0, g, theta = 287.0, 1004.0, 1.0e5, 9.81, 300.0
    dens = lambda p: (p0 / (R * theta)) * (p / p0) ** ((cp - R) / cp)  # noqa: E731
    lm = lambda a, b: a if a == b else (a - b) / math.log1p((a - b) / b)  # noqa: E731
    pb, rb = [], []
    for k in range(nz):
        q = p0 if k == 0 else pb[-1] - g * dz * rb[-1]
        for _ in range(200):
            last, q = q, (p0 - g * dz / 2 * dens(q)) if k == 0 else pb[-1] - g * dz * lm(rb[-1], dens(q))
            if abs(last - q) <= 1e-15 * q:
                break
        pb.append(q)
        rb.append(dens(q))
    rho = np.array(rb)
    rf = np.concatenate([[rho[0]], [lm(rho[k - 1], rho[k]) for k in range(1, nz)], [rho[-1]]])
    pad = lambda a, lo, hi: np.concatenate([a[0] * (a[0] / a[1]) ** np.arange(lo, 0, -1), a, a[-1] * (a[-1] / a[-2]) ** np.arange(1, hi + 1)])  # noqa: E731
    Wc, Wf = _col(pad(rho, H, H)), _col(pad(rf, H, H - 1))
    ix, iy, iz = 1 / dx, 1 / dy, 1 / dz
    I = (slice(H, H + nz), slice(H, -H), slice(H, -H))
    idz2 = iz * iz
    lower = np.array([rf[k] * idz2 if k else 0.0 for k in range(nz)])
    upper = np.array([rf[k + 1] * idz2 if k < nz - 1 else 0.0 for k in range(nz)])
    mid = lambda a, ax: 0.5 * (_ax(a, ax, -1) + a)  # noqa: E731
    cen = lambda a, ax: 0.5 * (a + _ax(a, ax, 1))  # noqa: E731
    lap = lambda a: sum((_ax(a, ax, 1) - 2 * a + _ax(a, ax, -1)) * q * q for ax, q in ((2, ix), (1, iy), (0, iz)))  # noqa: E731
    p = torch.zeros_like(f[0])

    def fill(q):
        for a, z in zip(q, ("mirror", "mirror", "wall", "mirror")):
            _fill_halo(a, H, z)

    def euler(f):
        f = [a.clone() for a in f]
        fill(f)
        u, v, w, th = f
        t = [-((_diff(mid(u, 2) ** 2, 2) * ix + _diff(mid(v, 2) * mid(u, 1), 1) * iy) + _diff(Wf * mid(w, 2) * mid(u, 0), 0) * iz / Wc),
             -((_diff(mid(u, 1) * mid(v, 2), 2) * ix + _diff(mid(v, 1) ** 2, 1) * iy) + _diff(Wf * mid(w, 1) * mid(v, 0), 0) * iz / Wc),
             -((_diff(mid(u, 0) * mid(w, 2), 2) * ix + _diff(mid(v, 0) * mid(w, 1), 1) * iy)
               + (Wc * cen(w, 0) ** 2 - sh(Wc, -1) * mid(w, 0) ** 2) * iz / Wf),
             -((_diff(u * mid(th, 2), 2) * ix + _diff(v * mid(th, 1), 1) * iy) + _diff(Wf * w * mid(th, 0), 0) * iz / Wc)]
        t = [a + kw["nu"] * lap(q) for a, q in zip(t, f)]
        t[2] = t[2] + g / theta * (mid(th, 0) - theta)
        t[0] = t[0] + kw["f_coriolis"] * cen(mid(v, 2), 1)
        t[1] = t[1] - kw["f_coriolis"] * cen(mid(u, 1), 2)
        t[3][H] += kw["flux_bot"] * iz
        for a, tt in zip(f, t):
            a[I] += dt * tt[I]
        th_halo = th
        for a, z in zip(f[:3], ("mirror", "mirror", "wall")):
            _fill_halo(a, H, z)
        div = (Wc * (_diff(u, 2) * ix + _diff(v, 1) * iy) + _diff(Wf * w, 0) * iz)[I]
        phi = torch.zeros_like(u)
        phi[I] = _column_solve(div.contiguous(), dx, dy, lower, upper, rho, np.full(nz, dz ** 2), 1 / rf, np.ones(nz))
        _fill_halo(phi, H)
        for a, ax, q in ((u, 2, ix), (v, 1, iy), (w, 0, iz)):
            a[I] -= ((phi - _ax(phi, ax, -1)) * q)[I]
        p[I] = phi[I] / dt
        return [u, v, w, th_halo]

    start = [a.clone() for a in f]
    f = euler(euler(f))
    f = [0.75 * s + 0.25 * a for s, a in zip(start, f)]
    f = euler(f)
    f = [s / 3 + a * (2.0 / 3) for s, a in zip(start, f)]
    return dict(u=f[0], v=f[1], w=f[2], theta=f[3], p=p)


class _Terrain:
    """The anelastic core over a Gal-Chen grid, z = h + s (lid - h)/lid, rho = rho0 exp(-z/Hs)."""

    def __init__(self, c, h):
        self.c, self.H = c, HALO
        H, ph = HALO, W.TERRAIN_PHYS
        self.dx, self.lid, self.dt = _terrain_setup(c)
        self.dz = self.lid / c["nz"]
        lid = self.lid
        hp = torch.tensor(np.pad(h, H, mode="wrap"), device="cuda")
        mx, my = (lambda a: (sh(a, 0, 0, -1) + a) / 2), (lambda a: (sh(a, 0, -1) + a) / 2)
        J = lambda a: (lid - a) / lid  # noqa: E731
        n = c["nz"] + 2 * H
        sf = _col((np.arange(n) - H) * self.dz)
        sc = sf + 0.5 * self.dz
        rho = lambda a, s: ph["rho0"] * torch.exp(-(a + s * J(a)) / ph["Hs"])  # noqa: E731
        hx, hy, hxy = mx(hp), my(hp), my(mx(hp))
        self.J, self.Jx, self.Jy, self.Jxy = J(hp), J(hx), J(hy), J(hxy)
        self.rc, self.rx, self.ry, self.rs = rho(hp, sc), rho(hx, sc), rho(hy, sc), rho(hp, sf)
        self.rxy, self.rxs, self.rys = rho(hxy, sc), rho(hx, sf), rho(hy, sf)
        sl = -(lid - sf) / (lid - hp)
        self.sx = sl * ((sh(hp, 0, 0, 1) - sh(hp, 0, 0, -1)) / (2 * self.dx))
        self.sy = sl * ((sh(hp, 0, 1) - sh(hp, 0, -1)) / (2 * self.dx))
        self.zf, self.ph = hp + sf * self.J, ph
        self.I = (slice(H, H + c["nz"]), slice(H, -H), slice(H, -H))
        # interior coefficients of B, G and L; sigma faces 0 .. nz
        K = slice(H, H + c["nz"] + 1)
        self.mxi, self.myi = (self.rx * self.Jx)[self.I], (self.ry * self.Jy)[self.I]
        self.rsi, self.Ji = self.rs[K, H:-H, H:-H].clone(), self.J[H:-H, H:-H]
        self.sxi, self.syi = self.sx[K, H:-H, H:-H], self.sy[K, H:-H, H:-H]
        self.rsi[0] = self.rsi[-1] = 0.0
        cz = (self.rsi * self.Ji * (self.sxi ** 2 + self.syi ** 2 + 1 / self.Ji ** 2)).mean((1, 2)).cpu().numpy()
        nz, i2 = c["nz"], 1 / self.dz ** 2
        self.pre = (np.concatenate([[0.0], cz[1:nz] * i2]), np.concatenate([cz[1:nz] * i2, [0.0]]),
                    self.mxi.mean((1, 2)).cpu().numpy(), np.full(nz, self.dz ** 2),
                    np.concatenate([[1.0], 1 / cz[1:nz], [1.0]]), np.ones(nz))

    def omega(self, u, v, w):
        ub, vb = (0.25 * (sh(u, -1) + sh(u, -1, 0, 1) + u + sh(u, 0, 0, 1)), 0.25 * (sh(v, -1) + sh(v, -1, 1) + v + sh(v, 0, 1)))
        o = w + self.J * (self.sx * ub + self.sy * vb)
        o[self.H] = 0.0
        o[self.H + self.c["nz"]] = 0.0
        return o

    def fill(self, u, v, w, th=None):
        H, nz = self.H, self.c["nz"]
        for a in (u, v) + (() if th is None else (th,)):
            _fill_halo(a, H)
        ub = 0.25 * (sh(u, -1) + sh(u, -1, 0, 1) + u + sh(u, 0, 0, 1))
        vb = 0.25 * (sh(v, -1) + sh(v, -1, 1) + v + sh(v, 0, 1))
        wall = -self.J * (self.sx * ub + self.sy * vb)
        for k in (H, H + nz):
            w[k] = wall[k]
        for q in range(1, H + 1):
            w[H - q] = 2 * w[H] - w[H + q]
            if H + nz + q < w.shape[0]:
                w[H + nz + q] = 2 * w[H + nz] - w[H + nz - q]
        _periodic(w, H, (2, 1))

    def tendencies(self, u, v, w, th):
        i, iz, om = 1 / self.dx, 1 / self.dz, self.omega(u, v, w)
        mx, my, mz = ((lambda a, ax=ax: (_ax(a, ax, -1) + a) / 2) for ax in (2, 1, 0))

        def t(f, X, Y, Z, M):
            return -((_diff(X * _face(f, 2, X), 2) * i + _diff(Y * _face(f, 1, Y), 1) * i) + _diff(Z * _face(f, 0, Z), 0) * iz) / M
        cJ = self.rc * self.J
        xy = self.rxy * self.Jxy
        tu = t(u, sh(cJ, 0, 0, -1) * mx(u), xy * mx(v), self.rxs * mx(om), self.rx * self.Jx)
        tv = t(v, xy * my(u), sh(cJ, 0, -1) * my(v), self.rys * my(om), self.ry * self.Jy)
        tw = t(w, self.rxs * self.Jx * mz(u), self.rys * self.Jy * mz(v), sh(self.rc, -1) * mz(om), self.rs * self.J)
        tt = t(th, self.rx * self.Jx * u, self.ry * self.Jy * v, self.rs * om, cJ)
        tb = self.ph["theta0"] + self.ph["gamma"] * self.zf
        tw = tw + self.ph["g_accel"] / tb * (0.5 * (sh(th, -1) + th) - tb)
        tw[self.H] = 0.0
        return tu, tv, tw, tt

    def div(self, u, v, w):
        om, i = self.omega(u, v, w), 1 / self.dx
        return (_diff(self.rx * self.Jx * u, 2) * i + _diff(self.ry * self.Jy * v, 1) * i + _diff(self.rs * om, 0) / self.dz)[self.I].contiguous()

    def grad(self, phi):
        d = torch.zeros_like(self.rsi)
        d[1:-1] = (phi[1:] - phi[:-1]) / self.dz
        q = 0.25 * self.rsi * self.Ji * d
        Sx, Sy = q * self.sxi, q * self.syi
        Sx, Sy = Sx[1:] + Sx[:-1], Sy[1:] + Sy[:-1]
        gx = (phi - torch.roll(phi, 1, 2)) / self.dx + (Sx + torch.roll(Sx, 1, 2)) / self.mxi
        gy = (phi - torch.roll(phi, 1, 1)) / self.dx + (Sy + torch.roll(Sy, 1, 1)) / self.myi
        return gx, gy, d / self.Ji

    def apply(self, phi):
        gx, gy, gw = self.grad(phi)
        cx, cy = 0.25 * (gx + torch.roll(gx, -1, 2)), 0.25 * (gy + torch.roll(gy, -1, 1))
        gw[1:-1] += self.Ji * (self.sxi[1:-1] * (cx[1:] + cx[:-1]) + self.syi[1:-1] * (cy[1:] + cy[:-1]))
        gw *= self.rsi
        fx, fy = self.mxi * gx, self.myi * gy
        return (torch.roll(fx, -1, 2) - fx) / self.dx + (torch.roll(fy, -1, 1) - fy) / self.dx + (gw[1:] - gw[:-1]) / self.dz

    def solve(self, b):
        return _pcg(self.apply, lambda r: _column_solve(r, self.dx, self.dx, *self.pre), b, 1e-12, 80)

    def step(self, f):
        f = [a.clone() for a in f]
        self.fill(*f)
        ground = f[2][self.H].clone()
        t = self.tendencies(*f)
        I = self.I
        for a, q in zip(f, t):
            a[I] += self.dt * q[I]
        self.fill(*f[:3])
        phi = self.solve(self.div(*f[:3]))
        self.correct(f, phi)
        return f, phi / self.dt, ground

    def correct(self, f, phi):
        for a, g in zip(f, self.grad(phi)):
            a[self.I] -= g[: self.c["nz"]]


def _pcg(A, M, b, tol, maxit, keep=None):
    """Flexible CG on a negative semidefinite operator with the constants in its kernel."""
    mean = (lambda a: a.mean()) if keep is None else (lambda a: (a * keep).sum() / keep.sum())
    proj = (lambda a: a - mean(a)) if keep is None else (lambda a: (a - mean(a)) * keep)
    r, x = proj(b), torch.zeros_like(b)
    stop = tol * r.norm()
    p = None
    for _ in range(maxit):
        z = proj(M(r))
        p = z if p is None else z - ((z * q).sum() / pq) * p
        q = A(p)
        pq = (p * q).sum()
        a = (p * r).sum() / pq
        x = x + a * p
        r = r - a * q
        if r.norm() <= stop:
            break
    return proj(x)


def _exact_terrain(c, seed):
    h, f = _terrain_state(c, seed)
    T = _Terrain(c, h)
    T.fill(*f)
    T.correct(f, T.solve(T.div(*f[:3])))
    T.fill(*f[:3])
    start = [a.clone() for a in f]
    f = T.step(T.step(f)[0])[0]
    f = [0.75 * s + 0.25 * a for s, a in zip(start, f)]
    f, p, ground = T.step(f)
    f = [s / 3 + a * (2.0 / 3) for s, a in zip(start, f)]
    f[2][HALO] = ground  # w on the ground is diagnostic: as the last substage found it
    I = T.I
    return dict(u=f[0][I], v=f[1][I], w=f[2][I], theta=f[3][I], p=p)


def _exact_cutcell(c, seed):
    N = (c["nx"], c["ny"], c["nz"])
    _, ve, ax, ay, az = CC.heightmap_geometry(N, (2.0,) * 3, 1, _cutcell_heights(c, seed))
    ve, ax, ay, az = (torch.tensor(np.ascontiguousarray(a.T), device="cuda") for a in (ve, ax, ay, az))
    fluid = _inner(ve, 1) > 0
    b = _cutcell_source(c, seed, ax, ay, az, fluid)
    # face coefficients a^2 on the lower faces of the interior cells and the closing one
    cx, cy, cz = (a[1:, 1:, 1:][:c["nz"] + (q == 0), :c["ny"] + (q == 1), :c["nx"] + (q == 2)] ** 2 for q, a in ((2, ax), (1, ay), (0, az)))

    def lower(p, ax_):  # p[i] - p[i - 1] on the lower faces and the closing one (periodic x and y, none through the ends of z)
        d = p - torch.roll(p, 1, ax_)
        if ax_ == 0:
            d[0] = 0.0
        close = torch.zeros_like(d.narrow(ax_, 0, 1)) if ax_ == 0 else d.narrow(ax_, 0, 1)
        return torch.cat([d, close], ax_)

    def A(p):
        t = 0.0
        for co, ax_ in ((cx, 2), (cy, 1), (cz, 0)):
            F = co * lower(p, ax_)
            n = p.shape[ax_]
            t = t + (F.narrow(ax_, 1, n) - F.narrow(ax_, 0, n)) / 4.0
        return t
    pre = _stretched_solve(2.0, 2.0, np.full(c["nz"], 2.0), np.full(c["nz"] + 1, 2.0))
    p = _pcg(A, pre, b, 1e-12, 600, keep=fluid.double())
    out = []
    for a, ax_ in ((ax, 2), (ay, 1), (az, 0)):
        g = torch.zeros_like(ax)
        g[1:-1, 1:-1, 1:-1] = _inner(a, 1) * (lower(p, ax_).narrow(ax_, 0, p.shape[ax_])) / 2.0
        out.append(g)
    return out


def _exact_advection(c, seed):
    u, v, w, phi = _advection_state(c, seed)
    H, out = _halo(c["scheme"]), torch.zeros_like(phi)
    vel = ((u, 2), (v, 1), (w, 0))
    F = [a * _face(phi, ax, a, c["scheme"]) for a, ax in vel]
    if c["kind"] == "tracer":
        dt = 0.05
        Lo = [a * _face(phi, ax, a, "upwind") for a, ax in vel]
        A = [f - l for f, l in zip(F, Lo)]
        Pm = dt * sum(torch.clamp(_ax(a, ax, 1), min=0) + torch.clamp(-a, min=0) for a, (_, ax) in zip(A, vel))
        Q = torch.clamp(phi - dt * sum(_diff(l, ax) for l, (_, ax) in zip(Lo, vel)), min=0)
        R = torch.where(Pm > 0, torch.clamp(Q / torch.where(Pm > 0, Pm, torch.ones_like(Pm)), max=1), torch.ones_like(Pm))
        _periodic(R, H, (2, 1, 0))
        F = [l + torch.where(a >= 0, _ax(R, ax, -1), R) * a for a, l, (_, ax) in zip(A, Lo, vel)]
    d = sum(_diff(f, ax) for f, (_, ax) in zip(F, vel))
    _inner(out, H).copy_(-_inner(d, H))
    return out


def _exact_unet(c, seed):
    params = torch.tensor(_unet_params(seed).astype(np.float64), device="cuda", requires_grad=True)
    src, mask, target = _unet_inputs(c, seed)
    off = 0

    def take(n):
        nonlocal off
        off += n
        return params[off - n:off]

    def conv(x, ci, co):  # x [z, y, x, channel]; W[tap][c][n], tap = (dx+1) + 3(dy+1) + 9(dz+1)
        Wt, b = take(27 * ci * co).reshape(3, 3, 3, ci, co), take(co)
        nz, ny, nx, _ = x.shape
        xp = torch.nn.functional.pad(x, (0, 0, 0, 0, 0, 0, 1, 1))
        y = b
        for dz in range(3):
            for dy in range(3):
                for dx in range(3):
                    y = y + torch.roll(xp[dz:dz + nz], (1 - dy, 1 - dx), (1, 2)).reshape(-1, ci) @ Wt[dz, dy, dx]
        return torch.relu(y).reshape(nz, ny, nx, co)

    def pool(x):
        nz, ny, nx, k = x.shape
        return x.reshape(nz // 2, 2, ny // 2, 2, nx // 2, 2, k).mean((1, 3, 5))

    def up(x):
        return x.repeat_interleave(2, 0).repeat_interleave(2, 1).repeat_interleave(2, 2)
    rms = src.square().mean().sqrt()
    a = conv(conv(torch.stack([src / rms, mask], -1), 2, 16), 16, 16)
    b = conv(conv(pool(a), 16, 32), 32, 32)
    d = conv(conv(pool(b), 32, 64), 64, 64)
    e = conv(conv(torch.cat([up(d), b], -1), 96, 32), 32, 32)
    g = conv(conv(torch.cat([up(e), a], -1), 48, 16), 16, 16)
    y = g @ take(16) + take(1)
    loss = (y - target / rms).square().mean()
    loss.backward()
    return float(loss), params.grad.cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "boussinesq":
        return _exact_boussinesq(case, seed)
    if kind == "anelastic":
        return _exact_anelastic(case, seed)
    if kind == "terrain":
        return _exact_terrain(case, seed)
    if kind == "cutcell":
        return _exact_cutcell(case, seed)
    if kind == "unet":
        return _exact_unet(case, seed)
    return _exact_advection(case, seed)
