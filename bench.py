"""Benchmark: one full SSP-RK3 step of the anelastic core over Gal-Chen
terrain at 512 x 512 x 256 on one MI355X, projected to ||r|| <= 1e-8 ||b||
by MG-preconditioned CG at every substage.

Workload: three seeded Gaussian hills (heights U[100, 400] m, half-widths
U[500, 2000] m) on a 50 m grid under a 10 km lid, reference density
1.2 exp(-z/8 km), 10 m/s westerly, θ = 300 K + 3 K/km, WENO-Z5 advection of
momentum and θ, buoyancy about θ̄(z). Synthetic seeded input, spun up from
its projected start, resident in HBM before the timed region.

Prints ONE JSON line: value = cell-updates/s of the FP64 form (the
reference's arithmetic: FP64 tendencies, MG-PCG with an FP64 red-black
V-cycle from a zero guess); beside it the fast form (FP32 WENO arithmetic on
the FP64 state, FP32 Jacobi V-cycle inside the FP64 CG, extrapolated warm
start) with its speed-up, field errors and constraint residual; the roofline
of the dominant kernel (the finest level's red-black pass); the STREAM
triad; the CPU oracle timed on the host cores on a bounded sample of the
same workload, in turns with GPU steps; and extra legs (the DCBL
256x256x128 step, the cut-cell Poisson solve with the learned FCG, the
positive tracer advection).
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
for p in (ROOT, os.path.join(ROOT, "aeolus.jl_amd")):
    if p not in sys.path:
        sys.path.insert(0, p)

import numpy as np  # noqa: E402

METRIC = "cell-updates/s per RK3 step + Poisson ms to 1e-8 residual (learned vs MG-PCG)"
HBM_PEAK_GBS = 8000.0
NX, NY, NZ = 256, 256, 128
DT = 0.5


def tendency_bytes_per_launch(esz):
    """Compulsory HBM bytes of one launch of the fused tendency kernel over the
    interior: reads u, v, w, θ, writes u*, v*, w*, θ' (8 arrays), plus θ0 in
    the combined substages 2 and 3 (9 arrays); averaged over the 3 launches of
    a step: (8 + 9 + 9) / 3 arrays."""
    return NX * NY * NZ * esz * (8 + 9 + 9) / 3.0


def read_traffic():
    """HBM bytes per tendency launch from the committed rocprofv3 --pmc summary
    (FETCH_SIZE + WRITE_SIZE per dispatch, scaled by the copy-kernel factor)."""
    path = os.path.join(ROOT, "profiles", "tendency_dcbl_256x256x128_pmc.txt")
    if not os.path.exists(path):
        return None
    vals = {}
    for line in open(path):
        if "=" in line and not line.lstrip().startswith("#"):
            k, v = line.split("=", 1)
            try:
                vals[k.strip()] = float(v.split()[0])
            except ValueError:
                pass
    if "traffic_bytes_per_launch" in vals:
        return vals["traffic_bytes_per_launch"]
    return None


def read_terrain_valu():
    """VALU wave-instructions per launch of the finest-level FP64 red-black
    pass from the committed rocprofv3 --pmc summary (SQ_INSTS_VALU)."""
    path = os.path.join(ROOT, "profiles", "rbgs_f64_terrain_512x512x256_pmc.txt")
    if not os.path.exists(path):
        return None
    for line in open(path):
        if line.startswith("valu_insts_per_launch"):
            try:
                return float(line.split("=", 1)[1].split()[0])
            except ValueError:
                return None
    return None


def read_terrain_traffic():
    """HBM bytes per launch of the finest-level FP64 red-black pass from the
    committed rocprofv3 --pmc summary (FETCH_SIZE + WRITE_SIZE per dispatch,
    scaled by the STREAM-triad dispatch's factors)."""
    path = os.path.join(ROOT, "profiles", "rbgs_f64_terrain_512x512x256_pmc.txt")
    if not os.path.exists(path):
        return None
    for line in open(path):
        if line.startswith("traffic_bytes_per_launch"):
            try:
                return float(line.split("=", 1)[1].split()[0])
            except ValueError:
                return None
    return None


def run_gpu(steps, warmup, precision):
    import aeolus_hip as hip
    from aeolus_hip import _lib as L
    from aeolus_hip import workloads as W

    hip.init(0)
    g = W.dcbl_grid((NX, NY, NZ))
    sim = hip.BoussinesqSimulation(g, scheme="weno_z5", precision=precision, **W.DCBL_PHYS)
    sim.set(*W.dcbl_state(g))
    lib = L.init()
    for _ in range(warmup):
        sim.step_rk3(DT)
    hip.sync()
    L.check(lib.aeo_profile_enable(1))
    L.check(lib.aeo_profile_reset())
    t0 = time.perf_counter()
    for _ in range(steps):
        sim.step_rk3(DT)
    hip.sync()
    t1 = time.perf_counter()
    prof = {}
    import ctypes
    for name in ("tendency", "poisson", "halo", "divergence", "correct", "shell"):
        c = ctypes.c_int()
        ms = ctypes.c_double()
        L.check(lib.aeo_profile_get(name.encode(), ctypes.byref(c), ctypes.byref(ms)))
        prof[name] = (c.value, ms.value)
    L.check(lib.aeo_profile_enable(0))
    div = sim.max_divergence()
    return (t1 - t0) / steps, prof, div


def poisson_ms(reps=20):
    """The direct column solve (exact to round-off) at the workload's size."""
    import aeolus_hip as hip
    from aeolus_hip import workloads as W
    g = W.dcbl_grid((NX, NY, NZ))
    s = hip.solver_for(g)
    src = np.random.default_rng(1).normal(size=(NX, NY, NZ))
    hip.solve_interior(s, src)
    phi = hip.DeviceArray((NX, NY, NZ))
    hip.sync()
    t0 = time.perf_counter()
    for _ in range(reps):
        hip.solve_source_buffer(phi, s)
    hip.sync()
    return (time.perf_counter() - t0) / reps * 1e3


CUT_N = (512, 512, 192)
CUT_DX = 2.0


def _residual64(solver, x_dev, b):
    """‖(b − mean b) − A x‖ / ‖b − mean b‖ recomputed in FP64 with the solver's operator."""
    import aeolus_hip as hip
    ax = hip.DeviceArray(CUT_N)
    solver.apply(ax, x_dev)
    r = (b - b.mean()) - ax.download()
    return float(np.linalg.norm(r) / np.linalg.norm(b - b.mean()))


def poisson_legs(reps=3, weights=None, log=print):
    """The standalone cut-cell Poisson solve at 512x512x192, Δ = 2 m, 64 seeded
    buildings, source = divergence of a seeded k^-5/3 velocity: ms per solve
    to ‖r‖ ≤ 1e-8‖b‖ for MG-PCG (FP32 V-cycle, 2+2 Jacobi; and FP64 V-cycle,
    red-black Gauss-Seidel) and for the learned flexible CG."""
    import ctypes
    import aeolus_hip as hip
    from aeolus_hip import _lib as L
    from aeolus_hip import workloads as W
    from aeolus_hip.learned import FlexibleCG, UNet
    t0 = time.perf_counter()
    w = W.cutcell_workload(CUT_N, CUT_DX, n_buildings=64)
    log(f"cut-cell workload built in {time.perf_counter() - t0:.1f} s")
    b = w["source"]
    out = {}

    def run(name, solver):
        n = CUT_N[0] * CUT_N[1] * CUT_N[2]
        buf = ctypes.c_void_p(hip.source_buffer(solver))
        phi = hip.DeviceArray(CUT_N)
        ms = []
        for rep in range(reps + 1):
            L.check(L.init().aeo_memcpy_h2d(buf, np.asfortranarray(b).ctypes.data_as(ctypes.c_void_p), 8 * n))
            hip.sync()
            t = time.perf_counter()
            hip.solve_source_buffer(phi, solver)
            hip.sync()
            if rep:
                ms.append((time.perf_counter() - t) * 1e3)
        it, rel = hip.solver_stats(solver)
        base = solver if hasattr(solver, "apply") else solver._keep[0]
        out[name] = {"ms": float(np.median(ms)), "iterations": it, "residual": rel,
                     "residual_fp64_recomputed": _residual64(base, phi, b), "status": solver.last_status}
        log(f"{name}: {out[name]}")

    mg32 = hip.MGPreconditionedCG(CUT_N, (CUT_DX,) * 3, coeff=w["coeff"], tol=1e-8, maxit=500, nu1=2, nu2=2,
                                  smoother="jacobi", omega=0.8, vcycle="f32")
    run("mgpcg_f32_jacobi", mg32)
    mg64 = hip.MGPreconditionedCG(CUT_N, (CUT_DX,) * 3, coeff=w["coeff"], tol=1e-8, maxit=500, nu1=2, nu2=2,
                                  smoother="rbgs", vcycle="f64")
    run("mgpcg_f64_rbgs", mg64)
    del mg64
    if weights is not None and os.path.exists(weights):
        net = UNet(CUT_N, in_channels=2, seed=0)
        net.set_params(np.load(weights, allow_pickle=False))
        mask = hip.DeviceArray.from_numpy(w["mask"])
        run("fcg_net_guess_vcycle", FlexibleCG(mg32, net, mask, mode="vcycle", guess=True, tol=1e-8, maxit=500))
        # the network as the preconditioner of every iteration: it is trained on
        # sources, not on the residuals FCG hands it, and does not converge
        # here; capped so the leg reports its status without holding the GPU
        run("fcg_net_vcycle", FlexibleCG(mg32, net, mask, mode="net+vcycle", guess=True, tol=1e-8, maxit=60))
        run("fcg_vcycle", FlexibleCG(mg32, None, None, mode="vcycle", guess=False, tol=1e-8, maxit=500))
    return out


def tracer_leg(reps=20, warmup=3):
    """advect_positive (WENO-Z5, FP64) of a sharp positive tracer on the
    256x256x128 grid (regular, periodic; the WENO stencils need uniform
    spacing) in a seeded random flow, with a reusable workspace: ms per call
    (the library's event timer on its stream), the compulsory HBM bytes
    (read u, v, w, ϕ; write tend: 5 arrays) and the rate they imply."""
    import ctypes
    import aeolus_hip as hip
    from aeolus_hip import _lib as L
    hip.init(0)
    g = hip.Grid((NX, NY, NZ), (float(NX), float(NY), float(NZ)), halo=3)
    rng = np.random.default_rng(11)
    bcs = ("periodic",) * 3
    dev = []
    for loc in (1, 2, 3):
        d = hip.DeviceArray.from_numpy(np.asfortranarray(rng.standard_normal(g.storage)))
        hip.fill_halos(g, d, loc, bcs)
        dev.append(d)
    phi = hip.DeviceArray.from_numpy(np.asfortranarray(rng.uniform(0, 1, g.storage) ** 4))
    hip.fill_halos(g, phi, 0, bcs)
    tend = hip.DeviceArray(g.storage)
    ws = hip.FluxLimiterWorkspace(g)
    dt = 0.05
    for _ in range(warmup):
        hip.advect_positive(g, tend, *dev, phi, dt, workspace=ws, accumulate=False)
    hip.sync()
    lib = L.init()
    L.check(lib.aeo_profile_enable(1))
    L.check(lib.aeo_profile_reset())
    t0 = time.perf_counter()
    for _ in range(reps):
        hip.advect_positive(g, tend, *dev, phi, dt, workspace=ws, accumulate=False)
    hip.sync()
    wall = (time.perf_counter() - t0) / reps
    c, ms = ctypes.c_int(), ctypes.c_double()
    L.check(lib.aeo_profile_get(b"advect_positive", ctypes.byref(c), ctypes.byref(ms)))
    L.check(lib.aeo_profile_enable(0))
    ev_ms = ms.value / max(c.value, 1)
    alg = NX * NY * NZ * 8 * 5
    return {"ms_per_call": ev_ms, "wall_ms_per_call": wall * 1e3, "compulsory_bytes": alg,
            "compulsory_GBs": alg / (ev_ms / 1e3) / 1e9,
            "workload": "advect_positive WENO-Z5 FP64, 256x256x128 regular periodic grid, seeded random flow, "
                        "tracer uniform(0,1)^4, reusable workspace, accumulate=false"}


TARGET_N = (512, 512, 256)


def target_leg(steps=2, log=print):
    """A full SSP-RK3 step at 512x512x256 projected by MG-PCG to ||r|| <= 1e-8
    ||b||, in the plain FP64 form (FP64 WENO-Z5 tendencies, FP64 red-black
    V-cycle) and in the FP32 form (FP32 state and tendencies, FP32 Jacobi V-cycle inside
    the FP64 CG). Convective boundary layer on a regular 20 m grid (periodic
    x-y, walls in z): theta = 300 K to 1 km then +3 K/km, seeded +-0.1 K noise in
    the lowest 10 levels, seeded +-0.5 m/s horizontal velocity, surface flux
    0.1 K m/s. Each form: one forward-Euler step that projects the random start
    (RK3 keeps a third of its start's divergence, so it must start solenoidal),
    one warm-up RK3 step, then `steps` timed steps; the FP32 forms' fields are
    compared with the FP64 form's after the same steps."""
    import aeolus_hip as hip
    from aeolus_hip import workloads as W
    hip.init(0)
    N, dx = TARGET_N, 20.0
    g = hip.Grid(N, (N[0] * dx, N[1] * dx, N[2] * dx), halo=3)
    H, I = g.H, g.interior
    zc = (np.arange(N[2]) + 0.5) * dx
    rng = np.random.default_rng(W.DCBL_SEED)
    th = np.zeros(g.storage, order="F")
    th[:, :, H:H + N[2]] = np.where(zc <= 1000.0, 300.0, 300.0 + 0.003 * (zc - 1000.0))[None, None, :]
    th[H:H + N[0], H:H + N[1], H:H + 10] += rng.uniform(-0.1, 0.1, (N[0], N[1], 10))
    u, v, w = (np.zeros(g.storage, order="F") for _ in range(3))
    u[I] = 0.5 * rng.uniform(-1, 1, N)
    v[I] = 0.5 * rng.uniform(-1, 1, N)
    out, fields = {}, {}
    forms = (("fp64_mgpcg", 0, dict(smoother="rbgs", vcycle="f64")),
             ("fp32_mgpcg", 1, dict(smoother="jacobi", omega=0.8, vcycle="f32")),
             ("fp32_mgpcg_rbgs", 1, dict(smoother="rbgs", vcycle="f32")))
    for name, prec, kw in forms:
        solver = hip.MGPreconditionedCG(N, (dx,) * 3, bcs=("periodic", "periodic", "neumann"), tol=1e-8, maxit=200,
                                        nu1=2, nu2=2, **kw)
        sim = hip.BoussinesqSimulation(g, scheme="weno_z5", precision=prec, solver=solver, **W.DCBL_PHYS)
        sim.set(u, v, w, th)
        sim.step(DT)
        sim.step_rk3(DT)
        hip.sync()
        t0 = time.perf_counter()
        for _ in range(steps):
            sim.step_rk3(DT)
        hip.sync()
        ms = (time.perf_counter() - t0) / steps * 1e3
        its, res = hip.solver_stats(solver)
        out[name] = {"ms_per_step": ms, "cell_updates_per_s": N[0] * N[1] * N[2] / (ms / 1e3),
                     "last_solve_iterations": its, "last_solve_residual": res, "status": solver.last_status,
                     "max_divergence_after_step": sim.max_divergence()}
        fields[name] = {n: a[I].astype(np.float64) for n, a in sim.state().items() if n != "p"}
        log(f"target {name}: {out[name]}")
        del sim, solver
    a = fields["fp64_mgpcg"]
    for name in ("fp32_mgpcg", "fp32_mgpcg_rbgs"):
        b = fields[name]
        err = {n: float(np.abs(b[n] - a[n]).max() / np.abs(a[n]).max()) for n in ("u", "v", "w")}
        err["theta"] = float(np.abs(b["theta"] - a["theta"]).max() / np.abs(a["theta"]).max())
        err["theta_minus_300"] = float(np.abs(b["theta"] - a["theta"]).max() / np.abs(a["theta"] - 300.0).max())
        out[name]["rel_error_vs_fp64"] = err
        out[name]["speedup_vs_fp64"] = out["fp64_mgpcg"]["ms_per_step"] / out[name]["ms_per_step"]
    out["workload"] = ("convective boundary layer 512x512x256, regular 20 m grid, WENO-Z5, SSP-RK3, MG-PCG "
                       "projection to 1e-8 (FP64 form: FP64 tendencies + FP64 RBGS V-cycle; FP32 forms: FP32 "
                       "tendencies + FP32 Jacobi or RBGS V-cycle in FP64 CG)")
    return out


TERRAIN_FORMS = {
    # the reference's arithmetic: FP64 tendencies, MG-PCG with an FP64 red-black V-cycle, zero guess
    "fp64_mgpcg": dict(flux_precision="f64", vcycle="f64", smoother="rbgs", warm_start=False),
    # FP32 WENO fluxes (state FP64), FP32 V-cycle in the FP64 CG, the previous solve's φ as initial guess
    "fp32_mgpcg_warm": dict(flux_precision="f32", vcycle="f32", smoother="rbgs", warm_start=True),
    # the same with the guess extrapolated from the same substage of the last two steps
    "fp32_mgpcg_extrap": dict(flux_precision="f32", vcycle="f32", smoother="rbgs", warm_start="extrapolate"),
    "fp32_jacobi_extrap": dict(flux_precision="f32", vcycle="f32", smoother="jacobi", warm_start="extrapolate"),
    "fp32_rbgs11_extrap": dict(flux_precision="f32", vcycle="f32", smoother="rbgs", nu1=1, nu2=1,
                               warm_start="extrapolate"),
    "fp32_jacobi_quad": dict(flux_precision="f32", vcycle="f32", smoother="jacobi", warm_start="quadratic"),
    "fp32_jacobi33_extrap": dict(flux_precision="f32", vcycle="f32", smoother="jacobi", nu1=3, nu2=3,
                                 warm_start="extrapolate"),
    "fp32_jacobi11_extrap": dict(flux_precision="f32", vcycle="f32", smoother="jacobi", nu1=1, nu2=1,
                                 warm_start="extrapolate"),
    "fp32_jacobi_lsq3": dict(flux_precision="f32", vcycle="f32", smoother="jacobi", warm_start="least_squares",
                             basis=3),
    "fp32_jacobi_lsq6": dict(flux_precision="f32", vcycle="f32", smoother="jacobi", warm_start="least_squares",
                             basis=6),
    "fp32_jacobi_lsq9": dict(flux_precision="f32", vcycle="f32", smoother="jacobi", warm_start="least_squares",
                             basis=9),
}


def terrain_leg(steps=2, warmup=2, N=TARGET_N, forms=TERRAIN_FORMS, log=print, profile=False, spinup=40):
    """The anelastic core over Gal-Chen terrain at N (three seeded Gaussian
    hills, exponential reference density with an 8 km scale height, 10 m/s
    westerly, θ = 300 K + 3 K/km): a full SSP-RK3 step with WENO-Z5 advection
    and the density-weighted projection solved to ||r|| <= 1e-8 ||b|| at every
    substage. The flow is first spun up from its projected start for `spinup`
    steps (untimed, with the last form); each form then starts from that
    state, takes `warmup` untimed steps and `steps` timed ones; the other
    forms' fields are compared with the first form's after the same steps."""
    import ctypes
    import aeolus_hip as hip
    from aeolus_hip import _lib as L
    from aeolus_hip import workloads as W
    from aeolus_hip.terrain import AnelasticTerrainSimulation, TerrainFollowingGrid
    hip.init(0)
    t0 = time.perf_counter()
    g, h, state, dt = W.terrain_workload(N)
    tg = TerrainFollowingGrid(g, h, g.Lz)
    log(f"terrain workload built in {time.perf_counter() - t0:.1f} s")
    out, fields = {}, {}
    lib = L.init()
    spin = AnelasticTerrainSimulation(tg, scheme="weno_z5", tol=1e-8, maxit=200, **W.TERRAIN_PHYS,
                                      **list(forms.values())[-1])
    spin.set(*state)
    spin.project()
    out["initial_constraint_residual"] = spin.constraint_residual()
    t0 = time.perf_counter()
    for _ in range(spinup):
        spin.step_rk3(dt)
    hip.sync()
    start = {n: getattr(spin, n).download() for n in ("u", "v", "w", "theta")}
    out["spinup"] = {"steps": spinup, "t_s": spinup * dt, "wall_s": time.perf_counter() - t0,
                     "constraint_residual": spin.constraint_residual()}
    log(f"terrain spin-up: {out['spinup']}")
    del spin
    for name, kw in forms.items():
        t0 = time.perf_counter()
        sim = AnelasticTerrainSimulation(tg, scheme="weno_z5", tol=1e-8, maxit=200, **W.TERRAIN_PHYS, **kw)
        sim.set(start["u"], start["v"], start["w"], start["theta"])
        log(f"terrain {name}: set up in {time.perf_counter() - t0:.1f} s")
        for _ in range(warmup):
            sim.step_rk3(dt)
        hip.sync()
        if profile:
            L.check(lib.aeo_profile_enable(1))
            L.check(lib.aeo_profile_reset())
        iters, hist = [], []
        t0 = time.perf_counter()
        for _ in range(steps):
            sim.step_rk3(dt)
            hist.append(sim.step_history())
            iters.append(sum(hist[-1][0]))
        hip.sync()
        ms = (time.perf_counter() - t0) / steps * 1e3
        prof = {}
        if profile:
            for k in ("tf_halo", "tf_tendency", "tf_div", "tf_solve", "tf_correct", "tf_apply", "mg_rbgs_f64_l0",
                      "mg_rbgs_f32_l0", "mg_jacobi_f32_l0", "mg_jacobi_f64_l0"):
                c, t = ctypes.c_int(), ctypes.c_double()
                L.check(lib.aeo_profile_get(k.encode(), ctypes.byref(c), ctypes.byref(t)))
                if c.value:
                    prof[k] = {"launches_per_step": c.value / steps, "ms_per_step": t.value / steps,
                               "ms_per_launch": t.value / c.value}
            L.check(lib.aeo_profile_enable(0))
        st = sim.solver_stats()
        out[name] = {"ms_per_step": ms, "cell_updates_per_s": N[0] * N[1] * N[2] / (ms / 1e3),
                     "solve_iterations_per_step": iters, "last_solve": st,
                     "substage_iterations_and_initial_residuals": hist,
                     "constraint_residual_after_step": sim.constraint_residual(), "by_phase": prof, **kw}
        fields[name] = {n: getattr(sim, n).download()[g.interior] for n in ("u", "v", "w", "theta")}
        log(f"terrain {name}: {out[name]}")
        del sim
    names = list(forms)
    a = fields[names[0]]
    H = g.H
    plane = tg.plane
    J = (g.Lz - plane[H:H + g.Nx, H:H + g.Ny]) / g.Lz
    zc = plane[H:H + g.Nx, H:H + g.Ny, None] + ((np.arange(g.Nz) + 0.5) * g.dz)[None, None, :] * J[:, :, None]
    thbar = W.TERRAIN_PHYS["theta0"] + W.TERRAIN_PHYS["gamma"] * zc
    for name in names[1:]:
        b = fields[name]
        err = {n: float(np.abs(b[n] - a[n]).max() / np.abs(a[n]).max()) for n in ("u", "v", "w")}
        err["theta_minus_thetabar"] = float(np.abs(b["theta"] - a["theta"]).max() / np.abs(a["theta"] - thbar).max())
        out[name]["rel_error_vs_" + names[0]] = err
        out[name]["speedup_vs_" + names[0]] = out[names[0]]["ms_per_step"] / out[name]["ms_per_step"]
    out["workload"] = (f"anelastic flow over terrain {N[0]}x{N[1]}x{N[2]}, Gal-Chen grid dx = dy = 50 m, lid 10 km, "
                       "3 seeded Gaussian hills (heights U[100, 400] m, half-widths U[500, 2000] m), rho = 1.2 "
                       "exp(-z/8 km), 10 m/s westerly, theta = 300 K + 3 K/km with seeded +-0.1 K noise near the "
                       f"ground, WENO-Z5, SSP-RK3 dt = {dt} s, density-weighted terrain projection to 1e-8 per "
                       "substage")
    out["dt"] = dt
    return out


def read_valu_insts():
    """VALU wave-instructions per tendency launch from the committed
    rocprofv3 --pmc SQ summary (SQ_INSTS_VALU per dispatch)."""
    path = os.path.join(ROOT, "profiles", "step_dcbl_256x256x128_f64_sq.txt")
    if not os.path.exists(path):
        return None
    cols = None
    for line in open(path):
        if line.startswith("kernel "):
            cols = line.split()[1:]
        elif cols and line.startswith("void aeo::adv_tile_kernel<2, 4, 2, double"):
            vals = line.split()[-len(cols):]
            return float(vals[cols.index("INSTS_VALU")])
    return None


# one wave64 VALU instruction occupies a 16-lane SIMD for 4 cycles; MI355X:
# 256 CUs x 4 SIMDs at 2.4 GHz
VALU_CYCLES_PER_INST = 4
N_SIMD = 1024
CLOCK_HZ = 2.4e9


def learned_ms(legs):
    """The fastest converged leg that uses the network (None without one)."""
    if not legs:
        return None
    ms = [v["ms"] for k, v in legs.items() if k.startswith("fcg_net") and v["status"] == "converged"]
    return min(ms) if ms else None


def cpu_baseline(threads):
    """The CPU oracle (FP64, OpenMP) on a bounded sample of the same workload:
    the full 256x256x128 grid, one warm-up step, then the minimum of two timed
    RK3 steps on `threads` threads and one timed step on one thread."""
    os.environ["OMP_NUM_THREADS"] = str(threads)
    from oracle import oracle as orc
    from aeolus_hip import workloads as W
    from aeolus_hip.fields import Grid
    zf, Lz = W.dcbl_faces(NZ)
    extent = (20.0 * NX, 20.0 * NY, Lz)
    og = orc.Grid((NX, NY, NZ), extent, 3, zf)
    g = Grid((NX, NY, NZ), extent, halo=3, zf=zf)
    u, v, w, th = W.dcbl_state(g)
    p = og.zeros()
    st = orc.Stepper(og, scheme="weno_z5", **W.DCBL_PHYS)
    orc.lib().orc_set_threads(threads)
    st.rk3(u, v, w, th, p, DT)
    times = []
    for _ in range(2):
        t0 = time.perf_counter()
        st.rk3(u, v, w, th, p, DT)
        times.append(time.perf_counter() - t0)
    orc.lib().orc_set_threads(1)
    t0 = time.perf_counter()
    st.rk3(u, v, w, th, p, DT)
    t1 = time.perf_counter() - t0
    orc.lib().orc_set_threads(threads)
    return NX * NY * NZ / min(times), min(times), NX * NY * NZ / t1, t1


TRIAD_N = 1 << 27  # doubles per array: 1 GiB each


def stream_triad(reps=1, n=TRIAD_N):
    """The STREAM triad a = b + s·c over n doubles (library kernel, 8-byte
    accesses like the solver's vector kernels): ms per call from the
    library's event timer and the bandwidth 24n bytes / time. One call is
    also the dispatch that calibrates FETCH_SIZE / WRITE_SIZE (it reads 16n
    bytes and writes 8n)."""
    import ctypes
    import aeolus_hip as hip
    from aeolus_hip import _lib as L
    lib = L.init()
    a, b, c = (hip.DeviceArray((n,)) for _ in range(3))
    args = (ctypes.c_void_p(a.ptr), ctypes.c_void_p(b.ptr), ctypes.c_void_p(c.ptr), 0.5, n)
    L.check(lib.aeo_stream_triad(*args))  # warm
    hip.sync()
    L.check(lib.aeo_profile_enable(1))
    L.check(lib.aeo_profile_reset())
    for _ in range(reps):
        L.check(lib.aeo_stream_triad(*args))
    hip.sync()
    cnt, ms = ctypes.c_int(), ctypes.c_double()
    L.check(lib.aeo_profile_get(b"triad", ctypes.byref(cnt), ctypes.byref(ms)))
    L.check(lib.aeo_profile_enable(0))
    t = ms.value / max(cnt.value, 1)
    return {"ms_per_call": t, "GBs": 24 * n / (t / 1e3) / 1e9, "bytes_read": 16 * n, "bytes_written": 8 * n,
            "calls": reps}


def copy_calibration():
    """One triad dispatch after the workload: the FETCH_SIZE / WRITE_SIZE reference."""
    return stream_triad(reps=1)


def profile_pass(steps, warmup):
    t, _, _ = run_gpu(steps, warmup, 0)
    cal = copy_calibration()
    print(json.dumps({"profile_pass": True, "ms_per_step": t * 1e3, "calibration": cal}), flush=True)


# the headline's forms: the reference's arithmetic and the fast form beside it
HEAD_FORM = "fp64_mgpcg"
FAST_FORM = "fp32_jacobi_extrap"


def host_sensors():
    """CPU clocks (kHz, mean/min/max of scaling_cur_freq) and the hwmon
    power (W) and temperature (C) readings of the amdgpu, k10temp and
    coretemp devices, where the host exposes them (the reference's benchmark
    protocol logs these next to the step times)."""
    import glob
    out = {}
    freqs = []
    for f in glob.glob("/sys/devices/system/cpu/cpu[0-9]*/cpufreq/scaling_cur_freq"):
        try:
            freqs.append(int(open(f).read()))
        except (OSError, ValueError):
            pass
    if freqs:
        out["cpu_khz"] = {"mean": sum(freqs) / len(freqs), "min": min(freqs), "max": max(freqs), "n": len(freqs)}
    for d in glob.glob("/sys/class/hwmon/hwmon*"):
        try:
            name = open(os.path.join(d, "name")).read().strip()
        except OSError:
            continue
        if name not in ("amdgpu", "k10temp", "coretemp"):
            continue
        rec = {}
        for key, fn, scale in (("power_W", "power1_average", 1e-6), ("power_W", "power1_input", 1e-6),
                               ("temp_C", "temp1_input", 1e-3), ("sclk_MHz", "freq1_input", 1e-6)):
            if key in rec:
                continue
            try:
                rec[key] = int(open(os.path.join(d, fn)).read()) * scale
            except (OSError, ValueError):
                pass
        if rec:
            out.setdefault(name, []).append(rec)
    return out


TERRAIN_CPU_N = (96, 96, 48)


def terrain_cpu_baseline(threads, reps=5, gpu_turn=None, log=print):
    """The CPU oracle (FP64, OpenMP, MG-preconditioned CG) on a bounded sample
    of the terrain workload: the same construction at TERRAIN_CPU_N (dx = 50 m,
    3 seeded hills, lid 10 km), projected start, one warm-up RK3 step, then
    `reps` timed steps on `threads` threads, alternating with `gpu_turn` (a
    GPU step of the headline) in turns, the host sensors read beside each
    CPU step; then one step on 1 thread. Returns min and median s/step."""
    os.environ["OMP_NUM_THREADS"] = str(threads)
    from oracle import oracle as orc
    from aeolus_hip import workloads as W
    from aeolus_hip.terrain import storage_plane
    extent, h, (u, v, w, th), dt = W.terrain_state(TERRAIN_CPU_N)
    og = orc.Grid(TERRAIN_CPU_N, extent, halo=3)
    plane = storage_plane(h, TERRAIN_CPU_N, 3)
    phys = {k: W.TERRAIN_PHYS[k] for k in ("rho0", "Hs", "theta0", "gamma", "g_accel")}
    core = orc.TerrainCore(og, plane, extent[2], buoyancy=True, scheme="weno_z5", **phys)
    core.use_multigrid()
    orc.lib().orc_set_threads(threads)
    core.fill_halos(u, v, w, th)
    b = core.divergence(u, v, w)
    phi, _, _ = core.solve(b, tol=1e-10)
    gx, gy, gw = core.gradient(phi)
    H, I = og.H, og.interior
    u[I] -= gx
    v[I] -= gy
    w[H:H + og.Nx, H:H + og.Ny, H + 1:H + og.Nz] -= gw[:, :, 1:og.Nz]
    core.fill_halos(u, v, w, th)
    p = og.zeros()
    core.step_rk3(u, v, w, th, p, dt, tol=1e-8)
    times, sensors = [], []
    for _ in range(reps):
        s0 = host_sensors()
        t0 = time.perf_counter()
        core.step_rk3(u, v, w, th, p, dt, tol=1e-8)
        times.append(time.perf_counter() - t0)
        sensors.append({"before": s0, "after": host_sensors()})
        log(f"cpu terrain step {len(times)}: {times[-1]:.3f} s")
        if gpu_turn is not None:
            gpu_turn()
    orc.lib().orc_set_threads(1)
    t0 = time.perf_counter()
    core.step_rk3(u, v, w, th, p, dt, tol=1e-8)
    t1 = time.perf_counter() - t0
    orc.lib().orc_set_threads(threads)
    return {"min_s": min(times), "median_s": float(np.median(times)), "times_s": times, "one_thread_s": t1,
            "sensors": sensors}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--cpu-threads", type=int, default=0)
    ap.add_argument("--cpu-reps", type=int, default=5)
    ap.add_argument("--no-extra", action="store_true",
                    help="skip the extra legs (DCBL 256x256x128 step, cut-cell Poisson, advect_positive)")
    ap.add_argument("--no-poisson", action="store_true", help="skip the cut-cell Poisson leg")
    ap.add_argument("--weights", default=os.path.join(ROOT, "aeolus.jl_amd", "aeolus_hip", "weights",
                                                      "unet_cutcell_dx2.npy"))
    ap.add_argument("--poisson-pass", action="store_true", help="only the cut-cell Poisson legs, for kernel traces")
    ap.add_argument("--target-pass", action="store_true", help="only the 512x512x256 boundary-layer MG-PCG leg")
    ap.add_argument("--spinup", type=int, default=40, help="untimed steps of the terrain flow before its forms")
    ap.add_argument("--terrain-pass", action="store_true",
                    help="only the 512x512x256 anelastic terrain step (FP64 and fast forms), with per-phase times")
    ap.add_argument("--forms", default="", help="comma-separated terrain forms for --terrain-pass (default: all)")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="end --terrain-pass with one STREAM triad over 1 GiB arrays (the FETCH_SIZE / WRITE_SIZE "
                         "reference)")
    ap.add_argument("--tracer-pass", action="store_true",
                    help="only the advect_positive leg (--steps calls), for rocprofv3 kernel traces")
    ap.add_argument("--profile-pass", action="store_true",
                    help="a short DCBL FP64 run for rocprofv3 counter passes, then one STREAM triad (the "
                         "calibration of FETCH_SIZE / WRITE_SIZE)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py runs on one GPU: this build has no multi-GPU path (asked for --gpus {args.gpus})",
              file=sys.stderr)
        sys.exit(2)
    log = lambda m: print(m, file=sys.stderr, flush=True)  # noqa: E731
    if args.poisson_pass:
        legs = poisson_legs(weights=args.weights, log=log)
        print(json.dumps({"poisson_pass": True, "legs": legs}), flush=True)
        return
    if args.target_pass:
        print(json.dumps({"target_pass": True, **target_leg(log=log)}), flush=True)
        return
    if args.terrain_pass:
        forms = TERRAIN_FORMS
        if args.forms:
            forms = {k: TERRAIN_FORMS[k] for k in args.forms.split(",")}
        res = terrain_leg(steps=args.steps, warmup=args.warmup, log=log, profile=True, spinup=args.spinup,
                          forms=forms)
        if args.copy_calibration:
            res["calibration"] = copy_calibration()
        print(json.dumps({"terrain_pass": True, **res}), flush=True)
        return
    if args.tracer_pass:
        print(json.dumps({"tracer_pass": True, **tracer_leg(args.steps, args.warmup)}), flush=True)
        return
    if args.profile_pass:
        profile_pass(args.steps, args.warmup)
        return
    rank = int(os.environ.get("RANK", "0"))

    from aeolus_hip.provenance import provenance
    sensors0 = host_sensors()
    triad = stream_triad(reps=20)
    log(f"STREAM triad: {triad}")
    forms = {HEAD_FORM: TERRAIN_FORMS[HEAD_FORM], FAST_FORM: TERRAIN_FORMS[FAST_FORM]}
    ter = terrain_leg(steps=args.steps, warmup=args.warmup, forms=forms, log=log, profile=True, spinup=args.spinup)
    N = TARGET_N
    cells = N[0] * N[1] * N[2]
    head, fast = ter[HEAD_FORM], ter[FAST_FORM]

    # the dominant kernel of the headline form: the finest level's red-black
    # colour pass of the FP64 V-cycle, which evaluates the face coefficients
    # from the terrain metrics. Algorithmic bytes per launch: the elements a
    # colour pass cannot avoid, the other colour's half of φ and the colour's
    # half of b read and its half of φ written (3 × 4 B per cell; φ and b are
    # stored colour-split, a cell's own old value is not read); beside it the
    # VALU issue of its FP64 arithmetic
    rb = head["by_phase"]["mg_rbgs_f64_l0"]
    avg_s = rb["ms_per_launch"] / 1e3
    alg = 3 * 4 * cells
    achieved = alg / avg_s / 1e9
    valu = read_terrain_valu()
    roofline = {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": achieved / HBM_PEAK_GBS, "traffic": read_terrain_traffic(),
                "kernel": "rbgs_tf_kernel (mg.hip) on the finest level (512x512x256), one colour pass",
                "valu_insts_per_launch": valu,
                "valu_issue_ms": valu * VALU_CYCLES_PER_INST / (N_SIMD * CLOCK_HZ) * 1e3 if valu else None,
                "valu_issue_frac": (valu * VALU_CYCLES_PER_INST / (N_SIMD * CLOCK_HZ)) / avg_s if valu else None,
                "avg_launch_ms": rb["ms_per_launch"], "launches_per_step": rb["launches_per_step"],
                "share_of_step": rb["ms_per_step"] / head["ms_per_step"],
                "algorithmic_bytes_per_launch": alg,
                "stream_triad_GBs": triad["GBs"], "frac_of_triad": achieved / triad["GBs"]}
    # beside it, the whole arrays the pass touches, each once (φ, b read, φ
    # written: 3 × 8 B per cell), the count used before φ and b were split
    arr = 3 * 8 * cells
    roofline["whole_array_bytes_per_launch"] = arr
    roofline["achieved_whole_arrays"] = arr / avg_s / 1e9

    extra = {}
    if not args.no_extra:
        t64, prof64, div64 = run_gpu(args.steps, args.warmup, 0)
        t32, prof32, div32 = run_gpu(args.steps, args.warmup, 1)
        extra["dcbl_256x256x128"] = {
            "value": NX * NY * NZ / t64, "ms_per_step": t64 * 1e3, "dtype": "f64",
            "fp32_state": {"value": NX * NY * NZ / t32, "ms_per_step": t32 * 1e3,
                           "form": "FP32 state (u, v, w, theta, p) and tendencies; FP64 projection"},
            "poisson_direct_ms": poisson_ms(), "max_divergence_after_step": div64,
            "ms_per_step_by_phase_f64": {k: round(v[1] / args.steps, 4) for k, v in prof64.items()},
            "workload": "dcbl 256x256x128 stretched-z, WENO-Z5 momentum+theta, SSP-RK3, FFT-xy + FP64 Thomas-z "
                        "projection per substage"}
        # the step's dominant kernel: the tiled tendency kernel, FP64
        n_t, ms_t = prof64["tendency"]
        tend_ms = ms_t / n_t if n_t else None
        alg_t = tendency_bytes_per_launch(8)
        valu = read_valu_insts()
        extra["dcbl_256x256x128"]["tendency_kernel"] = {
            "kernel": "adv_tile_kernel<MODE_STEP, WENO-Z5, double> (stencil.hip)",
            "avg_launch_ms": tend_ms, "algorithmic_bytes_per_launch": alg_t,
            "achieved_GBs": alg_t / (tend_ms / 1e3) / 1e9 if tend_ms else None,
            "traffic_bytes_per_launch": read_traffic(),
            "valu_insts_per_launch": valu,
            "valu_issue_floor_ms": valu * VALU_CYCLES_PER_INST / (N_SIMD * CLOCK_HZ) * 1e3 if valu else None}
        extra["advect_positive"] = tracer_leg()
        if not args.no_poisson:
            legs = poisson_legs(weights=args.weights, log=log)
            extra["poisson_cutcell_512x512x192"] = {
                "mgpcg_ms": legs["mgpcg_f32_jacobi"]["ms"], "learned_fcg_ms": learned_ms(legs), "legs": legs,
                "workload": "cut-cell 512x512x192, dx 2 m, 64 seeded buildings, source = div of a seeded k^-5/3 "
                            "velocity; to ||r|| <= 1e-8 ||b||"}

    cpu = None
    if rank == 0 and not args.no_cpu:
        threads = args.cpu_threads or min(os.cpu_count() or 1, 16)
        import aeolus_hip as hip
        from aeolus_hip import workloads as W
        from aeolus_hip.terrain import AnelasticTerrainSimulation, TerrainFollowingGrid
        # the GPU turn of the A/B alternation: one headline-form step on the target
        g, h, state, dt = W.terrain_workload(N)
        tg = TerrainFollowingGrid(g, h, g.Lz)
        sim = AnelasticTerrainSimulation(tg, scheme="weno_z5", tol=1e-8, maxit=200, **W.TERRAIN_PHYS,
                                         **TERRAIN_FORMS[HEAD_FORM])
        sim.set(*state)
        sim.project()
        gpu_ms = []

        def gpu_turn():
            hip.sync()
            t0 = time.perf_counter()
            sim.step_rk3(dt)
            hip.sync()
            gpu_ms.append((time.perf_counter() - t0) * 1e3)

        c = terrain_cpu_baseline(threads, reps=args.cpu_reps, gpu_turn=gpu_turn, log=log)
        del sim
        n_cpu = TERRAIN_CPU_N[0] * TERRAIN_CPU_N[1] * TERRAIN_CPU_N[2]
        cpu = {"value": n_cpu / c["min_s"], "unit": "cell-updates/s", "cores": threads, "kind": "port",
               "sample": f"CPU oracle (FP64, OpenMP, MG-PCG), the terrain workload at {TERRAIN_CPU_N[0]}x"
                         f"{TERRAIN_CPU_N[1]}x{TERRAIN_CPU_N[2]} (dx 50 m, 3 seeded hills), WENO-Z5 RK3 step "
                         f"projected to 1e-8, 1 warm-up then min of {args.cpu_reps} steps on {threads} threads "
                         f"({c['min_s']:.2f} s/step, median {c['median_s']:.2f}), alternating in turns with a GPU "
                         f"step of the FP64 form; one step on 1 thread {c['one_thread_s']:.2f} s",
               "value_median": n_cpu / c["median_s"], "value_1thread": n_cpu / c["one_thread_s"],
               "times_s": c["times_s"], "gpu_turn_ms": gpu_ms, "sensors": c["sensors"],
               "nproc": os.cpu_count()}

    out = {
        "metric": METRIC,
        "value": cells / (head["ms_per_step"] / 1e3),
        "unit": "cell-updates/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": head["ms_per_step"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {"workload": "anelastic flow over terrain 512x512x256 (Gal-Chen over 3 seeded Gaussian hills, "
                               "rho = 1.2 exp(-z/8 km), 10 m/s westerly), WENO-Z5 SSP-RK3 step, density-weighted "
                               "projection by MG-PCG to ||r|| <= 1e-8 ||b|| at every substage",
                   "grid": list(N), "dt": ter["dt"], "form": HEAD_FORM, "parallelism": "single-gpu"},
        "terrain": {
            HEAD_FORM: head,
            FAST_FORM: fast,
            "fast_form": {"name": FAST_FORM, "ms_per_step": fast["ms_per_step"],
                          "speedup_vs_fp64": fast["speedup_vs_" + HEAD_FORM],
                          "rel_error_vs_fp64": fast["rel_error_vs_" + HEAD_FORM],
                          "constraint_residual": fast["constraint_residual_after_step"],
                          "constraint_residual_fp64": head["constraint_residual_after_step"]},
            "learned_form": None,
            "spinup": ter["spinup"], "workload": ter["workload"],
        },
        "poisson_ms": {"mgpcg": None, "learned_fcg": None},
        "roofline": roofline,
        "stream_triad": triad,
        "cpu_baseline": cpu,
        "extra": extra,
        "host_sensors": {"start": sensors0, "end": host_sensors()},
        "provenance": provenance(device=0),
    }
    pc = extra.get("poisson_cutcell_512x512x192")
    if pc:
        out["poisson_ms"] = {"mgpcg": pc["mgpcg_ms"], "learned_fcg": pc["learned_fcg_ms"],
                             "workload": pc["workload"]}
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
