/*
 * libaeolus_hip — the C ABI of the MI355X (gfx950) dynamical-core step.
 *
 * Drop-in replacement, behind a C ABI, for the CPU path of badulion/Aeolus.jl
 * (Julia) for one fractional-step dynamical-core step: the WENO advection
 * tendencies (AdvectionSchemes), the SSP-RK3 stage updates (Simulations) and
 * the pressure projection (PressureSolvers). Every entry point cites the
 * reference interface it replaces (paths relative to the reference root).
 *
 * Conventions
 *  - All functions return an int status: AEO_OK (0) or a negative AEO_ERR_*;
 *    aeo_last_error() gives the text of the last failure (thread-local).
 *    Nothing throws across the ABI.
 *  - Field arrays are device pointers in the reference's storage layout
 *    (src/Grids.jl:98-140): (Nx+2H) x (Ny+2H) x (Nz+2H), column-major, x
 *    fastest, interior H .. H+N-1 (0-based) on every axis; FaceX/FaceY/FaceZ
 *    fields share this shape, face i being the west/south/bottom face of cell
 *    i. `precision` selects the element type: AEO_F64 (double) or AEO_F32
 *    (float). Solver buffers are FP64.
 *  - All work of the library is ordered on one HIP stream of the current
 *    context; calls return when the work is queued (aeo_sync waits).
 *    Use one context per host thread.
 */
#ifndef AEOLUS_HIP_H
#define AEOLUS_HIP_H
#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

enum {
    AEO_OK = 0,
    AEO_ERR_ARG = -1,          /* bad argument (reference: ArgumentError / DimensionMismatch) */
    AEO_ERR_HIP = -2,          /* a HIP runtime call failed                                  */
    AEO_ERR_UNSUPPORTED = -3,  /* a configuration this build does not implement              */
    AEO_ERR_STATE = -4         /* no context (aeo_init not called)                           */
};
enum { AEO_F64 = 0, AEO_F32 = 1 };
/* field locations, src/Grids.jl:60-83 */
enum { AEO_CELL = 0, AEO_FACE_X = 1, AEO_FACE_Y = 2, AEO_FACE_Z = 3 };
/* per-axis boundary kinds: Periodic, NoFlux (mirror), ImpermeableWall
 * (src/BoundaryConditions.jl:182-259) */
enum { AEO_PERIODIC = 0, AEO_NOFLUX = 1, AEO_WALL = 2 };
/* face reconstructions, advection_scheme names (src/AdvectionSchemes.jl:1704-1775) */
enum {
    AEO_CENTERED = 0, /* :centered  (advect_centered!, momentum_advect!)       */
    AEO_UPWIND = 1,   /* :upwind                                              */
    AEO_WENO5 = 2,    /* :weno5     (FiniteVolume advect_weno5!)              */
    AEO_WENO_JS5 = 3, /* :weno_js5                                            */
    AEO_WENO_Z5 = 4,  /* :weno_z5                                             */
    AEO_WENO_Z7 = 5,  /* :weno_z7                                             */
    AEO_TENO5 = 6,    /* :teno5     (TENO(5; C_T = 1e-5), q = 6)              */
    AEO_TENO8 = 7,    /* :teno8     (TENO(8; C_T = 1e-5), q = 6; halo 5)      */
    AEO_VARIANCE_CONSERVING = 8 /* :variance_conserving (regular grids)      */
};
/* pressure-solver status, pcg! (src/Backends.jl:1482-1487) */
enum { AEO_CONVERGED = 0, AEO_MAXIT = 1, AEO_BREAKDOWN = 2, AEO_ZERO_RHS = 3, AEO_DIRECT = 4 };

/* ---- context ------------------------------------------------------------ */
/* provenance of a run (provenance(), src/io/run_folder.jl:215-260): the
 * compiler, HIP version and target the library was built with (a static
 * string), and the device's name, gfx architecture, compute units and HBM */
const char *aeo_build_info(void);
int aeo_device_info(int device, char *name, size_t name_len, char *arch, size_t arch_len, int *cus,
                    size_t *mem_bytes);
/* No reference counterpart: selects the device and creates the stream. */
int aeo_init(int device);
int aeo_shutdown(void);
int aeo_sync(void);
const char *aeo_last_error(void);

/* ---- device memory (replaces the reference's Array storage of Field.data,
 *      src/Fields.jl:21-39; the caller owns what it allocates here) -------- */
int aeo_malloc(void **dptr, size_t bytes);
int aeo_free(void *dptr);
int aeo_memcpy_h2d(void *dst, const void *src, size_t bytes);
int aeo_memcpy_d2h(void *dst, const void *src, size_t bytes);
int aeo_memset(void *dptr, int value, size_t bytes);
/* device-to-device copy on the library's stream: a plain streaming copy kernel
 * when pointers and size are 16-byte aligned (also the kernel that calibrates
 * the HBM-traffic counters), the runtime's copy otherwise */
int aeo_memcpy_d2d(void *dst, const void *src, size_t bytes);
/* The STREAM triad a = b + s·c over n doubles on the library's stream
 * (timed under the name "triad"): no counterpart in the reference; the
 * device-bandwidth reference of the measurements (16n bytes read, 8n
 * written, 8-byte accesses like the solver's vector kernels). */
int aeo_stream_triad(double *a, const double *b, const double *c, double s, long long n);

/* ---- grids ---------------------------------------------------------------
 * RegularGrid (src/Grids.jl:98-140) when zf_interior is NULL (uniform dz);
 * StretchedGrid with (:custom, zf) stretching (src/StretchedGrids.jl:117-402)
 * when zf_interior holds the Nz+1 interior face heights: the faces are
 * extended into the halo (_extend_faces, :319-337) and the per-level metrics
 * built as level_metrics does (:570-600). */
typedef struct aeo_grid aeo_grid;
int aeo_grid_create(int Nx, int Ny, int Nz, int H, double dx, double dy, double dz, const double *zf_interior,
                    aeo_grid **g);
int aeo_grid_destroy(aeo_grid *g);
/* the storage-level metric vectors (host copies): idzc (Nz+2H), idzf (Nz+2H+1) */
int aeo_grid_metrics(const aeo_grid *g, double *idzc, double *idzf);

/* fill_halos!(field, bcs), src/BoundaryConditions.jl:182-259 */
int aeo_fill_halos(aeo_grid *g, int precision, void *field, int loc, int bc_x, int bc_y, int bc_z);

/* ---- advection operators: the AdvectionScheme callable
 * scheme(tend, u, v, w, ϕ) (src/AdvectionSchemes.jl:1712-1718), which ADDS
 * −∂(uⱼϕ)/∂xⱼ to tend; `p` is the WENO-Z τ exponent (1 or 2). Halos of the
 * inputs must be filled and H >= required_halo(scheme) (1 centred, upwind and
 * variance-conserving; 3 WENO-5 and TENO5; 4 WENO-Z7; 5 TENO8). The TENO
 * schemes use C_T = 1e-5 here (advection_scheme(:teno5), :1765-1767);
 * AEO_VARIANCE_CONSERVING is advect_variance_conserving! (:1428-1446). */
int aeo_advect_scalar(aeo_grid *g, int precision, int scheme, int p, void *tend, const void *u, const void *v,
                      const void *w, const void *phi);
/* advect_teno!(tend, u, v, w, ϕ; order, C_T, q) (src/AdvectionSchemes.jl:750-756):
 * order 5 or 8, cut-off C_T > 0; q = 6 (the reference's default) only */
int aeo_advect_teno(aeo_grid *g, int precision, int order, double C_T, int q, void *tend, const void *u,
                    const void *v, const void *w, const void *phi);
/* FluxLimiterWorkspace(mesh) (src/AdvectionSchemes.jl:800-822): scratch of
 * aeo_advect_positive for one grid and precision: the limiter ratio R, one
 * storage array (the face fluxes are recomputed where they are used) */
typedef struct aeo_flux_workspace aeo_flux_workspace;
int aeo_flux_limiter_workspace_create(aeo_grid *g, int precision, aeo_flux_workspace **ws);
int aeo_flux_limiter_workspace_destroy(aeo_flux_workspace *ws);
/* advect_positive!(tend, u, v, w, ϕ, dt; scheme, p, workspace, bcs, accumulate)
 * (src/AdvectionSchemes.jl:1135-1160): adds (accumulate = 1) or writes
 * (accumulate = 0) −∇·(u ϕ) over tend's interior with the face fluxes limited
 * so that ϕ + dt·tend ≥ 0 for ϕ ≥ 0 (halos included) under the first-order
 * CFL condition. scheme: AEO_CENTERED, AEO_WENO5 or AEO_WENO_JS5 (both
 * WENO-JS5 on this path), AEO_WENO_Z5, AEO_WENO_Z7, AEO_TENO5, AEO_TENO8
 * (cut-off C_T, ignored by the others); a stretched grid takes AEO_CENTERED
 * only. bcs: three AEO_* of ϕ for the limiter's halo, or NULL
 * for the reference's one-layer periodic wrap. ws may be NULL (a workspace
 * is then allocated and freed inside the call). */
int aeo_advect_positive(aeo_grid *g, int precision, int scheme, int p, double C_T, void *tend, const void *u,
                        const void *v, const void *w, const void *phi, double dt, aeo_flux_workspace *ws,
                        const int *bcs, int accumulate);
/* momentum_advect_weno_z!(tu, tv, tw, u, v, w) (src/AdvectionSchemes.jl:1195-1270)
 * and the momentum_advection keyword of step! (src/Simulations.jl:418-425):
 * ADDS −∂(uⱼuᵢ)/∂xⱼ to the face-centred tendencies. */
int aeo_advect_momentum(aeo_grid *g, int precision, int scheme, int p, void *tu, void *tv, void *tw, const void *u,
                        const void *v, const void *w);

/* ---- pressure solvers: AbstractPressureSolver (src/PressureSolvers.jl:19-80) */
typedef struct aeo_poisson aeo_poisson;
/* Sizes of the spectral solvers (FFTW takes any length; these hand-written
 * LDS transforms take mixed radices 2, 3, 4, 5): Nx even with Nx/2 a
 * product of 2, 3 and 5, Nx ≤ 2048; Ny a product of 2, 3 and 5, ≤ 512; for
 * the triply periodic solver Nz likewise, ≤ 512. Other sizes are refused
 * with AEO_ERR_ARG. */
/* FFTPoissonSolver(mesh), src/PressureSolvers.jl:103-174 (triply periodic) */
int aeo_poisson_fft_create(int Nx, int Ny, int Nz, double dx, double dy, double dz, aeo_poisson **h);
/* ColumnTridiagonalSolver(T, (Nx,Ny,Nz), (dx,dy); lower, upper, hweight,
 * measure, inv_coupling, gauge, bc_x, bc_y), src/PressureSolvers.jl:626-666.
 * Vectors are host arrays of length Nz (inv_coupling Nz+1). Lateral BCs:
 * AEO_PERIODIC (R2HC) or AEO_NOFLUX (REDFT10, the DCT-II). */
int aeo_poisson_column_create(int Nx, int Ny, int Nz, double dx, double dy, int bc_x, int bc_y,
                              const double *lower, const double *upper, const double *hweight,
                              const double *measure, const double *inv_coupling, const double *gauge,
                              aeo_poisson **h);
/* MGPreconditionedCG(mesh; coeff_x/y/z, rhs_scale, nu1, nu2, tol, maxit)
 * (src/Multigrid.jl:879-972): pcg! with one V-cycle as the preconditioner,
 * the mean projected, FP64 outer iteration. cx (nx+1, ny, nz), cy (nx,
 * ny+1, nz), cz (nx, ny, nz+1) are host face coefficients of ∇·(c∇φ) (all
 * NULL: the constant Laplacian); rhs_scale (nz, or NULL) scales the source
 * rows (the stretched operator, :632-658). smoother 0: red-black
 * Gauss-Seidel (the reference's), 1: damped Jacobi with weight omega.
 * vcycle_precision AEO_F64 or AEO_F32 (the V-cycle's arithmetic). BCs:
 * AEO_PERIODIC or AEO_NOFLUX per axis. stats: (CG iterations, ‖r‖/‖b‖,
 * status). */
int aeo_poisson_mgpcg_create(int nx, int ny, int nz, double dx, double dy, double dz, int bc_x, int bc_y, int bc_z,
                             const double *cx, const double *cy, const double *cz, const double *rhs_scale, int nu1,
                             int nu2, int smoother, double omega, int vcycle_precision, double tol, int maxit,
                             aeo_poisson **h);
/* MultigridPoissonSolver(mesh; ..., tol, maxcycles) (src/Multigrid.jl:531-861):
 * V-cycles (red-black Gauss-Seidel, FP64) until ‖r‖/‖b‖ < tol.
 * stats: (cycles, relative residual, status). */
int aeo_poisson_mg_create(int nx, int ny, int nz, double dx, double dy, double dz, int bc_x, int bc_y, int bc_z,
                          const double *cx, const double *cy, const double *cz, const double *rhs_scale, int nu1,
                          int nu2, double tol, int maxcycles, aeo_poisson **h);
/* cycle and fmg of MultigridPoissonSolver (src/Multigrid.jl:559-570,
 * 706-760): w_cycle 1 makes every cycle recurse twice on the coarser level
 * (:W; 0 is :V), in the multigrid solve and in MG-PCG's preconditioner; fmg 1
 * starts aeo_poisson_mg_create's cycles from the full-multigrid
 * (nested-iteration) guess. Multigrid-based solvers only. */
int aeo_poisson_mg_set_cycle(aeo_poisson *h, int w_cycle, int fmg);
/* mg_level_count (src/Multigrid.jl:628): the hierarchy depth (1 for direct solvers) */
int aeo_poisson_levels(aeo_poisson *h, int *levels);
/* _apply_fine! (src/Multigrid.jl:911-917): out = A x on interior-sized FP64
 * device arrays (multigrid solvers) */
int aeo_poisson_apply(aeo_poisson *h, double *out, const double *x);
/* source_buffer(solver) (src/PressureSolvers.jl:57-69): the device FP64
 * interior-sized (Nx, Ny, Nz) array the caller may write the source into */
int aeo_poisson_source_buffer(aeo_poisson *h, double **dptr);
/* solve_source_buffer!(p, solver) (:71-80): φ into the device FP64
 * interior-sized array phi (the buffer is overwritten) */
int aeo_poisson_solve_source_buffer(aeo_poisson *h, double *phi);
/* solve!(p, source, solver) (:19-41): storage-layout fields of halo H; p's
 * interior is written, its halo untouched */
int aeo_poisson_solve(aeo_poisson *h, int precision, void *p, const void *source, int H);
/* solve!(p::Field{CellCenter}, source::Field{CellCenter}, solver) (:19-41)
 * as `_project_velocity!` calls it (src/Simulations.jl:714-723) for a
 * solver whose source_buffer is nothing: p and source are HOST FP64
 * storage arrays of halo H (a CPU Field's data, column-major); the
 * source's interior goes up, φ comes back into p's interior, p's halo is
 * untouched. Returns when p is written. */
int aeo_poisson_solve_host(aeo_poisson *h, double *p, const double *source, int H);
/* solver_stats(solver) (:43-55): (iterations, residual); direct solvers (0, NaN) */
int aeo_poisson_stats(aeo_poisson *h, int *iterations, double *residual, int *status);
int aeo_poisson_destroy(aeo_poisson *h);

/* ---- the step: BoussinesqSimulation + step_rk3! / step! -------------------
 * (src/Simulations.jl:168-288, 531-650, 711-744, 843-904) with the momentum
 * advection and the scalar (θ) advection of the given schemes. */
typedef struct {
    int mom_scheme, scal_scheme, weno_p;
    double nu, theta0, g_accel, flux_bot, flux_top;
    int bc_x, bc_y, bc_z;    /* velocity BCs (sim.bcs)  */
    int tbc_x, tbc_y, tbc_z; /* θ BCs (sim.θ_bcs)        */
    int precision;           /* of the state arrays and the tendency arithmetic */
} aeo_step_params;
typedef struct aeo_stepper aeo_stepper;
int aeo_stepper_create(aeo_grid *g, const aeo_step_params *sp, aeo_poisson *solver, aeo_stepper **h);
int aeo_stepper_destroy(aeo_stepper *h);
/* step_rk3!(sim, dt): u, v, w, theta, p are the state arrays (device, storage
 * layout), updated in place */
int aeo_step_rk3(aeo_stepper *h, void *u, void *v, void *w, void *theta, void *p, double dt);
/* f_coriolis of BoussinesqSimulation (src/Simulations.jl:269-283): the
 * f-plane term tu += f·v̄, tv −= f·ū of _b_coriolis! (src/FiniteVolume.jl:900-911),
 * added after buoyancy (_euler_projection! step 6, :602-605); 0 turns it off */
int aeo_stepper_set_coriolis(aeo_stepper *h, double f);
/* sponge_α_max, sponge_z_start, sponge_target of BoussinesqSimulation and
 * add_velocity_sponge! (src/Simulations.jl:272-274, 334-381): the Rayleigh
 * sponge −λ(z)(f − f_target) on u, v, w with λ = α_max sin²(½π(z − z_start)/(z_top − z_start))
 * for z ≥ z_start (sponge_profile, damping_rate, src/FiniteVolume.jl:524-566).
 * zc, zf: the Nz interior level heights of centres (u, v) and z faces (w),
 * damping_coordinates (src/FiniteVolume.jl:695, src/StretchedGrids.jl:602);
 * target_u/v/w: Nz-level vectors, NULL for zero. α_max = 0 or z_start ≥ z_top
 * turns the sponge off. */
int aeo_stepper_set_sponge(aeo_stepper *h, double alpha_max, double z_start, double z_top, const double *zc,
                           const double *zf, const double *target_u, const double *target_v,
                           const double *target_w);
/* C_s and Pr_t of BoussinesqSimulation (src/Simulations.jl:237-238, 270):
 * the built-in closure StaticSmagorinsky(C_s) (src/operators/sgs_closures.jl:
 * 309-318, 403-425) with sgs_stress = :laplacian: νt = (C_s Δ_k)²|S|
 * (src/FiniteVolume.jl:930-944), ∂_j(νt ∂_j u_i) on u, v, w (:966-1042) and
 * (1/Pr_t)∂_j(νt ∂_j θ) on θ (:1280-1300), every substage, after ν∇².
 * C_s = 0 turns the closure off. */
int aeo_stepper_set_sgs(aeo_stepper *h, double C_s, double Pr_t);
/* The state maxima of cfl_diagnostics (src/TimeIntegration.jl:291-400):
 * fills the halos of u, v, w (the velocity BCs), then rate = max Σ|u_i|/Δx_i
 * (_max_advective_rate), nut_max = max νt of the step's Smagorinsky closure
 * computed from this state (0 without a closure), N = √max(0, max_k
 * g/θ₀·(θ̄_k − θ̄_{k−1})/Δz_f[k]) from the plane means θ̄_k of theta
 * (_brunt_vaisala, :209-232; 0 without buoyancy). The time-step limits
 * follow on the host (the Python mirror's cfl_diagnostics / adaptive_dt). */
int aeo_stepper_cfl(aeo_stepper *h, void *u, void *v, void *w, const void *theta, double *rate, double *nut_max,
                    double *N);
/* step!(sim, dt) (src/Simulations.jl:474-487): one projected forward-Euler step */
int aeo_step_euler(aeo_stepper *h, void *u, void *v, void *w, void *theta, void *p, double dt);

/* ---- the sound-proof (mass-weighted) core, regular grids ------------------
 * _mass_weighted_step! (src/Anelastic.jl:1791-1876) with the anelastic
 * weighting W = ρ̄: weighted momentum and scalar advection (centred, the
 * reference's forms :1170-1311), ν∇², the anelastic buoyancy
 * g(θ_face − θ̄_f)/θ̄_f (:1328-1360), the surface heat flux, the predictor,
 * _project_mass_weighted! (:1756-1778: ∇·(W∇φ) = ∇·(W u*) with `solver`, the
 * density-weighted column solver, u ← u* − ∇φ), θ += Δt tθ, p = φ/Δt.
 * Wc, Wf, thetabar_f: host arrays of the halo-padded ReferenceState
 * profiles ρ̄c_pad, ρ̄f_pad, θ̄f_pad (Nz + 2H entries, storage-level index). */
typedef struct {
    double nu, g_accel, flux_bot, flux_top;
    int buoyancy;
    int bc_x, bc_y, bc_z;    /* velocity BCs */
    int tbc_x, tbc_y, tbc_z; /* θ BCs */
    int precision;
} aeo_mw_params;
typedef struct aeo_mw_stepper aeo_mw_stepper;
int aeo_mw_stepper_create(aeo_grid *g, const aeo_mw_params *p, const double *Wc, const double *Wf,
                          const double *thetabar_f, aeo_poisson *solver, aeo_mw_stepper **h);
int aeo_mw_stepper_destroy(aeo_mw_stepper *h);
int aeo_mw_step(aeo_mw_stepper *h, void *u, void *v, void *w, void *theta, void *p, double dt);
/* f_coriolis and sponge_α_max, sponge_z_start, sponge_target of a sound-proof
 * core (_build_mass_weighted, src/Anelastic.jl:1559-1625; step 6 of
 * _mass_weighted_step!, :1849-1852): the same terms and arguments as
 * aeo_stepper_set_coriolis / aeo_stepper_set_sponge */
int aeo_mw_stepper_set_coriolis(aeo_mw_stepper *h, double f);
int aeo_mw_stepper_set_sponge(aeo_mw_stepper *h, double alpha_max, double z_start, double z_top, const double *zc,
                              const double *zf, const double *target_u, const double *target_v,
                              const double *target_w);
/* C_s and Pr_t of a sound-proof core: StaticSmagorinsky(C_s) with the
 * W-weighted SGS fluxes (1/W)∇·(W νt ∇u_i), (1/W)∇·(W κt ∇θ), κt = νt/Pr_t
 * (flux_weights, src/operators/sgs_closures.jl:200-217; _vertical_divergence,
 * src/FiniteVolume.jl:1556-1563). C_s = 0 turns the closure off. */
int aeo_mw_stepper_set_sgs(aeo_mw_stepper *h, double C_s, double Pr_t);
/* step_rk3! of the sound-proof core (src/Anelastic.jl:1905-1945): three
 * aeo_mw_step stages; the whole storage of u, v, w, θ combined as
 * ¾·start + ¼·f after the second and ⅓·start + ⅔·f after the third */
int aeo_mw_step_rk3(aeo_mw_stepper *h, void *u, void *v, void *w, void *theta, void *p, double dt);
/* weighted_divergence!(out, u, v, w, Wc, Wf; normalize) (src/Anelastic.jl:1082-1110):
 * out's interior; Wc, Wf device arrays (Nz + 2H + 1 entries) */
int aeo_weighted_divergence(aeo_grid *g, int precision, void *out, const void *u, const void *v, const void *w,
                            const double *Wc, const double *Wf, int normalize);

/* ---- the adaptive step's checks ------------------------------------------- */
/* step_guard(sim) (src/TimeIntegration.jl:673-710): fills the velocity halos
 * with the stepper's BCs, then in one sweep over the interior: *finite = 1
 * when every u, v, w, θ and p value is finite, *divergence = max |∇·u| (the
 * bits of aeo_max_divergence), *speed = max(|u|, |v|, |w|); both maxima
 * propagate NaN */
int aeo_stepper_guard(aeo_stepper *h, void *u, void *v, void *w, const void *theta, const void *p, int *finite,
                      double *divergence, double *speed);
/* step_guard(sim::MassWeightedSimulation) (src/Anelastic.jl:2333-2346): the
 * same, with *divergence the core's constraint residual max |(1/W_c)∇·(W u)|
 * (constraint_residual, :2035-2044) */
int aeo_mw_stepper_guard(aeo_mw_stepper *h, void *u, void *v, void *w, const void *theta, const void *p,
                         int *finite, double *divergence, double *speed);
/* the state maxima of adaptive_dt(sim::MassWeightedSimulation)
 * (src/Anelastic.jl:2240-2290): the advective rate, max νt of the closure
 * recomputed from the state (0 without one) and N from the plane means of θ
 * with their local mean as θ_ref (0 without buoyancy); the velocity halos are
 * filled */
int aeo_mw_stepper_cfl(aeo_mw_stepper *h, void *u, void *v, void *w, const void *theta, double *rate,
                       double *nut_max, double *N);

/* ---- diagnostics (halos of the inputs filled) ------------------------------ */
/* max_divergence (src/Simulations.jl:1045-1050) */
int aeo_max_divergence(aeo_grid *g, int precision, const void *u, const void *v, const void *w, double *out);
/* max_divergence without allocating. No counterpart in the reference: it is
 * for callers that cannot allocate device memory (code under HIP graph
 * capture, tight serving loops, harnesses that forbid hipMalloc). The same
 * value as aeo_max_divergence; its per-level partials live in a fixed device
 * array of the library (4097 doubles per device, bound at aeo_init), so it
 * calls no hipMalloc/hipFree and serves Nz <= 4096 (larger Nz is an
 * AEO_ERR_ARG). Every call on one device shares that device's array: calls
 * that overlap on one device (two threads or two contexts) race. */
int aeo_max_divergence_noalloc(aeo_grid *g, int precision, const void *u, const void *v, const void *w, double *out);
/* _max_advective_rate (src/TimeIntegration.jl:164-182): dt = C / rate */
int aeo_max_advective_rate(aeo_grid *g, int precision, const void *u, const void *v, const void *w, double *out);
/* kinetic_energy (src/Simulations.jl:992-1015): ½ Σ (u² + v² + w²) dV with u,
 * v, w as stored on their faces (per-level volumes on a stretched grid) */
int aeo_kinetic_energy(aeo_grid *g, int precision, const void *u, const void *v, const void *w, double *out);

/* ---- cut-cell operators on a regular grid (src/CutCell.jl:602-781) --------
 * Geometry arrays ax, ay, az (face apertures) and vol_eff (effective volume
 * fractions, 0 in solid cells) are FP64 storage-layout device arrays, as
 * CutCellGeometry holds them (:177-195). */
/* cutcell_divergence!(div, u, v, w, geom; redistribute = false) (:602-626):
 * div's interior; solid cells 0 */
int aeo_cutcell_divergence(aeo_grid *g, int precision, void *div, const void *u, const void *v, const void *w,
                           const double *ax, const double *ay, const double *az, const double *vol_eff);
/* _redistribute_small_cells! (src/CutCell.jl:628-648), the second half of
 * cutcell_divergence!(…; redistribute = true): for each (cell, partner)
 * pair in order, both take (V_s d_s + V_t d_t)/(V_s + V_t), V = vol_eff.
 * pairs: device int32 array of 2·npairs 0-based storage linear indices, the
 * small cells (not solid, vol < vol_min) of the interior in the loop order,
 * each with its merge partner (src/CutCell.jl:466-488). Pairs outside the
 * grid's storage are skipped. */
int aeo_cutcell_redistribute(aeo_grid *g, int precision, void *div, const double *vol_eff, const int *pairs,
                             int npairs);
/* cutcell_gradient_x!/_y!/_z! (:666-700): a·(p⁺ − p⁻)/Δ on the interior
 * faces (face i = west face of cell i); p FP64 storage layout, halo filled */
int aeo_cutcell_gradient(aeo_grid *g, int precision, void *gx, void *gy, void *gz, const double *p,
                         const double *ax, const double *ay, const double *az);
/* cutcell_laplacian!(out, f, geom; aperture_power) (:735-781); power 2 is D·G */
int aeo_cutcell_laplacian(aeo_grid *g, int precision, void *out, const void *f, const double *ax, const double *ay,
                          const double *az, const double *vol_eff, int aperture_power);
/* The cut-cell projection (the fractional step of :580-594 with D and G):
 * the source vol_eff·(D u*) of the symmetric operator vol_eff·D·G (face
 * coefficients a², an MG-preconditioned CG's form) into solver's source
 * buffer, projected to zero mean over the fluid cells (vol_eff > 0) with the
 * solid cells 0, so that the singular system is consistent; then, with φ from aeo_poisson_solve_source_buffer (interior-sized
 * FP64, boundary neighbours by bc: periodic or Neumann),
 * u ← u − scale·G φ on the interior faces. */
int aeo_cutcell_project_source(aeo_grid *g, int precision, aeo_poisson *solver, const void *u, const void *v,
                               const void *w, const double *ax, const double *ay, const double *az,
                               const double *vol_eff);
int aeo_cutcell_project_correct(aeo_grid *g, int precision, void *u, void *v, void *w, const double *phi,
                                const double *ax, const double *ay, const double *az, int bc_x, int bc_y, int bc_z,
                                double scale);

/* ---- terrain-following (Gal-Chen) operators, src/StretchedGrids.jl:608-1343 -
 * z = h + σ(H − h)/H over the regular base grid g. h_plane: the terrain on
 * the (Nx+2H) x (Ny+2H) storage plane (x fastest); lid: H (> max h);
 * sigc, sigf, dzc, dzf: σ of the cell centres and faces and Δσ_c, Δσ_f per
 * storage level (host, Nz+2H each). The metrics (J, J at faces, σ_x, σ_y at
 * faces, terrain_following_grid :777-835) are evaluated on the fly from the
 * plane and its centred slopes (_slopes, :742-762). bc_x, bc_y: the lateral
 * maps of interior-sized vectors (periodic or Neumann); σ is mirrored. */
typedef struct aeo_terrain aeo_terrain;
int aeo_terrain_create(aeo_grid *g, const double *h_plane, double lid, const double *sigc, const double *sigf,
                       const double *dzc, const double *dzf, int bc_x, int bc_y, aeo_terrain **t);
int aeo_terrain_destroy(aeo_terrain *t);
/* _b_tf_divergence! with _tf_Ω (:1180-1205): out's interior, FP64 storage fields with filled halos */
int aeo_terrain_divergence(aeo_terrain *t, double *out, const double *u, const double *v, const double *w);
/* _laplacian!(out, f, ::TerrainFollowingGrid) for a cell-centred f (:1285-1343) */
int aeo_terrain_laplacian(aeo_terrain *t, double *out, const double *f);
/* out = J·∇²x on interior-sized FP64 vectors (the symmetric operator of the terrain Poisson problem) */
int aeo_terrain_apply(aeo_terrain *t, double *out, const double *x);
/* The terrain Poisson solve J∇²φ = b (no reference counterpart: the
 * reference has no solver for this operator): flexible CG on the full
 * metric operator, preconditioned by one V-cycle of `base`, an
 * MG-preconditioned CG on its diagonal-metric 7-point part (face
 * coefficients J_x, J_y, J·G^σσ). Stats as for MGPreconditionedCG. */
int aeo_poisson_terrain_create(aeo_terrain *t, aeo_poisson *base, double tol, int maxit, aeo_poisson **h);

/* ---- the anelastic core over Gal-Chen terrain ------------------------------
 * No counterpart as a whole: the reference's cores refuse a terrain grid
 * (src/Simulations.jl:1160-1163; src/Anelastic.jl:1558-1559). It composes
 * the reference's terrain metrics and contravariant flux _tf_Ω
 * (src/StretchedGrids.jl:777-835, 1180-1205) with the W-weighted flux forms,
 * weighted_divergence! and the step structure of _mass_weighted_step!
 * (src/Anelastic.jl:1082-1110, 1192-1311, 1756-1876) and its SSP-RK3
 * (:1905-1945), W = ρ̄(z) = rho0·exp(−z/Hs) of the physical height z.
 * The pressure operator is L = B·G with B u = δx(ρJ_x u) + δy(ρJ_y v) + δσ(ρΩ)
 * and G = −M⁻¹Bᵀ (symmetric; over flat terrain the operator of
 * DirectWeightedPoissonSolver, :987-1050). It is solved by pcg!
 * (src/Backends.jl:1461-1591) on L with one multigrid V-cycle of L's
 * 7-point part as preconditioner (MGPreconditionedCG, src/Multigrid.jl:
 * 879-972). The terrain grid must have a uniform σ spacing, periodic
 * lateral maps and a halo of at least 3; every field is FP64 storage
 * layout; interior-sized vectors are (Nx, Ny, Nz) FP64, x fastest. */
typedef struct aeo_tf_stepper aeo_tf_stepper;
typedef struct {
    double rho0, Hs;          /* ρ̄(z) = rho0·exp(−z/Hs) */
    double theta0, gamma;     /* θ̄(z) = theta0 + gamma·z: the anelastic buoyancy's reference */
    double g_accel;
    int buoyancy;
    int scheme;               /* AEO_CENTERED or AEO_WENO_Z5 (p = 2), for u, v, w and θ */
    int flux_precision;       /* AEO_F64, or AEO_F32: the tendency arithmetic (the state stays FP64) */
    int vcycle_precision;     /* AEO_F64 or AEO_F32: the preconditioner's levels (the outer CG is FP64) */
    int smoother, nu1, nu2;   /* 0 red-black Gauss-Seidel, 1 Jacobi (damped, ω = 0.8); pre- and post-sweeps */
    double tol;               /* ‖r‖ ≤ tol·‖b‖ */
    int maxit;
    int warm_start;           /* 0: zero guess (pcg!'s zero_guess = true); 1: the previous solve's φ; 2: per
                               * substage, 2φ(n−1) − φ(n−2) of the same substage of the last two steps (φ(n−1)
                               * after one step, the previous solve's φ before); 3: per substage, the quadratic
                               * 3φ(n−1) − 3φ(n−2) + φ(n−3) (linear, then φ(n−1), while fewer steps are
                               * kept); 4: the least-squares guess, Σ α_i φ_i over the last `basis` solves (of every
                               * substage) with α minimising ‖b − Σ α_i b_i‖ over their sources b_i; 1 to 4
                               * are zero_guess = false */
    int basis;                /* warm_start 4: solutions kept, 1..16 */
} aeo_tf_params;
int aeo_tf_stepper_create(aeo_terrain *t, const aeo_tf_params *p, aeo_tf_stepper **h);
int aeo_tf_stepper_destroy(aeo_tf_stepper *h);
/* the state halos: u, v, θ periodic in x, y and mirrored below the ground and
 * above the lid; w's ground and lid faces from Ω = 0, its halos antisymmetric
 * about them (theta nullable) */
int aeo_tf_fill_halos(aeo_tf_stepper *h, double *u, double *v, double *w, double *theta);
/* the tendencies of _mass_weighted_step! (steps 2 and 5) over the terrain, from
 * the state as given (halos filled); tw is 0 on the ground face */
int aeo_tf_tendencies(aeo_tf_stepper *h, double *tu, double *tv, double *tw, double *tt, const double *u,
                      const double *v, const double *w, const double *theta);
/* B u (weighted_divergence!, normalize = false) into an interior-sized vector */
int aeo_tf_divergence(aeo_tf_stepper *h, double *out, const double *u, const double *v, const double *w);
/* G φ: gx, gy at the x-/y-face of each cell, gw at its bottom σ-face (0 on the ground) */
int aeo_tf_gradient(aeo_tf_stepper *h, double *gx, double *gy, double *gw, const double *phi);
/* L x = B(G x) */
int aeo_tf_apply(aeo_tf_stepper *h, double *out, const double *x);
/* L φ = b with the stepper's solver (solve!, src/PressureSolvers.jl:19-41) */
int aeo_tf_solve(aeo_tf_stepper *h, double *phi, const double *b);
/* one mass-weighted step: halos, tendencies, predictor, B u*, L φ = B u*,
 * u = u* − Gφ, θ += Δt tθ, p = φ/Δt (_mass_weighted_step!) */
int aeo_tf_step(aeo_tf_stepper *h, double *u, double *v, double *w, double *theta, double *p, double dt);
/* step_rk3! of the core: three substeps, (¾, ¼) and (⅓, ⅔) combinations */
int aeo_tf_step_rk3(aeo_tf_stepper *h, double *u, double *v, double *w, double *theta, double *p, double dt);
/* the projection alone (_project_mass_weighted!, src/Anelastic.jl:1756-1778):
 * u ← u − Gφ with Lφ = B u, so that B u = 0 (a solenoidal start for step_rk3) */
int aeo_tf_project(aeo_tf_stepper *h, double *u, double *v, double *w);
/* solver_stats of the last solve (relative residuals: the recursion's, the
 * one recomputed in FP64 from the solution and the initial guess's), and the
 * iterations of the last step */
int aeo_tf_stats(aeo_tf_stepper *h, int *iterations, double *residual, double *true_residual, int *status,
                 int *total_iterations, double *initial_residual);
/* the iterations and initial relative residuals of the last step's solves
 * (three for step_rk3, one for a step; arrays of 3) */
int aeo_tf_step_history(aeo_tf_stepper *h, int *iterations, double *initial_residuals);
/* constraint_residual (src/Anelastic.jl:2035-2044): max |B u|/(ρ̄ J), the
 * velocity halos filled first */
int aeo_tf_constraint_residual(aeo_tf_stepper *h, double *u, double *v, double *w, double *out);

/* ---- the learned preconditioner ------------------------------------------
 * No reference counterpart: the reference has no network (its nearest hook
 * is src/ML.jl:40-56). A 3-level 3-D U-Net on an nx x ny x nz grid (each
 * divisible by 4): 3x3x3 convolutions with 16/32/64 channels, bias and
 * ReLU, 2x2x2 mean pooling, nearest upsampling, skip concatenation and a
 * 1x1 head; periodic in x and y, zero-padded in z. BF16 weights and
 * activations on MFMA, FP32 accumulation, FP32 master weights and Adam.
 * The source is normalised by its RMS on the way in and the output scaled
 * back. in_channels: 1 (source) or 2 (source and fluid mask). */
typedef struct aeo_unet aeo_unet;
int aeo_unet_create(int nx, int ny, int nz, int in_channels, unsigned long long seed, aeo_unet **h);
int aeo_unet_destroy(aeo_unet *h);
int aeo_unet_num_params(aeo_unet *h, long long *n);
/* the FP32 master parameters (per 3x3x3 layer W[tap][c][n] then b[n]; the
 * head's 16 weights and bias last); setting them resets Adam */
int aeo_unet_get_params(aeo_unet *h, float *host);
int aeo_unet_set_params(aeo_unet *h, const float *host);
/* out = network(src, mask): FP64 interior-sized device arrays (mask NULL
 * for one input channel) */
int aeo_unet_forward(aeo_unet *h, const double *src, const double *mask, double *out);
/* the loss mean((net − target/rms(src))²) of one sample and, if grad_host,
 * its gradient (host FP32, num_params) */
int aeo_unet_gradients(aeo_unet *h, const double *src, const double *mask, const double *target, float *grad_host,
                       float *loss);
/* one Adam step (β = 0.9, 0.999) on one sample; loss may be NULL */
int aeo_unet_train_step(aeo_unet *h, const double *src, const double *mask, const double *target, float lr,
                        float *loss);
/* The weight and bias gradients of one 3x3x3 convolution of that network, the
 * kernels its training runs: in (nx*ny*nz x cin) and dy (x cout) are BF16,
 * channels last, x fastest among the voxels, dw[tap][c][n] (tap = dx + 1 +
 * 3 (dy + 1) + 9 (dz + 1)) and db[n] FP32, all on the device. (cin, cout) is one
 * of the layers': (8, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64),
 * (96, 32), (48, 16). plan, if given: the rows of a task, the tasks and the
 * blocks that shared them out. */
int aeo_conv3_weight_gradient(int cin, int cout, int nx, int ny, int nz, const void *in, const void *dy, float *dw,
                              float *db, int *plan);
/* Flexible CG (Notay 2000, one previous direction kept) on the operator of
 * an MG-preconditioned CG solver `base` (same grid as the network), with
 * the network as initial guess (use_guess) and preconditioner. mode 0: the
 * network; 1: the network, then one V-cycle of `base` on the residual it
 * leaves; 2: the V-cycle only. The operator's null space (constants) is
 * projected out. Stats as for MGPreconditionedCG. */
int aeo_poisson_fcg_create(aeo_poisson *base, aeo_unet *net, const double *mask, int mode, int use_guess, double tol,
                           int maxit, aeo_poisson **h);

/* ---- kernel timing (no reference counterpart; the timing the benchmark and
 * the roofline read): HIP events around every launch of the named kernels on
 * the library's stream */
int aeo_profile_enable(int on);
int aeo_profile_reset(void);
/* kernel names: "tendency", "advect", "halo", "divergence", "correct",
 * "poisson", "shell" */
int aeo_profile_get(const char *kernel, int *count, double *total_ms);

/* The levels of a column that one block of a marching kernel works through on
 * a grid of this size (no reference counterpart; computed on the host, no GPU
 * needed): "tendency" (also momentum advection), "scalar", "limited",
 * "terrain_tendency", "terrain_apply", "terrain_smooth", "terrain_prolong" */
int aeo_launch_levels(const char *kernel, int Nx, int Ny, int Nz, int *levels);

#ifdef __cplusplus
}
#endif
#endif
