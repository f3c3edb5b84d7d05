// Launchers of the gfx950 kernels (internal to libaeolus_hip).
#pragma once
#include "common.h"

namespace aeo {

// Set-up transfers. The library's stream is created hipStreamNonBlocking, so
// it does not wait for work queued on the null stream, where hipMemset and
// hipMemcpy run, and hipMemset may return before the memory is cleared.
// Memory cleared or uploaded at set-up is therefore waited for before the
// call returns: a kernel later launched on the library's stream sees it.
inline hipError_t zero_dev(void *p, size_t bytes) {
    const hipError_t e = hipMemset(p, 0, bytes);
    return e == hipSuccess ? hipDeviceSynchronize() : e;
}
inline hipError_t upload_dev(void *dst, const void *src, size_t bytes) {
    const hipError_t e = hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice);
    return e == hipSuccess ? hipDeviceSynchronize() : e;
}

// Physics of one substage of the step (src/Simulations.jl:168-288 fields).
struct StepPhys {
    double nu, dt, theta0, g_accel, flux_bot, flux_top;
    double idz_bot, idz_top;  // 1/Δz_c of the bottom and top interior levels
    double fcor;              // f-plane Coriolis parameter (0: off)
    // Rayleigh sponge: device vectors of the state's type, 5 × (Nz + 2H),
    // storage-level index: rate at centres, rate at z faces, targets of u, v, w
    // (nullptr: off)
    const void *sponge;
};

// The RK3 stage combination c(x, snap) = a·snap + b·x of step_rk3!
// (src/Simulations.jl:884-896): stage 2 (3/4, 1/4), stage 3 (1/3, 2/3).
template <typename T>
inline void stage_coeffs(int stage, const StepPhys *, T *a, T *b, int *combine) {
    if (stage == 2) { *a = T(0.75); *b = T(0.25); *combine = 1; }
    else if (stage == 3) { double inv3 = 1.0 / 3; *a = T(inv3); *b = T(2 * inv3); *combine = 1; }
    else { *a = T(0); *b = T(1); *combine = 0; }
}

template <typename T>
void launch_halo(hipStream_t st, T *d, int Nx, int Ny, int Nz, int H, int loc, int bcx, int bcy, int bcz);
// up to four fields of one grid, each with its own BCs; wall_w[f] = the field
// is w (FaceZ) under a z wall (the wall plane zeroed, an antisymmetric halo)
template <typename T> struct HaloSet {
    T *d[4];
    int bc[4][3];
    int wall_w[4];
    int n;
    void add(T *p, int loc, int bx, int by, int bz) {
        d[n] = p;
        bc[n][0] = bx; bc[n][1] = by; bc[n][2] = bz;
        wall_w[n] = (loc == LOC_FZ && bz == BC_WALL) ? 1 : 0;
        n++;
    }
};
template <typename T>
void launch_halo_multi(hipStream_t st, const HaloSet<T> &hs, int Nx, int Ny, int Nz, int H);
template <typename T>
int launch_advect(hipStream_t st, const Metrics<T> &m, int mode, int scheme, int p, const T *u, const T *v,
                  const T *w, const T *s, T *tu, T *tv, T *tw, T *ts);
template <typename T>
int launch_tendency_step(hipStream_t st, const Metrics<T> &m, int scheme, int p, const T *u, const T *v, const T *w,
                         const T *s, T *uo, T *vo, T *wo, T *so, const T *s0, const StepPhys &ph, int stage);
// the static Smagorinsky closure (sgs.hip)
template <typename T>
void launch_smag_nut(hipStream_t st, const Metrics<T> &m, T *nut, const T *u, const T *v, const T *w, const T *coef,
                     const T *idz_off);
template <typename T>
void launch_smag_apply(hipStream_t st, const Metrics<T> &m, T *us, T *vs, T *ws, T *so, const T *u, const T *v,
                       const T *w, const T *th, const T *nut, double dt, double bt, double sc);
template <typename T>
void launch_smag_apply_weighted(hipStream_t st, const Metrics<T> &m, T *us, T *vs, T *ws, T *tn, const T *u,
                                const T *v, const T *w, const T *th, const T *nut, T *kap, const double *Wc,
                                const double *Wf, double Pr_t, double dt);
template <typename T>
void launch_div_into(hipStream_t st, double *buf, const T *u, const T *v, const T *w, const Metrics<double> &md);
template <typename T>
void launch_correct(hipStream_t st, T *uo, T *vo, T *wo, const T *us, const T *vs, const T *ws, const T *u0,
                    const T *v0, const T *w0, const double *phi, T *p, const Metrics<double> &md, int bcx, int bcy,
                    int bcz, double ca, double cb, int combine, double dt, T *th = nullptr, const T *tn = nullptr,
                    const T *th0 = nullptr);
// up to four (out, x, snap) triples whose halo shells are combined in one launch
template <typename T> struct ShellSet {
    T *out[4];
    const T *x[4];
    const T *snap[4];
    int n;
    void add(T *o, const T *xx, const T *sn) {
        out[n] = o; x[n] = xx; snap[n] = sn;
        n++;
    }
};
template <typename T>
void launch_shell(hipStream_t st, const ShellSet<T> &ss, int Nx, int Ny, int Nz, int H, double ca, double cb);
template <typename T>
void launch_plane_sum(hipStream_t st, double *out, const T *f, const Metrics<double> &md);
template <typename T>
void launch_varcons(hipStream_t st, const Metrics<T> &m, T *tend, const T *u, const T *v, const T *w, const T *phi);
template <typename T>
int launch_advect_positive(hipStream_t st, const Metrics<T> &m, int scheme, int p, T *tend, const T *u, const T *v,
                           const T *w, const T *phi, T dt, T *ratio, const int *bcs, int accumulate);
template <typename T>
void launch_guard(hipStream_t st, double *part, int nblocks, const T *u, const T *v, const T *w, const T *th,
                  const T *p, const double *Wc, const double *Wf, const Metrics<double> &md);
template <typename T>
void launch_diag(hipStream_t st, double *part, int nblocks, const T *u, const T *v, const T *w,
                 const Metrics<double> &md, int what);

// ---- the allocation-free maximum divergence (noalloc.hip) ----
// Largest Nz it serves (one partial per level in a fixed device array), and
// the devices whose array address is kept.
constexpr int NOALLOC_MAX_LEVELS = 4096;
constexpr int NOALLOC_MAX_DEVICES = 64;
// with `device` current: bind the device's address of the file-scope scratch
hipError_t noalloc_bind(int device);
// the bound address (nullptr before noalloc_bind)
double *noalloc_scratch(int device);
// per-level maxima of |∇·u| into part[0 .. Nz), their maximum into part[NOALLOC_MAX_LEVELS]
template <typename T>
void launch_maxdiv_noalloc(hipStream_t st, double *part, const T *u, const T *v, const T *w,
                           const Metrics<double> &md);

// ---- the sound-proof core (anelastic.hip) ----
struct MWPhys {
    double nu, dt, g_accel, fb, ft;  // fb, ft: surface fluxes times 1/Δz
    int buoyancy;
    double fcor;         // f-plane Coriolis parameter (0: off)
    const void *sponge;  // as StepPhys::sponge (nullptr: off)
};
template <typename T>
void launch_mw_tendency(hipStream_t st, const Metrics<T> &m, T *us, T *vs, T *ws, T *tn, const T *u, const T *v,
                        const T *w, const T *th, const double *Wc, const double *Wf, const double *thf,
                        const MWPhys &ph);
template <typename T>
void launch_wdiv(hipStream_t st, const Metrics<double> &m, double *buf, T *out, const T *u, const T *v, const T *w,
                 const double *Wc, const double *Wf, int normalize);

// ---- terrain-following operators (terrain.hip): op 0 divergence, 1 Laplacian, 2 J·∇² on vectors ----
struct TFView {
    const double *h, *hx, *hy;   // storage planes (sx, sy): terrain and its centred slopes
    const double *sigc, *sigf;   // σ of the cell centres and faces, per storage level
    const double *dzc, *dzf;     // Δσ_c, Δσ_f per storage level
    double Hl, dx, dy;           // the lid, horizontal spacings
    int Nx, Ny, Nz, H, sx, sy;
    int bcx, bcy;                // lateral maps of interior-sized vectors
};
void launch_tf(hipStream_t st, int op, const TFView &t, double *out, const double *a, const double *b,
               const double *c);

// ---- the anelastic core over Gal-Chen terrain (tfstep.hip) ----
struct TFWView {
    const double *h, *hx, *hy;      // storage planes (sx × sy): terrain and its centred slopes
    double Hl, dx, dy, dz;          // lid, spacings (uniform σ)
    double rho0, Hs, theta0, gamma, g_accel;
    int Nx, Ny, Nz, H, sx, sy, buoyancy;
};
// ---------------------------------------------------------------------------
// the Gal-Chen metrics from the storage planes (shared by the terrain
// kernels and the multigrid, which evaluates its finest-level face
// coefficients from them)
// ---------------------------------------------------------------------------
template <typename TC>
struct TFM {
    const double *h, *hx, *hy;  // storage planes (sx × sy)
    TC Hl, iHl, dz, idx, idy, idz, rho0, iHs, theta0, gamma, g;
    int Nx, Ny, Nz, H, sx, sy, buoyancy;
    __device__ __forceinline__ TC hp(int i, int j) const { return (TC)h[i + sx * j]; }
    __device__ __forceinline__ TC sigc(int k) const { return (TC(k - H) + TC(0.5)) * dz; }
    __device__ __forceinline__ TC sigf(int k) const { return TC(k - H) * dz; }
    __device__ __forceinline__ TC J(int i, int j) const { return (Hl - hp(i, j)) * iHl; }
    __device__ __forceinline__ TC hxf(int i, int j) const { return (hp(i, j) + hp(i > 0 ? i - 1 : 0, j)) / TC(2); }
    __device__ __forceinline__ TC hyf(int i, int j) const { return (hp(i, j) + hp(i, j > 0 ? j - 1 : 0)) / TC(2); }
    __device__ __forceinline__ TC Jx(int i, int j) const { return (Hl - hxf(i, j)) * iHl; }
    __device__ __forceinline__ TC Jy(int i, int j) const { return (Hl - hyf(i, j)) * iHl; }
    // J·σ_x and J·σ_y at the σ-face k: −(H − σ_f) h_x/H (the (H − h) of σ_x cancels J's)
    __device__ __forceinline__ TC jsx(int i, int j, int k) const { return (sigf(k) - Hl) * iHl * (TC)hx[i + sx * j]; }
    __device__ __forceinline__ TC jsy(int i, int j, int k) const { return (sigf(k) - Hl) * iHl * (TC)hy[i + sx * j]; }
    __device__ __forceinline__ TC sxz(int i, int j, int k) const {
        return -(Hl - sigf(k)) * (TC)hx[i + sx * j] / (Hl - hp(i, j));
    }
    __device__ __forceinline__ TC syz(int i, int j, int k) const {
        return -(Hl - sigf(k)) * (TC)hy[i + sx * j] / (Hl - hp(i, j));
    }
    __device__ __forceinline__ TC rho(TC z) const {
        if constexpr (sizeof(TC) == 4) return rho0 * __expf(-z * iHs);
        else return rho0 * exp(-z * iHs);
    }
    __device__ __forceinline__ TC rho_c(int i, int j, int k) const { return rho(hp(i, j) + sigc(k) * J(i, j)); }
    __device__ __forceinline__ TC rho_xf(int i, int j, int k) const { return rho(hxf(i, j) + sigc(k) * Jx(i, j)); }
    __device__ __forceinline__ TC rho_yf(int i, int j, int k) const { return rho(hyf(i, j) + sigc(k) * Jy(i, j)); }
    __device__ __forceinline__ TC rho_sf(int i, int j, int k) const { return rho(hp(i, j) + sigf(k) * J(i, j)); }
};

template <typename TC>
inline TFM<TC> make_tfm(const TFWView &v) {
    TFM<TC> m;
    m.h = v.h; m.hx = v.hx; m.hy = v.hy;
    m.Hl = (TC)v.Hl; m.iHl = (TC)(1 / v.Hl); m.dz = (TC)v.dz; m.idx = (TC)(1 / v.dx); m.idy = (TC)(1 / v.dy); m.idz = (TC)(1 / v.dz);
    m.rho0 = (TC)v.rho0; m.iHs = (TC)(1 / v.Hs); m.theta0 = (TC)v.theta0; m.gamma = (TC)v.gamma;
    m.g = (TC)v.g_accel;
    m.Nx = v.Nx; m.Ny = v.Ny; m.Nz = v.Nz; m.H = v.H; m.sx = v.sx; m.sy = v.sy; m.buoyancy = v.buoyancy;
    return m;
}

// tendencies + predictor: us = u + dt·tu …, tn = c(θ0, θ + dt·tθ); scheme SCH_CENTERED or SCH_WENO_Z5;
// f32: the tendency arithmetic in FP32 (the state FP64)
int launch_tfw_tendency(hipStream_t st, const TFWView &v, int scheme, int f32, double *us, double *vs, double *ws,
                        double *tn, const double *u, const double *vv, const double *w, const double *th,
                        const double *th0, double dt, double ca, double cb, int combine, int raw);
void launch_tfw_halos(hipStream_t st, const TFWView &v, double *u, double *vv, double *w, double *th);
void launch_tfw_div(hipStream_t st, const TFWView &v, const double *bx, const double *by, const double *rs,
                    double *out, const double *u, const double *vv, const double *w);
void launch_tfw_grad(hipStream_t st, const TFWView &v, const double *bx, const double *by, const double *rs,
                     double *gx, double *gy, double *gw, const double *x);
// L x in one column-marching pass; with part, the block sums of x·(Lx); returns the block count
int launch_tfw_apply_march(hipStream_t st, const TFWView &v, double *out, const double *x, double *part, int cap);
void launch_tfw_correct(hipStream_t st, const TFWView &v, const double *bx, const double *by, const double *rs,
                        double *u, double *vv, double *w, double *th, double *p, const double *us, const double *vs,
                        const double *ws, const double *tn, const double *u0, const double *v0, const double *w0,
                        const double *phi, double dt, double ca, double cb, int combine);
void launch_tfw_coef(hipStream_t st, const TFWView &v, double *bx, double *by, double *rs);
void launch_tfw_mgcoef(hipStream_t st, const TFWView &v, double *cx, double *cy, double *cz);
// the least-squares guess from earlier solves (tfstep.hip)
constexpr int TFW_KMAX = 16;
struct TFBasis {
    const double *x[TFW_KMAX + 1];
};
// out[i] = X_i·b for i < k (k ≤ TFW_KMAX + 1); part holds (k × 1024) doubles
void launch_tfp_dots(hipStream_t st, const TFBasis &X, int k, const double *b, size_t n, double *part, double *out);
// x0 = Σ_{i<k} c_i X_i (c on the device)
void launch_tfp_combine(hipStream_t st, const TFBasis &X, int k, const double *c, size_t n, double *x0);
// block maxima of |b|/(ρ_c J) (the constraint residual of a mass-flux divergence b)
void launch_tfw_absdiv(hipStream_t st, const TFWView &v, double *part, int nblocks, const double *b);

// ---- cut-cell operators (cutcell.hip): op 0 divergence, 1 gradient/correction, 2 Laplacian ----
template <typename T>
void launch_redistribute(hipStream_t st, T *div, const double *ve, const int *pairs, int npairs, long long nstore);
void launch_fluid_mean(hipStream_t st, const Metrics<double> &m, double *buf, const double *ve);
template <typename T>
int launch_cutcell(hipStream_t st, int op, const Metrics<double> &m, T *a, T *b, T *c, const T *f0, const T *f1,
                   const T *f2, double *buf, const double *phi, int phi_interior, int bcx, int bcy, int bcz,
                   const double *ax, const double *ay, const double *az, const double *ve, int flag, double s);

// ---- spectral / column solvers (fft.hip) ----
struct SpectralPlan;  // opaque: twiddle tables and work arrays on the device
SpectralPlan *spectral_create(int Nx, int Ny, int Nz, hipStream_t st, char *err, size_t errlen);
void spectral_destroy(SpectralPlan *p);
// triply periodic: φ = L⁻¹(src − mean) with the exact 7-point eigenvalues
int spectral_fft_setup(SpectralPlan *p, double dx, double dy, double dz);
int spectral_fft_solve(SpectralPlan *p, hipStream_t st, double *phi, const double *src);
// column solver: periodic x-y transform + FP64 Thomas per wavenumber + mean mode
int spectral_column_setup(SpectralPlan *p, double dx, double dy, const double *lower, const double *upper,
                          const double *hweight, const double *measure, const double *inv_coupling,
                          const double *gauge, int neu_x, int neu_y);
int spectral_column_solve(SpectralPlan *p, hipStream_t st, double *phi, const double *src);
template <typename T>
int spectral_column_solve_div(SpectralPlan *p, hipStream_t st, double *phi, const T *u, const T *v, const T *w,
                              const Metrics<double> &md);
// the same for the W-weighted divergence of a sound-proof core
template <typename T>
int spectral_column_solve_wdiv(SpectralPlan *p, hipStream_t st, double *phi, const T *u, const T *v, const T *w,
                               const double *Wc, const double *Wf, const Metrics<double> &md);

// the levels per block of the marching kernels on a grid of nx × ny × nz cells (chunk_levels; aeo_launch_levels)
int chunk_tile(int nx, int ny, int nz);
int chunk_brick(int nx, int ny, int nz);
int chunk_limited(int nx, int ny, int nz);
int chunk_tfw_tendency(int nx, int ny, int nz);
int chunk_tfw_apply(int nx, int ny, int nz);
int chunk_tf_smooth(int nx, int ny, int nz);
int chunk_tf_prolong(int nx, int ny, int nz);

// A profile scope on the library stream (api.hip): with profiling on and a
// name, events bracket the launches made inside the scope and their time is
// booked under the name (aeo_profile_get)
struct ProfScope {
    void *impl = nullptr;
    explicit ProfScope(const char *name);
    ~ProfScope();
    ProfScope(const ProfScope &) = delete;
    ProfScope &operator=(const ProfScope &) = delete;
};

// ---- multigrid and MG-preconditioned CG (mg.hip) ----
struct MGPlan;
MGPlan *mg_create(int nx, int ny, int nz, double dx, double dy, double dz, int bcx, int bcy, int bcz, const double *cx,
                  const double *cy, const double *cz, const double *rhs_scale, int nu1, int nu2, int smoother,
                  double omega, int prec, int min_size, char *err, size_t errlen);
void mg_destroy(MGPlan *P);
int mg_levels(const MGPlan *P);
int mg_pcg_solve(MGPlan *P, hipStream_t st, double *xout, const double *bin, double tol, int maxit, int *iters_out,
                 double *resid_out, double *bnorm_out);
int mg_cycles_solve(MGPlan *P, hipStream_t st, double *xout, const double *bin, double tol, int maxcycles,
                    int *cycles_out, double *rel_out);
void mg_apply(MGPlan *P, hipStream_t st, double *out, const double *x);
struct FCGOp;
// pcg! with a caller's FP64 operator and the plan's V-cycle as preconditioner;
// x0 (nullable) the initial guess; true_resid (nullable) gets ‖b − Ax‖ recomputed
int mg_pcg_solve_op(MGPlan *P, hipStream_t st, const FCGOp &op, double *xout, const double *bin, const double *x0,
                    double tol, int maxit, int *iters_out, double *resid_out, double *bnorm_out, double *true_resid,
                    double *r0_out);
void mg_set_cycle(MGPlan *P, int wcycle, int fmg);
// the finest level's face coefficients are L's 7-point part on the terrain
// grid v (tfw_mgcoef_kernel's values): the FP64 red-black sweeps evaluate
// them from the metrics instead of reading the stored arrays (the same
// values), the FP32 Jacobi sweeps and residual in FP32
void mg_set_terrain_coef(MGPlan *P, const TFWView &v);
// z = one V-cycle of the preconditioner on r (its mean removed), z mean-free (FP64)
void mg_precond_apply(MGPlan *P, hipStream_t st, double *z, const double *r);

// ---- the learned preconditioner (unet.hip) ----
struct UNet;
UNet *unet_create(int nx, int ny, int nz, int inc, uint64_t seed, char *err, size_t errlen);
void unet_destroy(UNet *N);
size_t unet_num_params(const UNet *N);
int unet_dims_match(const UNet *N, int nx, int ny, int nz);
int unet_get_params(UNet *N, float *host);
int unet_set_params(UNet *N, hipStream_t st, const float *host);
int unet_forward(UNet *N, hipStream_t st, const double *src, const double *mask, double *out);
int unet_gradients(UNet *N, hipStream_t st, const double *src, const double *mask, const double *target,
                   float *grad_host, float *loss);
int unet_train_step(UNet *N, hipStream_t st, const double *src, const double *mask, const double *target, float lr,
                    float *loss);
// dW[tap][c][n] and db[n] of a 3³ convolution from BF16 channels-last in and dy (aeo_conv3_weight_gradient);
// −1: no such layer shape
int conv3_wgrad(hipStream_t st, int cin, int cout, int nx, int ny, int nz, const void *in, const void *dy, float *dw,
                float *db, int *plan);
struct FCGState;
// an operator on interior-sized FP64 vectors: apply(ctx, stream, out, x)
struct FCGOp {
    void (*apply)(void *ctx, hipStream_t st, double *out, const double *x) = nullptr;
    void *ctx = nullptr;
    // optional: out = A x with the block partial sums of x·out into part (at
    // most `cap` of them); returns how many it wrote
    int (*apply_dot)(void *ctx, hipStream_t st, double *out, const double *x, double *part, int cap) = nullptr;
};
FCGState *fcg_create(int n, FCGOp op = FCGOp());
void fcg_destroy(FCGState *F);
int fcg_solve(FCGState *F, MGPlan *P, UNet *N, const double *mask, int mode, int use_guess, hipStream_t st,
              double *xout, const double *bin, double tol, int maxit, int *iters_out, double *resid_out,
              double *bnorm_out);

}  // namespace aeo
