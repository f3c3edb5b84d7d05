// The anelastic core over Gal-Chen terrain (gfx950): the density-weighted
// terrain operators and the mass-weighted step on a terrain-following grid.
//
// The reference has no terrain core (its cores refuse a terrain grid,
// src/Simulations.jl:1160-1163, src/Anelastic.jl:1558-1559); this one
// composes its pieces:
//   - the Gal-Chen map z = h + σJ, J = (H − h)/H, the face metrics and the
//     contravariant flux Ω = w + J(σ_x ū + σ_y v̄), σ_x = −(H − σ_f) h_x/(H − h)
//     (terrain_following_grid, src/StretchedGrids.jl:777-835; _tf_Ω :1180-1205);
//   - the W-weighted flux forms of _mass_weighted_step! (src/Anelastic.jl:
//     1192-1311): each transporting mass flux is ρ̄ at the point where the
//     flux lives (ρ̄(z) = ρ0 e^{−z/Hs} of that point's physical height) times
//     the metric J there times the velocities the reference averages there;
//     the face values are centred or WENO-Z5, upwinded on the mass flux;
//   - B u = δx(ρJ_x u) + δy(ρJ_y v) + δσ(ρΩ) (weighted_divergence!,
//     :1082-1110), Ω = 0 on the ground and the lid;
//   - the projection with G = −M⁻¹Bᵀ (M: the masses ρJ of the velocity
//     volumes): L = B·G is symmetric negative semidefinite, so the outer
//     solve is the CG of pcg! with a multigrid V-cycle on L's 7-point part
//     (face coefficients ρJ_x, ρJ_y, ρJG^σσ) as preconditioner.
// Over flat terrain the tendencies are _mass_weighted_step!'s with
// W_c = ρ̄(z_c), W_f = ρ̄(z_f), and L is DirectWeightedPoissonSolver's ∇·(W∇φ).
//
// Layout: state fields in the storage layout (halo H ≥ 3), FP64; the operator
// works on interior-sized FP64 vectors (x fastest), periodic in x and y.
// Uniform σ spacing dz; σ_c(k) = (k − H + ½)dz, σ_f(k) = (k − H)dz for the
// 0-based storage level k; the ground is σ-face H, the lid σ-face H + Nz.
// The tendency arithmetic runs in TC (double, or float with the state still
// FP64): densities, metric terms, reconstructions and flux differences.
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace aeo {

// ---------------------------------------------------------------------------
// the tendencies + predictor (+ the θ stage combination)
// ---------------------------------------------------------------------------
// the face value between cells c and c+1 from d at element offsets o + m·st,
// o the offset of cell c − 2: centred, or WENO-Z5 (p = 2) upwinded on `vel`
template <int S, typename TC>
__device__ __forceinline__ TC tf_face(const double *__restrict__ d, uint32_t o, uint32_t st, TC vel) {
    if constexpr (S == SCH_CENTERED) {
        return ((TC)d[o + 2 * st] + (TC)d[o + 3 * st]) / TC(2);
    } else {
        const TC a0 = (TC)d[o], a1 = (TC)d[o + st], a2 = (TC)d[o + 2 * st], a3 = (TC)d[o + 3 * st],
                 a4 = (TC)d[o + 4 * st], a5 = (TC)d[o + 5 * st];
        const bool up = vel >= TC(0);
        return weno_z5<2, TC>(up ? a0 : a5, up ? a1 : a4, up ? a2 : a3, up ? a3 : a2, up ? a4 : a1);
    }
}

// the face value minus a base value q0, reconstructed from the stencil's
// differences to q0 (formed in FP64) in TC: centred and WENO-Z5 are
// translation invariant, so this is tf_face − q0 with TC's relative
// precision on the local variation instead of on the value
template <int S, typename TC>
__device__ __forceinline__ TC tf_face_dev(const double *__restrict__ d, uint32_t o, uint32_t st, TC vel, double q0) {
    if constexpr (S == SCH_CENTERED) {
        return ((TC)(d[o + 2 * st] - q0) + (TC)(d[o + 3 * st] - q0)) / TC(2);
    } else {
        const TC a0 = (TC)(d[o] - q0), a1 = (TC)(d[o + st] - q0), a2 = (TC)(d[o + 2 * st] - q0),
                 a3 = (TC)(d[o + 3 * st] - q0), a4 = (TC)(d[o + 4 * st] - q0), a5 = (TC)(d[o + 5 * st] - q0);
        const bool up = vel >= TC(0);
        return weno_z5<2, TC>(up ? a0 : a5, up ? a1 : a4, up ? a2 : a3, up ? a3 : a2, up ? a4 : a1);
    }
}

#ifndef TFW_TEND_CH
#define TFW_TEND_CH 32  // levels per thread of the marching tendency kernel
#endif

// the face value of six values a0..a5 along the line (the face between a2
// and a3): centred, or WENO-Z5 upwinded on `vel`
template <int S, typename TC>
__device__ __forceinline__ TC tf_face6(TC a0, TC a1, TC a2, TC a3, TC a4, TC a5, TC vel) {
    if constexpr (S == SCH_CENTERED) {
        return (a2 + a3) / TC(2);
    } else {
        const bool up = vel >= TC(0);
        return weno_z5<2, TC>(up ? a0 : a5, up ? a1 : a4, up ? a2 : a3, up ? a3 : a2, up ? a4 : a1);
    }
}

// The tendencies + predictor marching up the column: a thread owns the
// column (i, j) and CH levels. Per level it computes what is new there and
// carries the rest from the level below:
//   - the vertical fluxes of u, v, w, θ through the face below a level are
//     the ones through the face above the level before (same mass flux, same
//     stencil), so one vertical reconstruction per field and level;
//   - Ω on the faces of the own column and of the columns i − 1 and j − 1;
//   - each field's six values along σ stay in registers (one load per level);
//   - the reference densities of the fifteen (column, level kind) families
//     the fluxes use follow ρ̄(k+1) = ρ̄(k)·e^{−Δσ J/Hs} (J of the column),
//     from one exp per family at the chunk's start, in FP64.
// The buoyancy about θ̄(z) = θ0 + Γz at the w-face follows _anelastic_buoyancy
// (src/Anelastic.jl:1352-1360), formed in FP64 whatever TC (θ_face − θ̄ is a
// small difference of values near 300 K).
template <int S, typename TC, int CH>
__global__ void __launch_bounds__(256, sizeof(TC) == 4 ? 2 : 1) tfw_tendency_march_kernel(double *__restrict__ us, double *__restrict__ vs,
                                                                  double *__restrict__ ws, double *__restrict__ tn,
                                                                  const double *__restrict__ u,
                                                                  const double *__restrict__ v,
                                                                  const double *__restrict__ w,
                                                                  const double *__restrict__ th,
                                                                  const double *__restrict__ th0, TFM<TC> m,
                                                                  double dt, double ca, double cb, int combine,
                                                                  int raw) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + m.H;
    const int j = blockIdx.y * blockDim.y + threadIdx.y + m.H;
    if (i >= m.H + m.Nx || j >= m.H + m.Ny) return;
    const int H = m.H;
    const int kb = H + (int)blockIdx.z * CH;
    const int ke = kb + CH < H + m.Nz ? kb + CH : H + m.Nz;
    const int sxi = m.sx;
    const int sxyi = m.sx * m.sy;
    const uint32_t sx = (uint32_t)sxi, sxy = (uint32_t)sxyi;
    // FP64 plane values and the density families
    const double *hp = m.h;
    auto hd = [&](int a, int b) -> double { return hp[a + sxi * b]; };
    const double Hl = (double)m.Hl, iHl = 1.0 / Hl, dz = (double)m.dz, iHs = (double)m.iHs, rho0 = (double)m.rho0;
    auto hxfd = [&](int a, int b) -> double { return (hd(a, b) + hd(a - 1, b)) / 2; };
    auto hyfd = [&](int a, int b) -> double { return (hd(a, b) + hd(a, b - 1)) / 2; };
    auto hxyd = [&](int a, int b) -> double { return (hxfd(a, b) + hxfd(a, b - 1)) / 2; };
    struct Fam {
        double r, q;
    };
    // ρ̄ at σ-level index kk (σ = (kk − H + off)·dz) of a column with surface hs
    auto fam = [&](double hs, int kk, double off) -> Fam {
        const double J = (Hl - hs) * iHl;
        return Fam{rho0 * exp(-(hs + ((double)(kk - H) + off) * dz * J) * iHs), exp(-dz * J * iHs)};
    };
    // centre-level families at the chunk's first level kb
    Fam fc00 = fam(hd(i, j), kb, 0.5), fcm0 = fam(hd(i - 1, j), kb, 0.5), fc0m = fam(hd(i, j - 1), kb, 0.5);
    Fam fx00 = fam(hxfd(i, j), kb, 0.5), fx10 = fam(hxfd(i + 1, j), kb, 0.5);
    Fam fy00 = fam(hyfd(i, j), kb, 0.5), fy01 = fam(hyfd(i, j + 1), kb, 0.5);
    Fam fxy00 = fam(hxyd(i, j), kb, 0.5), fxy01 = fam(hxyd(i, j + 1), kb, 0.5), fxy10 = fam(hxyd(i + 1, j), kb, 0.5);
    // face-level families at the face kb (the level's bottom face)
    Fam fs00 = fam(hd(i, j), kb, 0.0), fxs00 = fam(hxfd(i, j), kb, 0.0), fxs10 = fam(hxfd(i + 1, j), kb, 0.0);
    Fam fys00 = fam(hyfd(i, j), kb, 0.0), fys01 = fam(hyfd(i, j + 1), kb, 0.0);
    // ρ̄ at the centre below the chunk (w's lower flux)
    double rc_below = fc00.r / fc00.q;

    auto U = [&](uint32_t c, int di, int dj, int dk) { return (TC)u[c + di + sxi * dj + sxyi * dk]; };
    auto V = [&](uint32_t c, int di, int dj, int dk) { return (TC)v[c + di + sxi * dj + sxyi * dk]; };
    // Ω at the σ-face kk of column (i + di, j + dj)
    auto Om = [&](int di, int dj, int kk) -> TC {
        if (kk == H || kk == H + m.Nz) return TC(0);
        const uint32_t c = lin(i + di, j + dj, kk, m.sx, m.sy);
        const TC ucm = (U(c, 0, 0, -1) + U(c, 1, 0, -1)) / TC(2), uck = (U(c, 0, 0, 0) + U(c, 1, 0, 0)) / TC(2);
        const TC vcm = (V(c, 0, 0, -1) + V(c, 0, 1, -1)) / TC(2), vck = (V(c, 0, 0, 0) + V(c, 0, 1, 0)) / TC(2);
        const TC ub = TC(0.5) * ucm + TC(0.5) * uck, vb = TC(0.5) * vcm + TC(0.5) * vck;
        return (TC)w[c] + (m.jsx(i + di, j + dj, kk) * ub + m.jsy(i + di, j + dj, kk) * vb);
    };
    const TC J00 = m.J(i, j), Jm0 = m.J(i - 1, j), J0m = m.J(i, j - 1);
    const TC Jx00 = m.Jx(i, j), Jx10 = m.Jx(i + 1, j), Jy00 = m.Jy(i, j), Jy01 = m.Jy(i, j + 1);
    const TC Jxy00 = m.Jxy(i, j), Jxy01 = m.Jxy(i, j + 1), Jxy10 = m.Jxy(i + 1, j);
    // the rolling σ-windows: F(k − 2 .. k + 3) of the own column at level k
    const uint32_t c0 = lin(i, j, kb, m.sx, m.sy);
    TC wu[6], wv[6], ww[6];
    double wt[6];
    for (int q = 0; q < 6; q++) {
        const uint32_t cq = c0 + (uint32_t)((q - 2) * sxyi);
        wu[q] = (TC)u[cq];
        wv[q] = (TC)v[cq];
        ww[q] = (TC)w[cq];
        wt[q] = th[cq];
    }
    // Ω carries: own column at faces kb − 1, kb; columns i − 1 and j − 1 at face kb
    TC OmB = Om(0, 0, kb - 1), Om0 = Om(0, 0, kb), Omm0 = Om(-1, 0, kb), Om0m = Om(0, -1, kb);
    // the vertical fluxes through the face kb (the level kb − 1's upper fluxes), from the same stencils
    // (θ's as its mass flux FBm_t and face value FBf_t; in FP32 the face value
    // less θ of the level, re-based when the level moves up)
    TC FBm_t, FBf_t, FB_u, FB_v, FB_w;
    {
        const TC Ft = (TC)fs00.r * Om0;
        const uint32_t oz = c0 - 3 * sxy;
        FBm_t = Ft;
        if constexpr (sizeof(TC) == 8)
            FBf_t = tf_face<S, TC>(th, oz, sxy, Ft);
        else
            FBf_t = tf_face_dev<S, TC>(th, oz, sxy, Ft, wt[2]);
        const TC Wu = (TC)fxs00.r * ((Omm0 + Om0) / TC(2));
        FB_u = Wu * tf_face<S, TC>(u, oz, sxy, Wu);
        const TC Wv = (TC)fys00.r * ((Om0m + Om0) / TC(2));
        FB_v = Wv * tf_face<S, TC>(v, oz, sxy, Wv);
        // w's: through the centre kb − 1 (between faces kb − 1 and kb)
        const TC Ww = (TC)rc_below * ((OmB + Om0) / TC(2));
        FB_w = Ww * tf_face<S, TC>(w, oz, sxy, Ww);
    }
    for (int k = kb; k < ke; k++) {
        const uint32_t c = lin(i, j, k, m.sx, m.sy);
        // Ω on the faces k + 1
        const TC Om1 = Om(0, 0, k + 1), Omm1 = Om(-1, 0, k + 1), Om0m1 = Om(0, -1, k + 1);
        const uint32_t ox = c - 3, oy = c - 3 * sx;
        const TC rc00 = (TC)fc00.r;
        // θ
        TC tt, FTf_t;
        {
            const TC FE = (TC)fx10.r * Jx10 * U(c, 1, 0, 0);
            const TC FW = (TC)fx00.r * Jx00 * U(c, 0, 0, 0);
            const TC FN = (TC)fy01.r * Jy01 * V(c, 0, 1, 0);
            const TC FS = (TC)fy00.r * Jy00 * V(c, 0, 0, 0);
            const TC FT = (TC)(fs00.r * fs00.q) * Om1;
            if constexpr (sizeof(TC) == 8) {
                FTf_t = tf_face6<S, TC>(wt[0], wt[1], wt[2], wt[3], wt[4], wt[5], FT);
                const TC d = ((FE * tf_face<S, TC>(th, ox + 1, 1, FE) - FW * tf_face<S, TC>(th, ox, 1, FW)) * m.idx +
                              (FN * tf_face<S, TC>(th, oy + sx, sx, FN) - FS * tf_face<S, TC>(th, oy, sx, FS)) * m.idy) +
                             (FT * FTf_t - FBm_t * FBf_t) * m.idz;
                tt = TC(0) - d / (rc00 * J00);
            } else {
                // the flux form less θ_c·(B u)/(ρJ): B u vanishes to the projection's tolerance, and its
                // FP32 rounding times θ ≈ 300 K would swamp the tendency of the perturbation
                const double q0 = wt[2];
                FTf_t = tf_face6<S, TC>((TC)(wt[0] - q0), (TC)(wt[1] - q0), TC(0), (TC)(wt[3] - q0),
                                        (TC)(wt[4] - q0), (TC)(wt[5] - q0), FT);
                const TC d = ((FE * tf_face_dev<S, TC>(th, ox + 1, 1, FE, q0) - FW * tf_face_dev<S, TC>(th, ox, 1, FW, q0)) * m.idx +
                              (FN * tf_face_dev<S, TC>(th, oy + sx, sx, FN, q0) - FS * tf_face_dev<S, TC>(th, oy, sx, FS, q0)) * m.idy) +
                             (FT * FTf_t - FBm_t * FBf_t) * m.idz;
                tt = TC(0) - d / (rc00 * J00);
            }
            FBm_t = FT;
        }
        // u at the x-face i
        TC tu, FT_u;
        {
            const TC UE = rc00 * J00 * ((U(c, 0, 0, 0) + U(c, 1, 0, 0)) / TC(2));
            const TC UW = (TC)fcm0.r * Jm0 * ((U(c, -1, 0, 0) + U(c, 0, 0, 0)) / TC(2));
            const TC VN = (TC)fxy01.r * Jxy01 * ((V(c, -1, 1, 0) + V(c, 0, 1, 0)) / TC(2));
            const TC VS = (TC)fxy00.r * Jxy00 * ((V(c, -1, 0, 0) + V(c, 0, 0, 0)) / TC(2));
            const TC WT = (TC)(fxs00.r * fxs00.q) * ((Omm1 + Om1) / TC(2));
            FT_u = WT * tf_face6<S, TC>(wu[0], wu[1], wu[2], wu[3], wu[4], wu[5], WT);
            const TC d = ((UE * tf_face<S, TC>(u, ox + 1, 1, UE) - UW * tf_face<S, TC>(u, ox, 1, UW)) * m.idx +
                          (VN * tf_face<S, TC>(u, oy + sx, sx, VN) - VS * tf_face<S, TC>(u, oy, sx, VS)) * m.idy) +
                         (FT_u - FB_u) * m.idz;
            tu = TC(0) - d / ((TC)fx00.r * Jx00);
        }
        // v at the y-face j
        TC tv, FT_v;
        {
            const TC VN = rc00 * J00 * ((V(c, 0, 0, 0) + V(c, 0, 1, 0)) / TC(2));
            const TC VS = (TC)fc0m.r * J0m * ((V(c, 0, -1, 0) + V(c, 0, 0, 0)) / TC(2));
            const TC UE = (TC)fxy10.r * Jxy10 * ((U(c, 1, -1, 0) + U(c, 1, 0, 0)) / TC(2));
            const TC UW = (TC)fxy00.r * Jxy00 * ((U(c, 0, -1, 0) + U(c, 0, 0, 0)) / TC(2));
            const TC WT = (TC)(fys00.r * fys00.q) * ((Om0m1 + Om1) / TC(2));
            FT_v = WT * tf_face6<S, TC>(wv[0], wv[1], wv[2], wv[3], wv[4], wv[5], WT);
            const TC d = ((UE * tf_face<S, TC>(v, ox + 1, 1, UE) - UW * tf_face<S, TC>(v, ox, 1, UW)) * m.idx +
                          (VN * tf_face<S, TC>(v, oy + sx, sx, VN) - VS * tf_face<S, TC>(v, oy, sx, VS)) * m.idy) +
                         (FT_v - FB_v) * m.idz;
            tv = TC(0) - d / ((TC)fy00.r * Jy00);
        }
        // w at the σ-face k (the ground face is diagnostic); its upper flux
        // through the centre k is carried whatever k
        TC tw = TC(0), FT_w;
        {
            const TC WT = rc00 * ((Om0 + Om1) / TC(2));
            // w(k − 2 .. k + 3): the face between the centre k's faces k and k + 1 is w(k), w(k+1)
            FT_w = WT * tf_face6<S, TC>(ww[0], ww[1], ww[2], ww[3], ww[4], ww[5], WT);
            if (k > H) {
                const TC UE = (TC)fxs10.r * Jx10 * ((U(c, 1, 0, -1) + U(c, 1, 0, 0)) / TC(2));
                const TC UW = (TC)fxs00.r * Jx00 * ((U(c, 0, 0, -1) + U(c, 0, 0, 0)) / TC(2));
                const TC VN = (TC)fys01.r * Jy01 * ((V(c, 0, 1, -1) + V(c, 0, 1, 0)) / TC(2));
                const TC VS = (TC)fys00.r * Jy00 * ((V(c, 0, 0, -1) + V(c, 0, 0, 0)) / TC(2));
                const TC d = ((UE * tf_face<S, TC>(w, ox + 1, 1, UE) - UW * tf_face<S, TC>(w, ox, 1, UW)) * m.idx +
                              (VN * tf_face<S, TC>(w, oy + sx, sx, VN) - VS * tf_face<S, TC>(w, oy, sx, VS)) * m.idy) +
                             (FT_w - FB_w) * m.idz;
                tw = TC(0) - d / ((TC)fs00.r * J00);
                if (m.buoyancy) {
                    const TC zf = m.hp(i, j) + m.sigf(k) * J00;
                    const double tb = (double)m.theta0 + (double)m.gamma * (double)zf;
                    const double coef = (double)m.g / tb;
                    const double tface = 0.5 * (wt[1] + wt[2]);
                    tw += (TC)(coef * (tface - tb));
                }
            }
        }
        if (raw) {
            us[c] = (double)tu;
            vs[c] = (double)tv;
            ws[c] = (double)tw;
            tn[c] = (double)tt;
        } else {
            us[c] = u[c] + dt * (double)tu;
            vs[c] = v[c] + dt * (double)tv;
            ws[c] = k > H ? w[c] + dt * (double)tw : w[c];
            const double tnew = wt[2] + dt * (double)tt;
            tn[c] = combine ? ca * th0[c] + cb * tnew : tnew;
        }
        // up one level: the carries and the windows
        FBf_t = FTf_t; FB_u = FT_u; FB_v = FT_v; FB_w = FT_w;
        OmB = Om0; Om0 = Om1; Omm0 = Omm1; Om0m = Om0m1;
        if (k + 1 < ke) {
            const uint32_t cn = c + 4 * sxy;  // level k + 4 = the new window top (k + 1) + 3
            for (int q = 0; q < 5; q++) {
                wu[q] = wu[q + 1]; wv[q] = wv[q + 1]; ww[q] = ww[q + 1]; wt[q] = wt[q + 1];
            }
            wu[5] = (TC)u[cn]; wv[5] = (TC)v[cn]; ww[5] = (TC)w[cn]; wt[5] = th[cn];
            if constexpr (sizeof(TC) == 4) FBf_t -= (TC)(wt[2] - wt[1]);  // re-based on θ of level k + 1
            fc00.r *= fc00.q; fcm0.r *= fcm0.q; fc0m.r *= fc0m.q;
            fx00.r *= fx00.q; fx10.r *= fx10.q; fy00.r *= fy00.q; fy01.r *= fy01.q;
            fxy00.r *= fxy00.q; fxy01.r *= fxy01.q; fxy10.r *= fxy10.q;
            fs00.r *= fs00.q; fxs00.r *= fxs00.q; fxs10.r *= fxs10.q; fys00.r *= fys00.q; fys01.r *= fys01.q;
        }
    }
}

// ---------------------------------------------------------------------------
// halos: u, v, θ periodic in x, y and mirrored in σ (the generic halo
// kernel); w: its ground and lid faces diagnosed from Ω = 0, its σ-halos
// antisymmetric about them, then periodic in x, y
// ---------------------------------------------------------------------------
__global__ void tfw_wall_w_kernel(double *__restrict__ w, const double *__restrict__ u, const double *__restrict__ v,
                                  TFM<double> m) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + m.H;
    const int j = blockIdx.y + m.H;
    if (i >= m.H + m.Nx) return;
    const uint32_t sx = m.sx, sxy = (uint32_t)m.sx * (uint32_t)m.sy;
    const int kw[2] = {m.H, m.H + m.Nz};
    for (int s = 0; s < 2; s++) {
        const int k = kw[s];
        const uint32_t c = lin(i, j, k, m.sx, m.sy);
        const double ucm = (u[c - sxy] + u[c - sxy + 1]) / 2, uck = (u[c] + u[c + 1]) / 2;
        const double vcm = (v[c - sxy] + v[c - sxy + sx]) / 2, vck = (v[c] + v[c + sx]) / 2;
        const double ub = 0.5 * ucm + 0.5 * uck, vb = 0.5 * vcm + 0.5 * vck;
        w[c] = 0.0 - m.J(i, j) * (m.sxz(i, j, k) * ub + m.syz(i, j, k) * vb);
    }
    const uint32_t cg = lin(i, j, m.H, m.sx, m.sy), ct = lin(i, j, m.H + m.Nz, m.sx, m.sy);
    const double wg = w[cg], wt = w[ct];
    for (int q = 1; q <= m.H; q++) {
        w[cg - q * sxy] = 2 * wg - w[cg + q * sxy];
        if (m.H + m.Nz + q < m.Nz + 2 * m.H) w[ct + q * sxy] = 2 * wt - w[ct - q * sxy];
    }
}
// periodic x, y halos of a field over every storage level
__global__ void tfw_xy_halo_kernel(double *__restrict__ f, TFM<double> m) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, k = blockIdx.z;
    if (i >= m.sx) return;
    const bool hi = i < m.H || i >= m.H + m.Nx, hj = j < m.H || j >= m.H + m.Ny;
    if (!hi && !hj) return;
    const int ii = i < m.H ? i + m.Nx : (i >= m.H + m.Nx ? i - m.Nx : i);
    const int jj = j < m.H ? j + m.Ny : (j >= m.H + m.Ny ? j - m.Ny : j);
    f[lin(i, j, k, m.sx, m.sy)] = f[lin(ii, jj, k, m.sx, m.sy)];
}

// ---------------------------------------------------------------------------
// the operator on interior-sized vectors
// ---------------------------------------------------------------------------
// S_x or S_y at the σ-face f of column (a, b): ρ_σ J σ_x δσφ (0 on the walls)
__device__ __forceinline__ int wrapi(int a, int n) { return a < 0 ? a + n : (a >= n ? a - n : a); }

struct TFOp {
    const double *bx, *by, *rs;  // ρ J_x (x-faces), ρ J_y (y-faces): nx·ny·nz; ρ at σ-faces: nx·ny·(nz+1)
    TFM<double> m;
    int nx, ny, nz;
    __device__ __forceinline__ uint32_t o(int a, int b, int c) const {
        return (uint32_t)a + (uint32_t)nx * ((uint32_t)b + (uint32_t)ny * (uint32_t)c);
    }
    __device__ __forceinline__ double phi(const double *p, int a, int b, int c) const {
        return p[o(wrapi(a, nx), wrapi(b, ny), c)];
    }
    // the metric term of column (a, b) at σ-face f (storage column a + H)
    __device__ __forceinline__ double S(const double *p, int which, int a, int b, int f) const {
        if (f == 0 || f == nz) return 0.0;
        const int i = a + m.H, j = b + m.H, k = f + m.H;
        const double ds = (phi(p, a, b, f) - phi(p, a, b, f - 1)) * m.idz;
        const double s = which == 0 ? m.sxz(i, j, k) : m.syz(i, j, k);
        const int aw = wrapi(a, nx), bw = wrapi(b, ny);
        return rs[(uint32_t)aw + (uint32_t)nx * ((uint32_t)bw + (uint32_t)ny * (uint32_t)f)] * m.J(i, j) * s * ds;
    }
    // G_x φ at the x-face a of level c (between cells a−1 and a)
    __device__ __forceinline__ double Gx(const double *p, int a, int b, int c) const {
        const double ax = 0.25 * ((S(p, 0, a - 1, b, c) + S(p, 0, a, b, c)) + (S(p, 0, a - 1, b, c + 1) + S(p, 0, a, b, c + 1)));
        return (phi(p, a, b, c) - phi(p, a - 1, b, c)) * m.idx + ax / bx[o(wrapi(a, nx), wrapi(b, ny), c)];
    }
    __device__ __forceinline__ double Gy(const double *p, int a, int b, int c) const {
        const double ay = 0.25 * ((S(p, 1, a, b - 1, c) + S(p, 1, a, b, c)) + (S(p, 1, a, b - 1, c + 1) + S(p, 1, a, b, c + 1)));
        return (phi(p, a, b, c) - phi(p, a, b - 1, c)) * m.idy + ay / by[o(wrapi(a, nx), wrapi(b, ny), c)];
    }
    // G_w φ at the σ-face f (interior faces only)
    __device__ __forceinline__ double Gw(const double *p, int a, int b, int f) const {
        return ((phi(p, a, b, f) - phi(p, a, b, f - 1)) * m.idz) / m.J(a + m.H, b + m.H);
    }
};

// G φ into face arrays (gx, gy: x-/y-face of the cell; gw: σ-face c, 0 on the ground)
__global__ void tfw_grad_kernel(double *__restrict__ gx, double *__restrict__ gy, double *__restrict__ gw,
                                const double *__restrict__ p, TFOp op) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y, c = blockIdx.z;
    if (a >= op.nx) return;
    const uint32_t q = op.o(a, b, c);
    gx[q] = op.Gx(p, a, b, c);
    gy[q] = op.Gy(p, a, b, c);
    gw[q] = c == 0 ? 0.0 : op.Gw(p, a, b, c);
}
// L φ = B(Gφ) in one pass. With D_f = ρ_σ δσφ on the σ-faces (zero on the
// walls), τ_f = H − σ_f, E_c = τ_c D_c + τ_{c+1} D_{c+1} and k = −h_x/H,
// the x mass flux of Gφ on the face between columns 1 and 0 is
//   q = ρJ_x δxφ + ¼ (k_1 E_1 + k_0 E_0),  G = q/ρJ_x,
// likewise in y, and with W_c = k_x (G_A + G_B) + k_y (G_C + G_D) of the
// cell's four faces the σ-face's flux is
//   ρΩ_f = D_f/J + ρ_σ τ_f ¼ (W_{f−1} + W_f).
// A thread owns a column and marches a chunk of levels with D and φ of its
// own and its four neighbours' columns, one level ahead of the output. ρ_σ
// (5 columns) and ρJ and its inverse (4 faces) are not read: each is
// evaluated by exp at the chunk's first level and carried by its ratio
// between levels, so that φ in and Lφ out are all the memory traffic and
// nothing is divided. The carried values are within about 64 ulp of the
// stored arrays' that B and G read. With part != nullptr, the block sums of
// φ·(Lφ) go to part[block] (the CG's curvature).
// Measured at 512×512×256: 942 us reading the three coefficient arrays
// (3.55 GB) with four divisions per cell → 448 us; 96×96×48 52 → 14 us
// (64 levels per block on every grid before).
constexpr int TFA_BY = 4;      // rows per block
constexpr int TFA_KC = 64;     // most levels per chunk
constexpr int TFA_FILL = 768;  // blocks a round: 3 waves per SIMD
__global__ void __launch_bounds__(64 * TFA_BY) tfw_apply_march_kernel(double *__restrict__ out,
                                                                      const double *__restrict__ p, TFOp op, int kc,
                                                                      double *__restrict__ part) {
    const int nx = op.nx, ny = op.ny, nz = op.nz;
    const TFM<double> &m = op.m;
    const int a = blockIdx.x * 64 + threadIdx.x, b = blockIdx.y * TFA_BY + threadIdx.y;
    double dot = 0.0;
    if (a < nx && b < ny) {
        const int c0 = blockIdx.z * kc, c1 = min(c0 + kc, nz);
        const uint32_t nxy = (uint32_t)nx * (uint32_t)ny;
        const int am = a > 0 ? a - 1 : nx - 1, ap = a + 1 < nx ? a + 1 : 0;
        const int bm = b > 0 ? b - 1 : ny - 1, bp = b + 1 < ny ? b + 1 : 0;
        // the columns: 0 (a, b), 1 (a−1, b), 2 (a+1, b), 3 (a, b−1), 4 (a, b+1)
        const uint32_t col[5] = {(uint32_t)a + nx * (uint32_t)b, (uint32_t)am + nx * (uint32_t)b,
                                 (uint32_t)ap + nx * (uint32_t)b, (uint32_t)a + nx * (uint32_t)bm,
                                 (uint32_t)a + nx * (uint32_t)bp};
        const int i = a + m.H, j = b + m.H;
        const double k4 = -0.25 / m.Hl;  // ¼ k of the columns
        const double kx0 = m.hx[i + m.sx * j] * k4, kx1 = m.hx[(i - 1) + m.sx * j] * k4, kx2 = m.hx[(i + 1) + m.sx * j] * k4;
        const double ky0 = m.hy[i + m.sx * j] * k4, ky3 = m.hy[i + m.sx * (j - 1)] * k4, ky4 = m.hy[i + m.sx * (j + 1)] * k4;
        const double idx = m.idx, idy = m.idy, idz = m.idz, dz = m.dz;
        const double iJ = 1.0 / m.J(i, j);
        const int ns = c0 > 0 ? c0 - 1 : 0;  // the first level worked: W below the chunk
        double tau = m.Hl - ns * dz;         // τ at the σ-face n
        // ρ_σ/Δσ at the σ-face n (stepped up as n is), its ratio per level; ρJ on the
        // faces A, B (west, east), C, D (south, north) at level n, the inverse, the ratios
        double r[5], qr[5], bf[4], ib[4], qb[4], qi[4];
        {
            const int I[5] = {i, i - 1, i + 1, i, i}, Jr[5] = {j, j, j, j - 1, j + 1};
#pragma unroll
            for (int q = 0; q < 5; q++) {
                const double Jc = m.J(I[q], Jr[q]);
                r[q] = m.rho(m.hp(I[q], Jr[q]) + ns * dz * Jc) * idz;
                qr[q] = exp(-(dz * Jc) * m.iHs);
            }
            const double sc = (ns + 0.5) * dz;
            const double hf[4] = {m.hxf(i, j), m.hxf(i + 1, j), m.hyf(i, j), m.hyf(i, j + 1)};
            const double Jf[4] = {m.Jx(i, j), m.Jx(i + 1, j), m.Jy(i, j), m.Jy(i, j + 1)};
#pragma unroll
            for (int q = 0; q < 4; q++) {
                bf[q] = m.rho(hf[q] + sc * Jf[q]) * Jf[q];
                ib[q] = 1.0 / bf[q];
                qb[q] = exp(-(dz * Jf[q]) * m.iHs);
                qi[q] = 1.0 / qb[q];
            }
        }
        double Pc[5], Pn[5], Dc[5];
#pragma unroll
        for (int q = 0; q < 5; q++) {
            Pc[q] = p[col[q] + nxy * (uint32_t)ns];
            Pn[q] = ns + 1 < nz ? p[col[q] + nxy * (uint32_t)(ns + 1)] : 0.0;
            Dc[q] = ns > 0 ? r[q] * (Pc[q] - p[col[q] + nxy * (uint32_t)(ns - 1)]) : 0.0;
        }
        double rp = r[0];                                       // ρ_σ/Δσ of the own column at the face n
        double Hp = 0.0, Wp = 0.0, omp = 0.0, Pp = 0.0;         // of the level below: the x-y part, W, ρΩ, φ
        const int ne = c1 < nz ? c1 : nz - 1;
        for (int n = ns; n <= ne; n++) {
            double Pf[5];  // φ two levels up, in flight over this level's arithmetic
#pragma unroll
            for (int q = 0; q < 5; q++) Pf[q] = n + 2 < nz && n < ne ? p[col[q] + nxy * (uint32_t)(n + 2)] : 0.0;
            const double tn = tau - dz;
            double E[5], Dn[5];
#pragma unroll
            for (int q = 0; q < 5; q++) {
                r[q] *= qr[q];
                Dn[q] = n + 1 < nz ? r[q] * (Pn[q] - Pc[q]) : 0.0;
                E[q] = __builtin_fma(tn, Dn[q], tau * Dc[q]);
            }
            const double dA = (Pc[0] - Pc[1]) * idx, dB = (Pc[2] - Pc[0]) * idx;
            const double dC = (Pc[0] - Pc[3]) * idy, dD = (Pc[4] - Pc[0]) * idy;
            const double ex = kx0 * E[0], ey = ky0 * E[0];
            const double sA = __builtin_fma(kx1, E[1], ex), sB = __builtin_fma(kx2, E[2], ex);
            const double sC = __builtin_fma(ky3, E[3], ey), sD = __builtin_fma(ky4, E[4], ey);
            const double H = (__builtin_fma(bf[1], dB, sB) - __builtin_fma(bf[0], dA, sA)) * idx +
                             (__builtin_fma(bf[3], dD, sD) - __builtin_fma(bf[2], dC, sC)) * idy;
            const double gx = __builtin_fma(sA, ib[0], dA) + __builtin_fma(sB, ib[1], dB);
            const double gy = __builtin_fma(sC, ib[2], dC) + __builtin_fma(sD, ib[3], dD);
            const double W = __builtin_fma(kx0, gx, ky0 * gy);
            const double om = n > 0 ? __builtin_fma(Dc[0], iJ, (rp * dz) * tau * (Wp + W)) : 0.0;
            if (n > c0) {
                const double v = __builtin_fma(om - omp, idz, Hp);
                out[col[0] + nxy * (uint32_t)(n - 1)] = v;
                dot = __builtin_fma(Pp, v, dot);
            }
            Hp = H; Wp = W; omp = om; Pp = Pc[0];
            rp = r[0];
            tau = tn;
#pragma unroll
            for (int q = 0; q < 5; q++) { Pc[q] = Pn[q]; Pn[q] = Pf[q]; Dc[q] = Dn[q]; }
#pragma unroll
            for (int q = 0; q < 4; q++) { bf[q] *= qb[q]; ib[q] *= qi[q]; }
        }
        if (c1 == nz) {  // the top level: no flux through the lid
            const double v = __builtin_fma(-omp, idz, Hp);
            out[col[0] + nxy * (uint32_t)(nz - 1)] = v;
            dot = __builtin_fma(Pp, v, dot);
        }
    }
    if (part) {
        __shared__ double sh[TFA_BY];
        for (int off = 32; off > 0; off >>= 1) dot += __shfl_down(dot, off, 64);
        if (threadIdx.x == 0) sh[threadIdx.y] = dot;
        __syncthreads();
        if (threadIdx.x == 0 && threadIdx.y == 0) {
            double t = 0.0;
            for (int w = 0; w < TFA_BY; w++) t += sh[w];
            part[blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)] = t;
        }
    }
}

// B u of storage-layout velocities into an interior-sized FP64 vector
__global__ void tfw_div_kernel(double *__restrict__ out, const double *__restrict__ u, const double *__restrict__ v,
                               const double *__restrict__ w, TFOp op) {
    int bxi, b, c;
    xcd_block3(bxi, b, c);
    const int a = bxi * blockDim.x + threadIdx.x;
    if (a >= op.nx) return;
    const TFM<double> &m = op.m;
    const int nx = op.nx, ny = op.ny, nz = op.nz;
    const int i = a + m.H, j = b + m.H, k = c + m.H;
    const uint32_t sx = m.sx, sxy = (uint32_t)m.sx * (uint32_t)m.sy;
    const uint32_t s = lin(i, j, k, m.sx, m.sy);
    const int ap = wrapi(a + 1, nx), bp = wrapi(b + 1, ny);
    const double FE = op.bx[op.o(ap, b, c)] * u[s + 1], FW = op.bx[op.o(a, b, c)] * u[s];
    const double FN = op.by[op.o(a, bp, c)] * v[s + sx], FS = op.by[op.o(a, b, c)] * v[s];
    double Omv[2];
    for (int q = 0; q < 2; q++) {
        const int f = c + q;
        if (f == 0 || f == nz) { Omv[q] = 0.0; continue; }
        const uint32_t t = s + q * sxy;
        const double ucm = (u[t - sxy] + u[t - sxy + 1]) / 2, uck = (u[t] + u[t + 1]) / 2;
        const double vcm = (v[t - sxy] + v[t - sxy + sx]) / 2, vck = (v[t] + v[t + sx]) / 2;
        const double ub = 0.5 * ucm + 0.5 * uck, vb = 0.5 * vcm + 0.5 * vck;
        Omv[q] = op.rs[(uint32_t)a + (uint32_t)nx * ((uint32_t)b + (uint32_t)ny * (uint32_t)f)] *
                 (w[t] + m.J(i, j) * (m.sxz(i, j, k + q) * ub + m.syz(i, j, k + q) * vb));
    }
    out[op.o(a, b, c)] = ((FE - FW) * m.idx + (FN - FS) * m.idy) + (Omv[1] - Omv[0]) * m.idz;
}

// u = c(u0, u* − Gxφ), v, w (interior σ-faces); θ = θ'; p = φ/Δt (p nullable)
__global__ void tfw_correct_kernel(double *__restrict__ u, double *__restrict__ v, double *__restrict__ w,
                                   double *__restrict__ th, double *__restrict__ p, const double *__restrict__ us,
                                   const double *__restrict__ vs, const double *__restrict__ ws,
                                   const double *__restrict__ tn, const double *__restrict__ u0,
                                   const double *__restrict__ v0, const double *__restrict__ w0,
                                   const double *__restrict__ phi, TFOp op, double dt, double ca, double cb,
                                   int combine) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y, c = blockIdx.z;
    if (a >= op.nx) return;
    const TFM<double> &m = op.m;
    const uint32_t s = lin(a + m.H, b + m.H, c + m.H, m.sx, m.sy);
    const double un = us[s] - op.Gx(phi, a, b, c);
    const double vn = vs[s] - op.Gy(phi, a, b, c);
    u[s] = combine ? ca * u0[s] + cb * un : un;
    v[s] = combine ? ca * v0[s] + cb * vn : vn;
    if (c > 0) {
        const double wn = ws[s] - op.Gw(phi, a, b, c);
        w[s] = combine ? ca * w0[s] + cb * wn : wn;
    }
    if (th) th[s] = tn[s];
    if (p) p[s] = phi[op.o(a, b, c)] / dt;
}

// block maxima of |b|/(ρ_c J) over an interior-sized vector (NaN propagates)
__global__ void __launch_bounds__(256) tfw_absdiv_kernel(double *__restrict__ part, const double *__restrict__ b,
                                                         TFOp op) {
    __shared__ double sh[256];
    const uint32_t n = (uint32_t)op.nx * op.ny * op.nz;
    double acc = 0.0;
    for (uint32_t e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x) {
        const int a = (int)(e % (uint32_t)op.nx);
        const uint32_t r = e / (uint32_t)op.nx;
        const int bb = (int)(r % (uint32_t)op.ny), c = (int)(r / (uint32_t)op.ny);
        const int i = a + op.m.H, j = bb + op.m.H, k = c + op.m.H;
        const double val = fabs(b[e]) / (op.m.rho_c(i, j, k) * op.m.J(i, j));
        acc = (val > acc || val != val) ? val : acc;
    }
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            const double x = sh[threadIdx.x], y = sh[threadIdx.x + s];
            sh[threadIdx.x] = (y > x || y != y) ? y : x;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// the correction by columns: thread (a, b) marches CH levels with rolling
// windows of φ on its own, west and south columns and of their metric terms
// S; the same G as tfw_correct_kernel without its recomputation
template <int CH>
__global__ void __launch_bounds__(256) tfw_correct_march_kernel(
    double *__restrict__ u, double *__restrict__ v, double *__restrict__ w, double *__restrict__ th,
    double *__restrict__ p, const double *__restrict__ us, const double *__restrict__ vs, const double *__restrict__ ws,
    const double *__restrict__ tn, const double *__restrict__ u0, const double *__restrict__ v0,
    const double *__restrict__ w0, const double *__restrict__ phi, TFOp op, double dt, double ca, double cb,
    int combine) {
    const int nx = op.nx, ny = op.ny, nz = op.nz;
    const TFM<double> &m = op.m;
    const int a = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y * blockDim.y + threadIdx.y;
    if (a >= nx || b >= ny) return;
    const int c0 = blockIdx.z * CH;
    const int c1 = c0 + CH < nz ? c0 + CH : nz;
    const uint32_t nxy = (uint32_t)nx * (uint32_t)ny;
    const int am = a > 0 ? a - 1 : nx - 1, bm = b > 0 ? b - 1 : ny - 1;
    // the columns: 0 (a, b), 1 (a−1, b), 2 (a, b−1)
    const uint32_t col[3] = {(uint32_t)a + nx * (uint32_t)b, (uint32_t)am + nx * (uint32_t)b,
                             (uint32_t)a + nx * (uint32_t)bm};
    const int i = a + m.H, j = b + m.H;
    const double iHl = 1.0 / m.Hl;
    const double kx0 = -m.hx[i + m.sx * j] * iHl, kx1 = -m.hx[(i - 1) + m.sx * j] * iHl;
    const double ky0 = -m.hy[i + m.sx * j] * iHl, ky2 = -m.hy[i + m.sx * (j - 1)] * iHl;
    const double iJ = m.Hl / (m.Hl - m.h[i + m.sx * j]);
    const double idx = m.idx, idy = m.idy, idz = m.idz, dz = m.dz, Hl = m.Hl;
    auto P = [&](int q, int c) -> double { return (c >= 0 && c < nz) ? phi[col[q] + nxy * (uint32_t)c] : 0.0; };
    auto Sv = [&](int q, double k, int f, double pm, double pc) -> double {
        if (f <= 0 || f >= nz) return 0.0;
        return op.rs[col[q] + nxy * (uint32_t)f] * k * (Hl - f * dz) * ((pc - pm) * idz);
    };
    double Pm[3], Pc[3], Pn[3];
    for (int q = 0; q < 3; q++) {
        Pm[q] = P(q, c0 - 1);
        Pc[q] = P(q, c0);
        Pn[q] = P(q, c0 + 1);
    }
    double sx00 = Sv(0, kx0, c0, Pm[0], Pc[0]), sx10 = Sv(1, kx1, c0, Pm[1], Pc[1]);
    double sy00 = Sv(0, ky0, c0, Pm[0], Pc[0]), sy20 = Sv(2, ky2, c0, Pm[2], Pc[2]);
    for (int c = c0; c < c1; c++) {
        const double sx01 = Sv(0, kx0, c + 1, Pc[0], Pn[0]), sx11 = Sv(1, kx1, c + 1, Pc[1], Pn[1]);
        const double sy01 = Sv(0, ky0, c + 1, Pc[0], Pn[0]), sy21 = Sv(2, ky2, c + 1, Pc[2], Pn[2]);
        const uint32_t q = col[0] + nxy * (uint32_t)c;
        const double gx = (Pc[0] - Pc[1]) * idx + 0.25 * ((sx10 + sx00) + (sx11 + sx01)) / op.bx[q];
        const double gy = (Pc[0] - Pc[2]) * idy + 0.25 * ((sy20 + sy00) + (sy21 + sy01)) / op.by[q];
        const uint32_t s = lin(i, j, c + m.H, m.sx, m.sy);
        const double un = us[s] - gx, vn = vs[s] - gy;
        u[s] = combine ? ca * u0[s] + cb * un : un;
        v[s] = combine ? ca * v0[s] + cb * vn : vn;
        if (c > 0) {
            const double wn = ws[s] - ((Pc[0] - Pm[0]) * idz) * iJ;
            w[s] = combine ? ca * w0[s] + cb * wn : wn;
        }
        if (th) th[s] = tn[s];
        if (p) p[s] = Pc[0] / dt;
        for (int t = 0; t < 3; t++) {
            Pm[t] = Pc[t];
            Pc[t] = Pn[t];
            Pn[t] = P(t, c + 2);
        }
        sx00 = sx01; sx10 = sx11; sy00 = sy01; sy20 = sy21;
    }
}

// the operator's face arrays: ρJ_x at x-faces, ρJ_y at y-faces, ρ at σ-faces
__global__ void tfw_coef_kernel(double *__restrict__ bx, double *__restrict__ by, double *__restrict__ rs, TFOp op) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y, c = blockIdx.z;  // c: 0 .. nz
    if (a >= op.nx) return;
    const TFM<double> &m = op.m;
    const int i = a + m.H, j = b + m.H, k = c + m.H;
    if (c < op.nz) {
        bx[op.o(a, b, c)] = m.rho_xf(i, j, k) * m.Jx(i, j);
        by[op.o(a, b, c)] = m.rho_yf(i, j, k) * m.Jy(i, j);
    }
    rs[(uint32_t)a + (uint32_t)op.nx * ((uint32_t)b + (uint32_t)op.ny * (uint32_t)c)] = m.rho_sf(i, j, k);
}

// the 7-point part of L for the multigrid (its face-coefficient layout):
// cx (nx+1, ny, nz) = ρJ_x, cy (nx, ny+1, nz) = ρJ_y, cz (nx, ny, nz+1) = ρ J G^σσ
__global__ void tfw_mgcoef_kernel(double *__restrict__ cx, double *__restrict__ cy, double *__restrict__ cz, TFOp op) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y, c = blockIdx.z;  // a: 0 .. nx, b: 0 .. ny
    const int nx = op.nx, ny = op.ny, nz = op.nz;
    if (a > nx) return;
    const TFM<double> &m = op.m;
    const int i = a + m.H, j = b + m.H, k = c + m.H;
    if (b < ny && c < nz) cx[(uint32_t)a + (uint32_t)(nx + 1) * ((uint32_t)b + (uint32_t)ny * c)] = m.rho_xf(i, j, k) * m.Jx(i, j);
    if (a < nx && c < nz) cy[(uint32_t)a + (uint32_t)nx * ((uint32_t)b + (uint32_t)(ny + 1) * c)] = m.rho_yf(i, j, k) * m.Jy(i, j);
    if (a < nx && b < ny) {
        const double sx_ = m.sxz(i, j, k), sy_ = m.syz(i, j, k), J = m.J(i, j);
        cz[(uint32_t)a + (uint32_t)nx * ((uint32_t)b + (uint32_t)ny * c)] =
            m.rho_sf(i, j, k) * J * ((sx_ * sx_ + sy_ * sy_) + 1 / (J * J));
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static TFOp make_op(const TFWView &v, const double *bx, const double *by, const double *rs) {
    TFOp op;
    op.bx = bx; op.by = by; op.rs = rs;
    op.m = make_tfm<double>(v);
    op.nx = v.Nx; op.ny = v.Ny; op.nz = v.Nz;
    return op;
}

int launch_tfw_tendency(hipStream_t st, const TFWView &v, int scheme, int f32, double *us, double *vs, double *ws,
                        double *tn, const double *u, const double *vv, const double *w, const double *th,
                        const double *th0, double dt, double ca, double cb, int combine, int raw) {
    constexpr int CH = TFW_TEND_CH;
    dim3 blk(64, 4), grid((v.Nx + 63) / 64, (v.Ny + 3) / 4, (v.Nz + CH - 1) / CH);
    if (scheme == SCH_CENTERED) {
        if (f32) hipLaunchKernelGGL((tfw_tendency_march_kernel<SCH_CENTERED, float, CH>), grid, blk, 0, st, us, vs, ws, tn, u, vv, w, th, th0, make_tfm<float>(v), dt, ca, cb, combine, raw);
        else hipLaunchKernelGGL((tfw_tendency_march_kernel<SCH_CENTERED, double, CH>), grid, blk, 0, st, us, vs, ws, tn, u, vv, w, th, th0, make_tfm<double>(v), dt, ca, cb, combine, raw);
    } else if (scheme == SCH_WENO_Z5) {
        if (f32) hipLaunchKernelGGL((tfw_tendency_march_kernel<SCH_WENO_Z5, float, CH>), grid, blk, 0, st, us, vs, ws, tn, u, vv, w, th, th0, make_tfm<float>(v), dt, ca, cb, combine, raw);
        else hipLaunchKernelGGL((tfw_tendency_march_kernel<SCH_WENO_Z5, double, CH>), grid, blk, 0, st, us, vs, ws, tn, u, vv, w, th, th0, make_tfm<double>(v), dt, ca, cb, combine, raw);
    } else {
        return -1;
    }
    return 0;
}

void launch_tfw_halos(hipStream_t st, const TFWView &v, double *u, double *vv, double *w, double *th) {
    HaloSet<double> hs{};
    hs.add(u, LOC_FX, BC_PERIODIC, BC_PERIODIC, BC_NOFLUX);
    hs.add(vv, LOC_FY, BC_PERIODIC, BC_PERIODIC, BC_NOFLUX);
    if (th) hs.add(th, LOC_CC, BC_PERIODIC, BC_PERIODIC, BC_NOFLUX);
    launch_halo_multi<double>(st, hs, v.Nx, v.Ny, v.Nz, v.H);
    const TFM<double> m = make_tfm<double>(v);
    hipLaunchKernelGGL(tfw_wall_w_kernel, dim3((v.Nx + 127) / 128, v.Ny), dim3(128), 0, st, w, u, vv, m);
    hipLaunchKernelGGL(tfw_xy_halo_kernel, dim3((v.sx + 127) / 128, v.sy, v.Nz + 2 * v.H), dim3(128), 0, st, w, m);
}

void launch_tfw_div(hipStream_t st, const TFWView &v, const double *bx, const double *by, const double *rs,
                    double *out, const double *u, const double *vv, const double *w) {
    dim3 grid((v.Nx + 127) / 128, v.Ny, v.Nz);
    hipLaunchKernelGGL(tfw_div_kernel, grid, dim3(128), 0, st, out, u, vv, w, make_op(v, bx, by, rs));
}

// L x with the block sums of x·Lx into part when part holds ≥ that many
// blocks (cap); returns the block count, or −1 when no sums were written
int launch_tfw_apply_march(hipStream_t st, const TFWView &v, double *out, const double *x, double *part, int cap) {
    const int tx = (v.Nx + 63) / 64, ty = (v.Ny + TFA_BY - 1) / TFA_BY;
    const int kc = chunk_levels(tx * ty, v.Nz, TFA_KC, TFA_FILL, 4);
    const dim3 grid(tx, ty, (v.Nz + kc - 1) / kc);
    const int nb = (int)(grid.x * grid.y * grid.z);
    if (part && nb > cap) part = nullptr;
    hipLaunchKernelGGL(tfw_apply_march_kernel, grid, dim3(64, TFA_BY), 0, st, out, x,
                       make_op(v, nullptr, nullptr, nullptr), kc, part);
    return part ? nb : -1;
}

void launch_tfw_grad(hipStream_t st, const TFWView &v, const double *bx, const double *by, const double *rs,
                     double *gx, double *gy, double *gw, const double *x) {
    dim3 grid((v.Nx + 127) / 128, v.Ny, v.Nz);
    hipLaunchKernelGGL(tfw_grad_kernel, grid, dim3(128), 0, st, gx, gy, gw, x, make_op(v, bx, by, rs));
}

void launch_tfw_correct(hipStream_t st, const TFWView &v, const double *bx, const double *by, const double *rs,
                        double *u, double *vv, double *w, double *th, double *p, const double *us, const double *vs,
                        const double *ws, const double *tn, const double *u0, const double *v0, const double *w0,
                        const double *phi, double dt, double ca, double cb, int combine) {
    dim3 blk(64, 4), grid((v.Nx + 63) / 64, (v.Ny + 3) / 4, (v.Nz + 15) / 16);
    hipLaunchKernelGGL(tfw_correct_march_kernel<16>, grid, blk, 0, st, u, vv, w, th, p, us, vs, ws, tn, u0, v0, w0,
                       phi, make_op(v, bx, by, rs), dt, ca, cb, combine);
}

void launch_tfw_coef(hipStream_t st, const TFWView &v, double *bx, double *by, double *rs) {
    dim3 grid((v.Nx + 127) / 128, v.Ny, v.Nz + 1);
    hipLaunchKernelGGL(tfw_coef_kernel, grid, dim3(128), 0, st, bx, by, rs, make_op(v, bx, by, rs));
}

void launch_tfw_mgcoef(hipStream_t st, const TFWView &v, double *cx, double *cy, double *cz) {
    dim3 grid((v.Nx + 1 + 127) / 128, v.Ny + 1, v.Nz + 1);
    hipLaunchKernelGGL(tfw_mgcoef_kernel, grid, dim3(128), 0, st, cx, cy, cz, make_op(v, nullptr, nullptr, nullptr));
}

}  // namespace aeo

namespace aeo {
void launch_tfw_absdiv(hipStream_t st, const TFWView &v, double *part, int nblocks, const double *b) {
    hipLaunchKernelGGL(tfw_absdiv_kernel, dim3(nblocks), dim3(256), 0, st, part, b, make_op(v, nullptr, nullptr, nullptr));
}
}  // namespace aeo

// ---------------------------------------------------------------------------
// the least-squares guess from earlier solves: with pairs (x_i, b_i) of
// earlier potentials and sources (L x_i = b_i to the tolerance), the guess
// x0 = Σ α_i x_i with α minimising ‖b − Σ α_i b_i‖ (the normal equations
// G α = g, G_ij = b_i·b_j, g_i = b_i·b, solved on the host) has the residual
// b − L x0 ≈ b − Σ α_i b_i, the least in the span: it contains the linear
// and quadratic extrapolations of the same substage. The sums run in a fixed
// order (block partials, then one block per component).
// ---------------------------------------------------------------------------
namespace aeo {
constexpr int TFP_BLOCKS = 1024;

__device__ __forceinline__ double tfp_block_sum(double v, double *sh) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) sh[w] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
        for (int q = 0; q < (int)(blockDim.x >> 6); q++) s += sh[q];
    return s;
}

// block sums of X_{i0+q}·b for q < cnt ≤ 8, one pass over b
__global__ void __launch_bounds__(256) tfp_multidot_kernel(TFBasis X, int i0, int cnt, const double *__restrict__ b,
                                                           size_t n, double *__restrict__ part) {
    __shared__ double sh[4];
    double acc[8] = {};
    for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) {
        const double bt = b[t];
#pragma unroll
        for (int q = 0; q < 8; q++)
            if (q < cnt) acc[q] += X.x[i0 + q][t] * bt;
    }
#pragma unroll
    for (int q = 0; q < 8; q++) {
        if (q >= cnt) break;
        const double s = tfp_block_sum(acc[q], sh);
        if (threadIdx.x == 0) part[(size_t)(i0 + q) * gridDim.x + blockIdx.x] = s;
    }
}

// out[c] = Σ part[c·nblk + q], one block per component
__global__ void tfp_finalize_kernel(double *__restrict__ out, const double *__restrict__ part, int nblk) {
    __shared__ double sh[4];
    double v = 0.0;
    for (int q = threadIdx.x; q < nblk; q += blockDim.x) v += part[(size_t)blockIdx.x * nblk + q];
    const double s = tfp_block_sum(v, sh);
    if (threadIdx.x == 0) out[blockIdx.x] = s;
}

__global__ void tfp_combine_kernel(double *__restrict__ x0, TFBasis X, int k, const double *__restrict__ c, size_t n) {
    for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int i = 0; i < k; i++) s += c[i] * X.x[i][t];
        x0[t] = s;
    }
}

void launch_tfp_dots(hipStream_t st, const TFBasis &X, int k, const double *b, size_t n, double *part, double *out) {
    for (int i0 = 0; i0 < k; i0 += 8)
        hipLaunchKernelGGL(tfp_multidot_kernel, dim3(TFP_BLOCKS), dim3(256), 0, st, X, i0, k - i0 < 8 ? k - i0 : 8, b,
                           n, part);
    hipLaunchKernelGGL(tfp_finalize_kernel, dim3(k), dim3(256), 0, st, out, part, TFP_BLOCKS);
}

void launch_tfp_combine(hipStream_t st, const TFBasis &X, int k, const double *c, size_t n, double *x0) {
    hipLaunchKernelGGL(tfp_combine_kernel, dim3(TFP_BLOCKS), dim3(256), 0, st, x0, X, k, c, n);
}
}  // namespace aeo
