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

// The tendencies + predictor: a block owns 64 × BY columns and marches a chunk
// of levels, each face flux of the x-y plane computed once.
//   - Every thread keeps its column's values of the four fields over the
//     reach of the σ-stencil (k − 2 .. k + 3) in registers, one load a level;
//     the σ-faces read these, and a level's top fluxes are the next one's
//     bottom fluxes.
//   - The block's tile with a 3-cell halo is in LDS (u, v, w at levels k and
//     k + 1, θ at k), the halo loaded a level ahead; the x- and y-faces read
//     it. A cell computes its west and south fluxes into LDS; its east and
//     north ones are its neighbours'. The last row's north faces take one
//     wave per field, the rows' last east faces 4·BY lanes.
//   - Ω on the faces k + 1 is computed once per column into LDS (and for the
//     row and the column of columns before the block), for the averages that
//     carry u and v up.
//   - ρ̄ J of the points the fluxes live at follows its ratio per (half) level
//     of its column, from one exp per column at the chunk's start, in FP64.
// Two barriers a level: after the tile is written, and after the x-y fluxes and
// Ω are. The buoyancy about θ̄(z) = θ0 + Γz at the w-face follows
// _anelastic_buoyancy (src/Anelastic.jl:1352-1360), formed in FP64 whatever TC
// (θ_face − θ̄ is a small difference of values near 300 K).
//
// What bounds it is the FP64 VALU: about 13 WENO faces a cell, where a thread
// per column that evaluates both faces of each direction has 20 and 15
// density families, and at one wave per SIMD (over 256 registers) issued
// half the time. At 512×512×256 7.95 → 3.58 ms, 320×256×160 with FP32
// fluxes 1.37 → 0.70, 96×96×48 250 → 49 us (chunks of 32 levels on every grid
// before). Two waves per SIMD (227 registers): three for the FP32 form spill
// (0.80 ms); blocks of 8 rows, one per CU: 3.79, 0.67 ms, 46 us.
#pragma clang fp contract(fast)
constexpr int TFT_BY = 4;
constexpr int TFT_KC = 32;     // most levels per chunk
constexpr int TFT_FILL = 512;  // blocks a round: two per CU
template <int S, typename TC, int BY>
__global__ void __launch_bounds__(64 * BY, 2)
    tfw_tendency_tile_kernel(double *__restrict__ us, double *__restrict__ vs, double *__restrict__ ws,
                             double *__restrict__ tn, const double *__restrict__ u, const double *__restrict__ v,
                             const double *__restrict__ w, const double *__restrict__ th,
                             const double *__restrict__ th0, TFM<TC> m, double dt, double ca, double cb, int combine,
                             int raw, int kc) {
    constexpr int R = 3, RL = 2, NW = 6;
    constexpr int TW = 64 + 2 * R, TH = BY + 2 * R, TN = TW * TH, NT = 64 * BY;
    constexpr int NHALO = TN - NT, NHP = (NHALO + NT - 1) / NT;
    constexpr bool DEV = sizeof(TC) == 4;  // θ's fluxes about the cell's own θ
    constexpr int XN = BY * 65, YN = (BY + 1) * 64;
    __shared__ TC tl[6 * TN];                // u, v, w: the levels of even and odd k − k0
    __shared__ double ts[TN];                // θ
    __shared__ TC xs[4 * XN], ys[4 * YN];    // west fluxes [F][row][c], south fluxes [F][r][lane]
    __shared__ TC xm[DEV ? XN : 1], ym[DEV ? YN : 1];  // θ's mass fluxes
    __shared__ TC om[(BY + 1) * 65];         // Ω(k + 1) of column (i0 − 1 + c, jb − 1 + r)
    int bx, by, bz;
    xcd_block3(bx, by, bz);
    const int H = m.H, lane = threadIdx.x, ty = threadIdx.y, tid = ty * 64 + lane;
    const int wv = __builtin_amdgcn_readfirstlane(ty);
    const int i0 = H + bx * 64, jb = H + by * BY, i = i0 + lane, j = jb + ty;
    const int k0 = H + bz * kc, k1 = min(k0 + kc, H + m.Nz);
    const int ilast = min(i0 + 63, H + m.Nx - 1), jlast = min(jb + BY - 1, H + m.Ny - 1);
    const bool ok = i <= ilast && j <= jlast;          // computes its cell
    const bool inb = i <= ilast + R && j <= jlast + R;  // its column feeds the tile
    const int at = (ty + R) * TW + lane + R;
    const int sxi = m.sx;
    const uint32_t sx = (uint32_t)m.sx, sxy = (uint32_t)m.sx * (uint32_t)m.sy;
    const double Hl = (double)m.Hl, iHl = 1.0 / Hl, dz = (double)m.dz, iHs = (double)m.iHs, rho0 = (double)m.rho0;

    // surfaces of the columns the fluxes live on
    auto hd = [&](int a, int b) -> double { return m.h[a + sxi * b]; };
    auto hxd = [&](int a, int b) -> double { return (hd(a, b) + hd(a - 1, b)) / 2; };
    auto hyd = [&](int a, int b) -> double { return (hd(a, b) + hd(a, b - 1)) / 2; };
    auto hxyd = [&](int a, int b) -> double { return (hxd(a, b) + hxd(a, b - 1)) / 2; };
    auto Jd = [&](double hs) -> double { return (Hl - hs) * iHl; };
    // ρ̄ at σ = (k0 − H + off)·dz over surface hs, and its ratio over f levels
    auto rho = [&](double hs, double off) -> double {
        return rho0 * exp(-(hs + ((double)(k0 - H) + off) * dz * Jd(hs)) * iHs);
    };
    auto ratio = [&](double hs, double f) -> double { return exp(-f * dz * Jd(hs) * iHs); };

    // the halo cells this thread loads: bottom and top R rows, then the left
    // and right R columns; cells past the last cell + R feed nothing
    uint32_t hof[NHP];
    int hat[NHP];
    bool hv[NHP];
#pragma unroll
    for (int p = 0; p < NHP; p++) {
        const int e = tid + p * NT;
        int r, c;
        if (e < 2 * R * TW) {
            r = e / TW;
            c = e % TW;
            if (r >= R) r += BY;
        } else {
            const int e2 = e - 2 * R * TW, q = e2 % (2 * R);
            r = R + e2 / (2 * R);
            c = q < R ? q : 64 + q;
        }
        const int hi = i0 - R + c, hj = jb - R + r;
        hv[p] = e < NHALO && hi <= ilast + R && hj <= jlast + R;
        hat[p] = r * TW + c;
        hof[p] = hv[p] ? lin(hi, hj, 0, m.sx, m.sy) : 0u;
    }
    const uint32_t cof = inb ? lin(i, j, 0, m.sx, m.sy) : 0u;

    TC win[3][NW];
    double wt[NW], nxt[4], hal[4][NHP];
#pragma unroll
    for (int n = 0; n < NW; n++) {
        const uint32_t c = cof + (uint32_t)(k0 - 1 - RL + n) * sxy;
        win[0][n] = inb ? (TC)u[c] : TC(0);
        win[1][n] = inb ? (TC)v[c] : TC(0);
        win[2][n] = inb ? (TC)w[c] : TC(0);
        wt[n] = inb ? th[c] : 0.0;
    }
    // the own column's top values and the tile's halo of level kk (u, v, w one further)
    auto load_level = [&](int kk) {
        const uint32_t c = cof + (uint32_t)(kk + R) * sxy;
        nxt[0] = inb ? u[c] : 0.0;
        nxt[1] = inb ? v[c] : 0.0;
        nxt[2] = inb ? w[c] : 0.0;
        nxt[3] = inb ? th[c] : 0.0;
#pragma unroll
        for (int p = 0; p < NHP; p++) {
            if (hv[p]) {
                const uint32_t h0 = hof[p] + (uint32_t)kk * sxy, h1 = h0 + sxy;
                hal[0][p] = u[h1];
                hal[1][p] = v[h1];
                hal[2][p] = w[h1];
                hal[3][p] = th[h0];
            }
        }
    };
    // the tile of u, v, w at k0
#pragma unroll
    for (int p = 0; p < NHP; p++) {
        if (hv[p]) {
            const uint32_t h0 = hof[p] + (uint32_t)k0 * sxy;
            tl[hat[p]] = (TC)u[h0];
            tl[2 * TN + hat[p]] = (TC)v[h0];
            tl[4 * TN + hat[p]] = (TC)w[h0];
        }
    }
    if (inb) {
        tl[at] = win[0][RL + 1];
        tl[2 * TN + at] = win[1][RL + 1];
        tl[4 * TN + at] = win[2][RL + 1];
    }
    load_level(k0);

    // the thread's metric terms: ρ̄ at the σ-face k of its column, x-face and
    // y-face (r), the ratio per half level (q), J; ρ̄J at the centres i − 1,
    // j − 1 and at the corner (i, j), and the ratios per level
    double r0 = 0, q0 = 0, rx = 0, qx = 0, ry = 0, qy = 0, ga = 0, qa = 0, gb = 0, qb = 0, gc = 0, qc = 0;
    TC J0 = 0, Jx = 0, Jy = 0, hx0 = 0, hy0 = 0, uc = 0, vc = 0;
    TC Om0 = 0, FBm = 0, FBf = 0, FBu = 0, FBv = 0, FBw = 0;
    if (ok) {
        const double h00 = hd(i, j), hw = hd(i - 1, j), hs = hd(i, j - 1), hx = hxd(i, j), hy = hyd(i, j), hc = hxyd(i, j);
        r0 = rho(h00, 0.0); q0 = ratio(h00, 0.5);
        rx = rho(hx, 0.0); qx = ratio(hx, 0.5);
        ry = rho(hy, 0.0); qy = ratio(hy, 0.5);
        ga = rho(hw, 0.5) * Jd(hw); qa = ratio(hw, 1.0);
        gb = rho(hs, 0.5) * Jd(hs); qb = ratio(hs, 1.0);
        gc = rho(hc, 0.5) * Jd(hc); qc = ratio(hc, 1.0);
        J0 = (TC)Jd(h00); Jx = (TC)Jd(hx); Jy = (TC)Jd(hy);
        hx0 = (TC)m.hx[i + sxi * j]; hy0 = (TC)m.hy[i + sxi * j];
        // Ω at the σ-face kk of column (i + di, j + dj)
        auto Om = [&](int di, int dj, int kk) -> TC {
            if (kk == H || kk == H + m.Nz) return TC(0);
            const uint32_t c = lin(i + di, j + dj, kk, m.sx, m.sy);
            const TC ub = TC(0.25) * (((TC)u[c - sxy] + (TC)u[c - sxy + 1]) + ((TC)u[c] + (TC)u[c + 1]));
            const TC vb = TC(0.25) * (((TC)v[c - sxy] + (TC)v[c - sxy + sx]) + ((TC)v[c] + (TC)v[c + sx]));
            return (TC)w[c] + (m.jsx(i + di, j + dj, kk) * ub + m.jsy(i + di, j + dj, kk) * vb);
        };
        const uint32_t c = cof + (uint32_t)k0 * sxy;
        uc = (TC)u[c] + (TC)u[c + 1];
        vc = (TC)v[c] + (TC)v[c + sx];
        Om0 = Om(0, 0, k0);
        // the fluxes through the faces k0 (w's: through the centre k0 − 1)
        const TC Ft = (TC)r0 * Om0;
        const TC Wu = (TC)rx * ((Om(-1, 0, k0) + Om0) * TC(0.5)), Wv = (TC)ry * ((Om(0, -1, k0) + Om0) * TC(0.5));
        const TC Ww = (TC)(r0 / q0) * ((Om(0, 0, k0 - 1) + Om0) * TC(0.5));
        FBm = Ft;
        if constexpr (DEV) {
            const double b = wt[RL + 1];  // about θ of level k0
            FBf = tf_face6<S, TC>((TC)(wt[0] - b), (TC)(wt[1] - b), (TC)(wt[2] - b), TC(0), (TC)(wt[4] - b), (TC)(wt[5] - b), Ft);
        } else {
            FBf = tf_face6<S, TC>(wt[0], wt[1], wt[2], wt[3], wt[4], wt[5], Ft);
        }
        FBu = Wu * tf_face6<S, TC>(win[0][0], win[0][1], win[0][2], win[0][3], win[0][4], win[0][5], Wu);
        FBv = Wv * tf_face6<S, TC>(win[1][0], win[1][1], win[1][2], win[1][3], win[1][4], win[1][5], Wv);
        FBw = Ww * tf_face6<S, TC>(win[2][0], win[2][1], win[2][2], win[2][3], win[2][4], win[2][5], Ww);
    }
    // a face of the block's far edges: the field's tile cell f whose west or
    // south face it is (stride st), the velocities at tile cells A and B (w:
    // one cell, at levels k − 1 and k), ρ̄J there and its ratio per level
    struct Item {
        double r, q;
        TC prev;
        int F, f, st, A, B, dst;
    };
    Item it[2];
    it[0].F = it[1].F = -1;
    auto set_item = [&](Item &t, int F, int a, int b, int dir) {  // the minus face of cell (a, b) in direction dir
        const int cell = (b - jb + R) * TW + (a - i0 + R), vel = dir == 0 ? 0 : 2 * TN;
        const int st = dir == 0 ? 1 : TW;
        t.F = F;
        t.f = cell;
        t.st = st;
        t.B = vel + cell;
        t.A = t.B;
        t.prev = TC(0);
        double hs, off = 0.5;
        if (F == 3) hs = dir == 0 ? hxd(a, b) : hyd(a, b);
        else if (F == dir) {
            hs = dir == 0 ? hd(a - 1, b) : hd(a, b - 1);
            t.A = t.B - st;
        } else if (F == 2) {
            hs = dir == 0 ? hxd(a, b) : hyd(a, b);
            off = 0.0;
            const uint32_t c = lin(a, b, k0 - 1, m.sx, m.sy);
            t.prev = (TC)(dir == 0 ? u[c] : v[c]);
        } else {
            hs = hxyd(a, b);
            t.A = t.B - (F == 0 ? 1 : TW);
        }
        t.r = rho(hs, off) * Jd(hs);
        t.q = ratio(hs, 1.0);
        t.dst = dir == 0 ? F * XN + (b - jb) * 65 + (a - i0) : F * YN + (b - jb) * 64 + (a - i0);
    };
    if (wv < 4 && i <= ilast) set_item(it[0], wv, i, jlast + 1, 1);
    constexpr int WE = BY == 4 ? 1 : 4;  // the waves of the east faces: u, v, w; θ
    if (wv == WE && lane < 3 * BY && jb + lane % BY <= jlast) set_item(it[1], lane / BY, ilast + 1, jb + lane % BY, 0);
    if (wv == WE + 1 && lane < BY && jb + lane <= jlast) set_item(it[1], 3, ilast + 1, jb + lane, 0);
    // Ω of the row (wave 0) and the column (wave 3) before the block
    int oat = -1, odst = 0;
    TC ohx = 0, ohy = 0;
    if ((wv == 0 && i <= ilast) || (wv == 3 && lane < BY && jb + lane <= jlast)) {
        const int a = wv == 0 ? i : i0 - 1, b = wv == 0 ? jb - 1 : jb + lane;
        oat = (b - jb + R) * TW + (a - i0 + R);
        odst = (b - jb + 1) * 65 + (a - i0 + 1);
        ohx = (TC)m.hx[a + sxi * b];
        ohy = (TC)m.hy[a + sxi * b];
    }

    // the minus face of tile cell f: a velocity vel, stride st
    auto face = [&](const TC *f, int st, TC vel) -> TC {
        return vel * tf_face6<S, TC>(f[-3 * st], f[-2 * st], f[-st], f[0], f[st], f[2 * st], vel);
    };
    // θ's: FP64 the flux; FP32 the flux of θ less the θ of the cell f
    auto face_t = [&](const double *f, int st, TC vel) -> TC {
        const double b = DEV ? f[0] : 0.0;
        return vel * tf_face6<S, TC>((TC)(f[-3 * st] - b), (TC)(f[-2 * st] - b), (TC)(f[-st] - b), (TC)(f[0] - b),
                                     (TC)(f[st] - b), (TC)(f[2 * st] - b), vel);
    };
    auto run_item = [&](Item &t, TC *out, TC *mout, int po) {
        if (t.F >= 0) {
            const TC B = tl[t.B + po];
            const TC A = t.F == 2 ? t.prev : tl[t.A + po];
            const TC vel = (TC)t.r * ((A + B) * TC(0.5));
            t.prev = B;
            t.r *= t.q;
            if (t.F == 3) {
                out[t.dst] = face_t(ts + t.f, t.st, vel);
                if constexpr (DEV) mout[t.dst - 3 * (out == xs ? XN : YN)] = vel;
            } else {
                out[t.dst] = face(tl + 2 * t.F * TN + t.f + po, t.st, vel);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    for (int k = k0; k < k1; k++) {
        const int po = ((k - k0) & 1) * TN, pn = TN - po;  // the slots of levels k and k + 1
#pragma unroll
        for (int n = 0; n < NW - 1; n++) {
            win[0][n] = win[0][n + 1]; win[1][n] = win[1][n + 1]; win[2][n] = win[2][n + 1];
            wt[n] = wt[n + 1];
        }
        win[0][NW - 1] = (TC)nxt[0]; win[1][NW - 1] = (TC)nxt[1]; win[2][NW - 1] = (TC)nxt[2];
        wt[NW - 1] = nxt[3];
#pragma unroll
        for (int p = 0; p < NHP; p++) {
            if (hv[p]) {
                tl[pn + hat[p]] = (TC)hal[0][p];
                tl[2 * TN + pn + hat[p]] = (TC)hal[1][p];
                tl[4 * TN + pn + hat[p]] = (TC)hal[2][p];
                ts[hat[p]] = hal[3][p];
            }
        }
        if (k + 1 < k1) load_level(k + 1);  // in flight over this level's faces
        if (inb) {
            tl[pn + at] = win[0][RL + 1];
            tl[2 * TN + pn + at] = win[1][RL + 1];
            tl[4 * TN + pn + at] = win[2][RL + 1];
            ts[at] = wt[RL];
        }
        __syncthreads();

        const TC *tu = tl + po + at, *tv = tu + 2 * TN, *tw = tu + 4 * TN;
        const double *tt_ = ts + at;
        const double rc = r0 * q0;                                   // ρ̄ at the centre k
        const TC mx = (TC)(rx * qx) * Jx, my = (TC)(ry * qy) * Jy;  // ρ̄J at the x- and the y-face
        const TC tauf = ((TC)(k + 1 - H) * m.dz - m.Hl) * m.iHl;    // −τ/H of the face k + 1
        TC Om1 = TC(0), de = TC(0), dn = TC(0);
        if (ok) {
            const TC U = win[0][RL], V = win[1][RL];
            // Ω(k + 1)
            const TC u1 = win[0][RL + 1] + tl[pn + at + 1], v1 = win[1][RL + 1] + tl[2 * TN + pn + at + TW];
            if (k + 1 < H + m.Nz)
                Om1 = win[2][RL + 1] + tauf * TC(0.25) * (hx0 * (uc + u1) + hy0 * (vc + v1));
            om[(ty + 1) * 65 + lane + 1] = Om1;
            uc = u1;
            vc = v1;
            TC *xo = xs + ty * 65 + lane, *yo = ys + ty * 64 + lane;
            const TC ul = tu[-1], vl = tv[-1], ud = tu[-TW], vd = tv[-TW];
            xo[0] = face(tu, 1, (TC)ga * ((ul + U) * TC(0.5)));
            __builtin_amdgcn_sched_barrier(0);
            yo[0] = face(tu, TW, (TC)gc * ((vl + V) * TC(0.5)));
            __builtin_amdgcn_sched_barrier(0);
            xo[XN] = face(tv, 1, (TC)gc * ((ud + U) * TC(0.5)));
            __builtin_amdgcn_sched_barrier(0);
            yo[YN] = face(tv, TW, (TC)gb * ((vd + V) * TC(0.5)));
            __builtin_amdgcn_sched_barrier(0);
            xo[2 * XN] = face(tw, 1, (TC)rx * Jx * ((win[0][RL - 1] + U) * TC(0.5)));
            __builtin_amdgcn_sched_barrier(0);
            yo[2 * YN] = face(tw, TW, (TC)ry * Jy * ((win[1][RL - 1] + V) * TC(0.5)));
            __builtin_amdgcn_sched_barrier(0);
            xo[3 * XN] = face_t(tt_, 1, mx * U);
            __builtin_amdgcn_sched_barrier(0);
            yo[3 * YN] = face_t(tt_, TW, my * V);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (DEV) {
                xm[ty * 65 + lane] = mx * U;
                ym[ty * 64 + lane] = my * V;
                de = (TC)(tt_[1] - wt[RL]);
                dn = (TC)(tt_[TW] - wt[RL]);
            }
        }
        run_item(it[0], ys, ym, po);
        run_item(it[1], xs, xm, po);
        if (oat >= 0) {
            TC o = TC(0);
            if (k + 1 < H + m.Nz) {
                const TC *a = tl + po + oat, *b = tl + pn + oat;
                const TC *av = a + 2 * TN, *bv = b + 2 * TN;
                o = b[4 * TN] + tauf * TC(0.25) * (ohx * ((a[0] + a[1]) + (b[0] + b[1])) + ohy * ((av[0] + av[TW]) + (bv[0] + bv[TW])));
            }
            om[odst] = o;
        }
        __syncthreads();

        if (ok) {
            const uint32_t c = cof + (uint32_t)k * sxy;
            const double r1 = rc * q0, rx1 = rx * qx * qx, ry1 = ry * qy * qy;  // at the faces k + 1
            const TC *xo = xs + ty * 65 + lane, *yo = ys + ty * 64 + lane;
            // u
            const TC Wu = (TC)rx1 * ((om[(ty + 1) * 65 + lane] + Om1) * TC(0.5));
            const TC FTu = Wu * tf_face6<S, TC>(win[0][0], win[0][1], win[0][2], win[0][3], win[0][4], win[0][5], Wu);
            const TC tu_ = -qdiv<TC>(((xo[1] - xo[0]) * m.idx + (yo[64] - yo[0]) * m.idy) + (FTu - FBu) * m.idz, mx);
            FBu = FTu;
            us[c] = raw ? (double)tu_ : (DEV ? u[c] : (double)win[0][RL]) + dt * (double)tu_;
            __builtin_amdgcn_sched_barrier(0);
            // v
            const TC Wv = (TC)ry1 * ((om[ty * 65 + lane + 1] + Om1) * TC(0.5));
            const TC FTv = Wv * tf_face6<S, TC>(win[1][0], win[1][1], win[1][2], win[1][3], win[1][4], win[1][5], Wv);
            const TC tv_ = -qdiv<TC>(((xo[XN + 1] - xo[XN]) * m.idx + (yo[YN + 64] - yo[YN]) * m.idy) + (FTv - FBv) * m.idz, my);
            FBv = FTv;
            vs[c] = raw ? (double)tv_ : (DEV ? v[c] : (double)win[1][RL]) + dt * (double)tv_;
            __builtin_amdgcn_sched_barrier(0);
            // w at the σ-face k (the ground face is diagnostic); its upper flux is carried whatever k
            const TC Ww = (TC)rc * ((Om0 + Om1) * TC(0.5));
            const TC FTw = Ww * tf_face6<S, TC>(win[2][0], win[2][1], win[2][2], win[2][3], win[2][4], win[2][5], Ww);
            TC tw_ = TC(0);
            if (k > H) {
                tw_ = -qdiv<TC>(((xo[2 * XN + 1] - xo[2 * XN]) * m.idx + (yo[2 * YN + 64] - yo[2 * YN]) * m.idy) +
                                    (FTw - FBw) * m.idz, (TC)r0 * J0);
                if (m.buoyancy) {
                    const TC zf = m.hp(i, j) + m.sigf(k) * J0;
                    const double tb = (double)m.theta0 + (double)m.gamma * (double)zf;
                    tw_ += (TC)((double)m.g / tb * (0.5 * (wt[RL - 1] + wt[RL]) - tb));
                }
            }
            FBw = FTw;
            const double w0 = DEV ? w[c] : (double)win[2][RL];
            ws[c] = raw ? (double)tw_ : k > H ? w0 + dt * (double)tw_ : w0;
            __builtin_amdgcn_sched_barrier(0);
            // θ
            const TC FT = (TC)r1 * Om1;
            TC d, FTf;
            if constexpr (DEV) {
                // the flux form less θ_c·(B u)/(ρJ): B u vanishes to the projection's tolerance, and its
                // FP32 rounding times θ ≈ 300 K would swamp the tendency of the perturbation
                const double b = wt[RL];
                FTf = tf_face6<S, TC>((TC)(wt[0] - b), (TC)(wt[1] - b), TC(0), (TC)(wt[3] - b), (TC)(wt[4] - b), (TC)(wt[5] - b), FT);
                const TC FE = xo[3 * XN + 1] + xm[ty * 65 + lane + 1] * de, FN = yo[3 * YN + 64] + ym[(ty + 1) * 64 + lane] * dn;
                d = ((FE - xo[3 * XN]) * m.idx + (FN - yo[3 * YN]) * m.idy) + (FT * FTf - FBm * FBf) * m.idz;
                FBf = FTf - (TC)(wt[RL + 1] - wt[RL]);  // re-based on θ of level k + 1
            } else {
                FTf = tf_face6<S, TC>(wt[0], wt[1], wt[2], wt[3], wt[4], wt[5], FT);
                d = ((xo[3 * XN + 1] - xo[3 * XN]) * m.idx + (yo[3 * YN + 64] - yo[3 * YN]) * m.idy) + (FT * FTf - FBm * FBf) * m.idz;
                FBf = FTf;
            }
            FBm = FT;
            const double tt = (double)-qdiv<TC>(d, (TC)rc * J0);
            const double tnew = wt[RL] + dt * tt;
            tn[c] = raw ? tt : combine ? ca * th0[c] + cb * tnew : tnew;
            Om0 = Om1;
            r0 = r1;
            rx = rx1;
            ry = ry1;
            ga *= qa;
            gb *= qb;
            gc *= qc;
        }
        // no barrier here: the next level's tile writes touch nothing this phase reads
    }
}
#pragma clang fp contract(off)

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
// periodic x, y halos of a field over every storage level: a work item per
// halo cell of level blockIdx.y, the 2H whole rows first, then 2H columns of
// the interior rows. Bound: latency and the columns' partial lines. An item per
// storage cell, most leaving at once: 284 us at 512×512×256 → 15 us.
__global__ void tfw_xy_halo_kernel(double *__restrict__ f, TFM<double> m) {
    const int H2 = 2 * m.H, k = blockIdx.y;
    int t = blockIdx.x * blockDim.x + threadIdx.x, i, j;
    if (t < H2 * m.sx) {
        const int r = t / m.sx;
        i = t - r * m.sx;
        j = r < m.H ? r : r + m.Ny;
    } else {
        t -= H2 * m.sx;
        if (t >= H2 * m.Ny) return;
        const int r = t / H2, q = t - r * H2;
        j = r + m.H;
        i = q < m.H ? q : q + m.Nx;
    }
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

// u = c(u0, u* − Gxφ), v, w (interior σ-faces); θ = θ'; p = φ/Δt (p nullable),
// by columns: thread (a, b) marches CH levels with rolling windows of φ on its
// own, west and south columns and of their metric terms S; the same G as
// tfw_grad_kernel without its recomputation
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

int chunk_tfw_tendency(int nx, int ny, int nz) {
    return chunk_levels(((nx + 63) / 64) * ((ny + TFT_BY - 1) / TFT_BY), nz, TFT_KC, TFT_FILL, 2);
}
int chunk_tfw_apply(int nx, int ny, int nz) {
    return chunk_levels(((nx + 63) / 64) * ((ny + TFA_BY - 1) / TFA_BY), nz, TFA_KC, TFA_FILL, 4);
}

template <int S, typename TC>
static void launch_tendency_tile(hipStream_t st, const TFWView &v, double *us, double *vs, double *ws, double *tn,
                                 const double *u, const double *vv, const double *w, const double *th,
                                 const double *th0, double dt, double ca, double cb, int combine, int raw) {
    constexpr int BY = TFT_BY;
    const int tx = (v.Nx + 63) / 64, ty = (v.Ny + BY - 1) / BY;
    const int kc = chunk_tfw_tendency(v.Nx, v.Ny, v.Nz);
    hipLaunchKernelGGL((tfw_tendency_tile_kernel<S, TC, BY>), dim3(tx, ty, (v.Nz + kc - 1) / kc), dim3(64, BY), 0, st,
                       us, vs, ws, tn, u, vv, w, th, th0, make_tfm<TC>(v), dt, ca, cb, combine, raw, kc);
}

int launch_tfw_tendency(hipStream_t st, const TFWView &v, int scheme, int f32, double *us, double *vs, double *ws,
                        double *tn, const double *u, const double *vv, const double *w, const double *th,
                        const double *th0, double dt, double ca, double cb, int combine, int raw) {
    if (scheme == SCH_CENTERED) {
        if (f32) launch_tendency_tile<SCH_CENTERED, float>(st, v, us, vs, ws, tn, u, vv, w, th, th0, dt, ca, cb, combine, raw);
        else launch_tendency_tile<SCH_CENTERED, double>(st, v, us, vs, ws, tn, u, vv, w, th, th0, dt, ca, cb, combine, raw);
    } else if (scheme == SCH_WENO_Z5) {
        if (f32) launch_tendency_tile<SCH_WENO_Z5, float>(st, v, us, vs, ws, tn, u, vv, w, th, th0, dt, ca, cb, combine, raw);
        else launch_tendency_tile<SCH_WENO_Z5, double>(st, v, us, vs, ws, tn, u, vv, w, th, th0, dt, ca, cb, combine, raw);
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
    hipLaunchKernelGGL(tfw_xy_halo_kernel, dim3((2 * v.H * (v.sx + v.Ny) + 255) / 256, v.Nz + 2 * v.H), dim3(256), 0, st, w, m);
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
    const int kc = chunk_tfw_apply(v.Nx, v.Ny, v.Nz);
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
