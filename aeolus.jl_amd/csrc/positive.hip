// Positivity-preserving scalar advection (advect_positive!,
// src/AdvectionSchemes.jl:758-1160): the high-order face fluxes are split
// into a first-order upwind part L and an antidiffusive remainder A = F − L,
// and A is scaled on every face by the ratio of the cell it flows out of,
//
//   P⁻_c = Δt Σ_faces max(outflowing A, 0)/Δx_d
//   Q_c  = max(ϕ_c − Δt ∇·L, 0)
//   R_c  = P⁻_c > 0 ? min(1, Q_c/P⁻_c) : 1,
//
// so a forward-Euler update with the same Δt cannot take ϕ below zero.
//
// R needs every face of its cell, and a face's limited flux needs R on both
// sides, with R's halo taken from the caller's boundary conditions (cells on
// the far side of the domain): the grid-wide dependency makes two passes.
//   1. pos_tile_kernel<POS_RATIO>: the face fluxes F (the reconstruction)
//      and L (first-order upwind) of every face of the cell (_b_rflux_*,
//      _b_uflux_*; :858-909) and R of every interior cell
//      (_b_limit_ratio!, :1026-1053);
//   then R's halo (fill_halos! with the caller's BCs, or the one-layer
//   periodic wrap of _wrap_one_layer!, :944-958);
//   2. pos_tile_kernel<POS_DIV>: F and L again, each face limited from R
//      on its two sides and differenced into tend (_b_limit_*!, :1056-1081,
//      fused with _b_flux_div!, :912-928). Both cells of a face evaluate the
//      same expression, so the flux telescopes exactly and Σϕ is conserved.
//
// Workspace (storage-sized, precision T): R. Recomputing F and L in the
// second pass costs their arithmetic twice and saves the six face arrays'
// round trip through memory.
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace aeo {

// Julia's max(x, 0) and min(1, x): NaN propagates
template <typename T> __device__ __forceinline__ T jl_max0(T x) { return x != x ? x : (x > T(0) ? x : T(0)); }
template <typename T> __device__ __forceinline__ T jl_min1(T x) { return x != x ? x : (x < T(1) ? x : T(1)); }

// the limited flux of a face: lo + c·a, a = F − lo, c the ratio of the cell
// below the face when a ≥ 0, of the cell above otherwise
template <typename T> __device__ __forceinline__ T pos_limited(T F, T lo, T r_below, T r_above) {
    const T a = F - lo;
    return lo + (a >= T(0) ? r_below : r_above) * a;
}

// ---------------------------------------------------------------------------
// The two passes, one kernel: a block is 64 x 8 cell columns marching a
// chunk of levels;
//   - every thread keeps its column of ϕ over the z-faces' reach (levels
//     k-R+1 .. k+R) in registers and shifts it up one level per step;
//   - at each level the block writes ϕ's x-y tile with an R-cell halo to
//     LDS (the tile's cells from the registers, the halo from memory, a
//     level ahead, with the level's velocities and, for the divergence,
//     R in the level's plane);
//   - each face (F, L) is computed once per pass: west and south faces into
//     LDS, the top face in a register (the next level's bottom face); wave
//     0 computes the north faces of the top row, wave 1 the east faces of
//     the rows' last cells.
// ---------------------------------------------------------------------------
enum { POS_RATIO = 0, POS_DIV = 1 };
constexpr int PW = 64;  // lanes per wave, cells per tile row
constexpr int PBY = 8;  // rows per tile
constexpr int PKC = 16; // levels per chunk (8 to 32 within 4 % at 256x256x128)

// the face between tile cells at - st and at (F and L), transported by vel
template <int S, int P, typename T>
__device__ __forceinline__ void pos_face(const T *tl, int at, int st, T vel, T ct, T &F, T &Lo) {
    constexpr int R = SchemeInfo<S>::R;
    T a[2 * R];
#pragma unroll
    for (int q = 0; q < 2 * R; q++) a[q] = tl[at + (q - R) * st];
    F = vel * face_of<S, P, T>(a, vel, ct);
    Lo = vel * (vel >= T(0) ? a[R - 1] : a[R]);
}

template <int MODE, int S, int P, typename T>
__global__ void __launch_bounds__(PW *PBY) pos_tile_kernel(T *__restrict__ out, const T *__restrict__ u,
                                                             const T *__restrict__ v, const T *__restrict__ w,
                                                             const T *__restrict__ phi, const T *__restrict__ Rd,
                                                             T dt, Metrics<T> m, int accumulate, int kc) {
    constexpr int R = SchemeInfo<S>::R;
    constexpr int NW = 2 * R;  // registers: levels k-R+1 .. k+R at level k
    constexpr int TW = PW + 2 * R, TH = PBY + 2 * R, TN = TW * TH;
    constexpr int NT = PW * PBY, NHALO = TN - NT, NHP = (NHALO + NT - 1) / NT;
    const int H = m.H;
    const uint32_t sx = m.sx, sxy = (uint32_t)m.sx * m.sy;
    const int lane = threadIdx.x, ty = threadIdx.y, tid = ty * PW + lane;
    int bx, by, bz;
    xcd_block3(bx, by, bz);
    const int i0 = H + bx * PW, jb = H + by * PBY;
    const int i = i0 + lane, j = jb + ty;
    const int k0 = H + bz * kc, k1 = min(k0 + kc, H + m.Nz);
    const int ilast = min(i0 + PW - 1, H + m.Nx - 1), jlast = min(jb + PBY - 1, H + m.Ny - 1);
    const bool ok = i <= ilast && j <= jlast;
    const bool inb = i <= ilast + R && j <= jlast + R;
    const int at = (ty + R) * TW + lane + R;

    __shared__ T tile[TN];
    __shared__ T xf[2][PBY][PW + 1];  // F, L of the west face of cell i0 + c (c = PW: a full row's east face)
    __shared__ T yf[2][PBY + 1][PW];  // F, L of the south face of row jb + r (r = PBY: a full top row's north face)

    uint32_t hoff[NHP];
    int hat[NHP];
    bool hv[NHP];
#pragma unroll
    for (int p = 0; p < NHP; p++) {
        const int h = tid + p * NT;
        int r = 0, c = 0;
        if (h < R * TW) { r = h / TW; c = h % TW; }
        else if (h < 2 * R * TW) { const int h2 = h - R * TW; r = R + PBY + h2 / TW; c = h2 % TW; }
        else { const int h3 = h - 2 * R * TW; r = R + h3 / (2 * R); const int q = h3 % (2 * R); c = q < R ? q : PW + q; }
        const int hi = i0 - R + c, hj = jb - R + r;
        hv[p] = h < NHALO && hi <= ilast + R && hj <= jlast + R;
        hat[p] = r * TW + c;
        hoff[p] = hv[p] ? lin(hi, hj, 0, m.sx, m.sy) : 0u;
    }
    const uint32_t cof = inb ? lin(i, j, 0, m.sx, m.sy) : 0u;

    T win[NW], nxt = T(0), hal[NHP];
#pragma unroll
    for (int n = 0; n < NW; n++) win[n] = T(0);
#pragma unroll
    for (int p = 0; p < NHP; p++) hal[p] = T(0);
    // a level's velocities (the own faces' and the boundary faces' of waves
    // 0 and 1) and, for the divergence, R in the level's plane (the column's
    // R below and at the cell are carried from the level below)
    const int wv = __builtin_amdgcn_readfirstlane(ty);
    T nvu = T(0), nvv = T(0), nvw = T(0), nvb = T(0);
    T nrc = T(0), nrw = T(0), nre = T(0), nrs = T(0), nrn = T(0), nra = T(0);
    auto load_level = [&](int kk) {
        if (inb) nxt = phi[cof + (uint32_t)(kk + R) * sxy];
#pragma unroll
        for (int p = 0; p < NHP; p++)
            if (hv[p]) hal[p] = phi[hoff[p] + (uint32_t)kk * sxy];
        const uint32_t c = cof + (uint32_t)kk * sxy;
        if (ok) {
            nvu = u[c];
            nvv = v[c];
            nvw = w[c + sxy];
            if constexpr (MODE == POS_DIV) {
                nrw = Rd[c - 1];
                nre = Rd[c + 1];
                nrs = Rd[c - sx];
                nrn = Rd[c + sx];
                nra = Rd[c + sxy];
            }
        }
        if (wv == 0 && i0 + lane <= ilast) nvb = v[lin(i0 + lane, jlast + 1, kk, m.sx, m.sy)];
        else if (wv == 1 && lane < PBY && jb + lane <= jlast) nvb = u[lin(ilast + 1, jb + lane, kk, m.sx, m.sy)];
    };
    // the registers at level k0 - 1 and the bottom face of k0 (the top face of k0 - 1)
    if (inb) {
#pragma unroll
        for (int n = 0; n < NW; n++) win[n] = phi[cof + (uint32_t)(k0 - R + n) * sxy];
    }
    T fzb = T(0), lzb = T(0), rb = T(0), rc = T(0);
    if (ok) {
        const T vel = w[cof + (uint32_t)k0 * sxy];
        fzb = vel * face_of<S, P, T>(win, vel, m.teno_ct);
        lzb = vel * (vel >= T(0) ? win[R - 1] : win[R]);
        if constexpr (MODE == POS_DIV) {
            rb = Rd[cof + (uint32_t)(k0 - 1) * sxy];
            rc = Rd[cof + (uint32_t)k0 * sxy];
        }
    }
    load_level(k0);

    for (int k = k0; k < k1; k++) {
#pragma unroll
        for (int n = 0; n < NW - 1; n++) win[n] = win[n + 1];
        win[NW - 1] = nxt;
#pragma unroll
        for (int p = 0; p < NHP; p++)
            if (hv[p]) tile[hat[p]] = hal[p];
        if (inb) tile[at] = win[R - 1];
        const uint32_t c = cof + (uint32_t)k * sxy;
        const T vu = nvu, vv = nvv, vw = nvw, vb = nvb;
        const T rw = nrw, re = nre, rs = nrs, rn = nrn, ra = nra;
        if (k + 1 < k1) load_level(k + 1);
        __syncthreads();

        T fzt = T(0), lzt = T(0);
        if (ok) {
            T F, Lo;
            pos_face<S, P, T>(tile, at, 1, vu, m.teno_ct, F, Lo);
            xf[0][ty][lane] = F;
            xf[1][ty][lane] = Lo;
            pos_face<S, P, T>(tile, at, TW, vv, m.teno_ct, F, Lo);
            yf[0][ty][lane] = F;
            yf[1][ty][lane] = Lo;
            fzt = vw * face_of<S, P, T>(win, vw, m.teno_ct);
            lzt = vw * (vw >= T(0) ? win[R - 1] : win[R]);
        }
        if (wv == 0) {
            const int ii = i0 + lane, rnb = jlast + 1 - jb;
            if (ii <= ilast) {
                T F, Lo;
                pos_face<S, P, T>(tile, (rnb + R) * TW + lane + R, TW, vb, m.teno_ct, F, Lo);
                yf[0][rnb][lane] = F;
                yf[1][rnb][lane] = Lo;
            }
        } else if (wv == 1) {
            const int jj = jb + lane, cb = ilast + 1 - i0;
            if (lane < PBY && jj <= jlast) {
                T F, Lo;
                pos_face<S, P, T>(tile, (lane + R) * TW + cb + R, 1, vb, m.teno_ct, F, Lo);
                xf[0][lane][cb] = F;
                xf[1][lane][cb] = Lo;
            }
        }
        __syncthreads();

        if (ok) {
            const T Fxw = xf[0][ty][lane], Lxw = xf[1][ty][lane], Fxe = xf[0][ty][lane + 1], Lxe = xf[1][ty][lane + 1];
            const T Fys = yf[0][ty][lane], Lys = yf[1][ty][lane], Fyn = yf[0][ty + 1][lane], Lyn = yf[1][ty + 1][lane];
            const T idz = m.m_idz(k);
            if constexpr (MODE == POS_RATIO) {
                // _b_limit_ratio! (src/AdvectionSchemes.jl:1026-1053)
                const T axe = Fxe - Lxe, axw = Fxw - Lxw;
                const T ayn = Fyn - Lyn, ays = Fys - Lys;
                const T azt = fzt - lzt, azb = fzb - lzb;
                const T Pm = dt * (((jl_max0(axe) + jl_max0(-axw)) * m.idx + (jl_max0(ayn) + jl_max0(-ays)) * m.idy) +
                                   (jl_max0(azt) + jl_max0(-azb)) * idz);
                const T div_lo = ((Lxe - Lxw) * m.idx + (Lyn - Lys) * m.idy) + (lzt - lzb) * idz;
                const T Q = jl_max0(win[R - 1] - dt * div_lo);
                out[c] = Pm > T(0) ? jl_min1(Q / Pm) : T(1);
            } else {
                // _b_limit_*! fused with _b_flux_div! (src/AdvectionSchemes.jl:1056-1081, 912-928)
                const T fxw = pos_limited(Fxw, Lxw, rw, rc);
                const T fxe = pos_limited(Fxe, Lxe, rc, re);
                const T fys = pos_limited(Fys, Lys, rs, rc);
                const T fyn = pos_limited(Fyn, Lyn, rc, rn);
                const T fzbl = pos_limited(fzb, lzb, rb, rc);
                const T fztl = pos_limited(fzt, lzt, rc, ra);
                const T d = ((fxe - fxw) * m.idx + (fyn - fys) * m.idy) + (fztl - fzbl) * idz;
                out[c] = accumulate ? out[c] - d : -d;
            }
        }
        fzb = fzt;
        lzb = lzt;
        rb = rc;  // R below and at the cell of the next level
        rc = ra;
    }
}

// two blocks per CU a round: 33×29×25 FP64 86 → 14 us, 100×80×60 FP32
// WENO-Z7 83 → 34 us, 256×256×128 as before (16 levels)
int chunk_limited(int nx, int ny, int nz) {
    return chunk_levels(((nx + PW - 1) / PW) * ((ny + PBY - 1) / PBY), nz, PKC, 512, 1);
}

template <int S, int P, typename T>
static void launch_pos_tile(hipStream_t st, T *tend, T *Rd, const T *u, const T *v, const T *w, const T *phi, T dt,
                            const Metrics<T> &m, const int *bcs, int accumulate) {
    const int kc = chunk_limited(m.Nx, m.Ny, m.Nz);
    const dim3 blk(PW, PBY), grd((m.Nx + PW - 1) / PW, (m.Ny + PBY - 1) / PBY, (m.Nz + kc - 1) / kc);
    hipLaunchKernelGGL((pos_tile_kernel<POS_RATIO, S, P, T>), grd, blk, 0, st, Rd, u, v, w, phi, (const T *)nullptr,
                       dt, m, 0, kc);
    // R's halo: the caller's BCs, or the periodic wrap (whose first layer is
    // the one-layer wrap of the reference; only that layer is read)
    if (bcs) launch_halo<T>(st, Rd, m.Nx, m.Ny, m.Nz, m.H, LOC_CC, bcs[0], bcs[1], bcs[2]);
    else launch_halo<T>(st, Rd, m.Nx, m.Ny, m.Nz, m.H, LOC_CC, BC_PERIODIC, BC_PERIODIC, BC_PERIODIC);
    hipLaunchKernelGGL((pos_tile_kernel<POS_DIV, S, P, T>), grd, blk, 0, st, tend, u, v, w, phi, (const T *)Rd, dt, m,
                       accumulate, kc);
}

template <typename T>
int launch_advect_positive(hipStream_t st, const Metrics<T> &m, int scheme, int p, T *tend, const T *u, const T *v,
                           const T *w, const T *phi, T dt, T *ratio, const int *bcs, int accumulate) {
    switch (scheme) {
    case SCH_CENTERED: launch_pos_tile<SCH_CENTERED, 0, T>(st, tend, ratio, u, v, w, phi, dt, m, bcs, accumulate); break;
    case SCH_WENO_JS5: launch_pos_tile<SCH_WENO_JS5, 0, T>(st, tend, ratio, u, v, w, phi, dt, m, bcs, accumulate); break;
    case SCH_WENO_Z5:
        if (p == 1) launch_pos_tile<SCH_WENO_Z5, 1, T>(st, tend, ratio, u, v, w, phi, dt, m, bcs, accumulate);
        else launch_pos_tile<SCH_WENO_Z5, 2, T>(st, tend, ratio, u, v, w, phi, dt, m, bcs, accumulate);
        break;
    case SCH_WENO_Z7:
        if (p == 1) launch_pos_tile<SCH_WENO_Z7, 1, T>(st, tend, ratio, u, v, w, phi, dt, m, bcs, accumulate);
        else launch_pos_tile<SCH_WENO_Z7, 2, T>(st, tend, ratio, u, v, w, phi, dt, m, bcs, accumulate);
        break;
    case SCH_TENO5: launch_pos_tile<SCH_TENO5, 0, T>(st, tend, ratio, u, v, w, phi, dt, m, bcs, accumulate); break;
    case SCH_TENO8: launch_pos_tile<SCH_TENO8, 0, T>(st, tend, ratio, u, v, w, phi, dt, m, bcs, accumulate); break;
    default: return -1;
    }
    return 0;
}
template int launch_advect_positive<double>(hipStream_t, const Metrics<double> &, int, int, double *, const double *,
                                            const double *, const double *, const double *, double, double *,
                                            const int *, int);
template int launch_advect_positive<float>(hipStream_t, const Metrics<float> &, int, int, float *, const float *,
                                           const float *, const float *, const float *, float, float *,
                                           const int *, int);

}  // namespace aeo
