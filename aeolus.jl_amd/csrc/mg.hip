// Geometric multigrid and the MG-preconditioned CG (gfx950).
//
// MultigridPoissonSolver / MGPreconditionedCG (src/Multigrid.jl:531-972) with
// the CG loop of pcg! (src/Backends.jl:1526-1589): cell-centred V-cycle,
// red-black Gauss-Seidel (the reference's smoother) or damped Jacobi,
// 8-cell mean restriction with the residual mean subtracted inside,
// trilinear (3/4, 1/4) prolongation, 4-face mean coefficient coarsening, 50
// red-black sweeps on the coarsest level, and the null-space (mean)
// projection after each smoothing, residual and prolongation.
//
// Device design: level arrays are interior-sized; the unit halo of the
// reference (periodic wrap or mirror) is an index map in the kernels, so no
// halo launches. Every mean projection stays on the device (block partial
// sums, one finalize launch writing the mean, the shift reads it), so a
// V-cycle runs without a host synchronisation. The coarsest level runs its
// 50 sweeps in one workgroup with the level in LDS. The V-cycle runs in T =
// float or double; the outer CG is FP64 (its residual and inner products).
// The reductions are deterministic (a fixed tree per launch geometry); their
// order differs from the reference's 8-lane plane order, so iterates agree
// with the CPU restatement to round-off, not bit for bit.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <vector>

#include "kernels.h"

namespace aeo {

constexpr int RB = 256;  // threads of the reduction / elementwise launches

__device__ __forceinline__ int wrapc(int i, int n, int bc) {
    if (i < 0) return bc == BC_PERIODIC ? i + n : 0;
    if (i >= n) return bc == BC_PERIODIC ? i - n : n - 1;
    return i;
}

template <typename T>
struct LevelD {
    int nx, ny, nz;
    T ix2, iy2, iz2;
    T *phi, *b, *r, *tmp;
    const T *cx, *cy, *cz;  // face coefficients or null (the constant operator)
    int bcx, bcy, bcz;
};

template <typename T>
__device__ __forceinline__ uint32_t lidx(const LevelD<T> &L, int i, int j, int k) {
    return (uint32_t)i + (uint32_t)L.nx * ((uint32_t)j + (uint32_t)L.ny * (uint32_t)k);
}

// The FP64 terrain solve keeps the finest level's φ colour-split: cell
// (i, j, k) at ((i + j + k) & 1)·half + (its linear index q ≫ 1), a
// bijection for even nx (q and q + 1 differ in colour). A red-black pass
// then writes whole lines of its colour's half and reads the other half as
// neighbours. half = 0: the natural layout.
struct SplitMap {
    uint32_t half;
    int nx, ny;
    int shx, shy;  // log2 nx, log2 ny when both are powers of two, else −1
};
__device__ __forceinline__ uint32_t split_at(uint32_t half, int i, int j, int k, uint32_t q) {
    return half ? (((i + j + k) & 1) ? half : 0u) + (q >> 1) : q;
}
// the same for a linear index t of the natural layout
__device__ __forceinline__ uint32_t split_t(const SplitMap &s, uint32_t t) {
    if (!s.half) return t;
    uint32_t par;
    if (s.shx >= 0) {  // the parities of i, j, k are bits of t
        par = (t ^ (t >> s.shx) ^ (t >> (s.shx + s.shy))) & 1u;
    } else {
        const uint32_t jk = t / (uint32_t)s.nx, i = t - jk * (uint32_t)s.nx;
        const uint32_t k = jk / (uint32_t)s.ny, j = jk - k * (uint32_t)s.ny;
        par = (i + j + k) & 1u;
    }
    return (par ? s.half : 0u) + (t >> 1);
}

// (Aφ) at interior (i, j, k): _Aφ, src/Multigrid.jl:171-192
// SH: every value read as f − m (a pending mean removal, shift_kernel's values)
template <typename T, bool SH = false>
__device__ __forceinline__ T applyA(const LevelD<T> &L, const T *__restrict__ f, int i, int j, int k, T m = T(0)) {
    auto rd = [&](uint32_t q) -> T { return SH ? f[q] - m : f[q]; };
    const T c = rd(lidx(L, i, j, k));
    const T xp = rd(lidx(L, wrapc(i + 1, L.nx, L.bcx), j, k)), xm = rd(lidx(L, wrapc(i - 1, L.nx, L.bcx), j, k));
    const T yp = rd(lidx(L, i, wrapc(j + 1, L.ny, L.bcy), k)), ym = rd(lidx(L, i, wrapc(j - 1, L.ny, L.bcy), k));
    const T zp = rd(lidx(L, i, j, wrapc(k + 1, L.nz, L.bcz))), zm = rd(lidx(L, i, j, wrapc(k - 1, L.nz, L.bcz)));
    if (!L.cx) {
        return (((xp - T(2) * c) + xm) * L.ix2 + ((yp - T(2) * c) + ym) * L.iy2) + ((zp - T(2) * c) + zm) * L.iz2;
    }
    const uint32_t nx1 = L.nx + 1, ny1 = L.ny + 1;
    const T fxp = L.cx[(uint32_t)(i + 1) + nx1 * ((uint32_t)j + (uint32_t)L.ny * k)];
    const T fxm = L.cx[(uint32_t)i + nx1 * ((uint32_t)j + (uint32_t)L.ny * k)];
    const T fyp = L.cy[(uint32_t)i + (uint32_t)L.nx * ((uint32_t)(j + 1) + ny1 * k)];
    const T fym = L.cy[(uint32_t)i + (uint32_t)L.nx * ((uint32_t)j + ny1 * k)];
    const T fzp = L.cz[lidx(L, i, j, k + 1)];
    const T fzm = L.cz[lidx(L, i, j, k)];
    return ((fxp * (xp - c) - fxm * (c - xm)) * L.ix2 + (fyp * (yp - c) - fym * (c - ym)) * L.iy2) +
           (fzp * (zp - c) - fzm * (c - zm)) * L.iz2;
}

template <typename T>
__device__ __forceinline__ T diagA(const LevelD<T> &L, int i, int j, int k) {
    if (!L.cx) return T(-2) * ((L.ix2 + L.iy2) + L.iz2);
    const uint32_t nx1 = L.nx + 1, ny1 = L.ny + 1;
    const T fxp = L.cx[(uint32_t)(i + 1) + nx1 * ((uint32_t)j + (uint32_t)L.ny * k)];
    const T fxm = L.cx[(uint32_t)i + nx1 * ((uint32_t)j + (uint32_t)L.ny * k)];
    const T fyp = L.cy[(uint32_t)i + (uint32_t)L.nx * ((uint32_t)(j + 1) + ny1 * k)];
    const T fym = L.cy[(uint32_t)i + (uint32_t)L.nx * ((uint32_t)j + ny1 * k)];
    const T fzp = L.cz[lidx(L, i, j, k + 1)];
    const T fzm = L.cz[lidx(L, i, j, k)];
    return -(((fxp + fxm) * L.ix2 + (fyp + fym) * L.iy2) + (fzp + fzm) * L.iz2);
}

// ---- block reduction: partial[blockIdx] = Σ over the block of v (FP64) ------
__device__ __forceinline__ double block_sum(double v, double *sh) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) sh[w] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0) {
        const int nw = (blockDim.x + 63) >> 6;
        for (int q = 0; q < nw; q++) s += sh[q];
    }
    __syncthreads();
    return s;
}

// out[0] = Σ partials (fixed order) * scale; `n` partials
__global__ void finalize_kernel(double *__restrict__ out, const double *__restrict__ partials, int n, double scale) {
    __shared__ double sh[RB / 64];
    double v = 0.0;
    for (int q = threadIdx.x; q < n; q += blockDim.x) v += partials[q];
    double s = block_sum(v, sh);
    if (threadIdx.x == 0) out[0] = s * scale;
}

// several sums at once: partials laid out [comp][n]
__global__ void finalize_multi_kernel(double *__restrict__ out, const double *__restrict__ partials, int n, int ncomp) {
    __shared__ double sh[RB / 64];
    for (int c = 0; c < ncomp; c++) {
        double v = 0.0;
        for (int q = threadIdx.x; q < n; q += blockDim.x) v += partials[(size_t)c * n + q];
        double s = block_sum(v, sh);
        if (threadIdx.x == 0) out[c] = s;
    }
}

// the first stage of a long multi-component list: block (c, q) sums the
// q-th of gridDim.y contiguous segments of component c into out[c·gridDim.y + q]
__global__ void fold_multi_kernel(double *__restrict__ out, const double *__restrict__ partials, int n) {
    __shared__ double sh[RB / 64];
    const int c = blockIdx.x, q = blockIdx.y, nseg = gridDim.y;
    const int lo = (int)((long long)n * q / nseg), hi = (int)((long long)n * (q + 1) / nseg);
    double v = 0.0;
    for (int t = lo + threadIdx.x; t < hi; t += blockDim.x) v += partials[(size_t)c * n + t];
    const double s = block_sum(v, sh);
    if (threadIdx.x == 0) out[(size_t)c * nseg + q] = s;
}

// ---- V-cycle kernels --------------------------------------------------------
// the red-black value of cell (i, j, k) from its six neighbours' values
// (_rbgs_body!, src/Multigrid.jl:307-337); a fully blocked cell keeps `self`
// with the six face coefficients given
template <typename T>
__device__ __forceinline__ T rb_value_c(const LevelD<T> &L, T bv, T fxp, T fxm, T fyp, T fym, T fzp, T fzm, T xp,
                                        T xm, T yp, T ym, T zp, T zm, T self) {
    const T diag = -(((fxp + fxm) * L.ix2 + (fyp + fym) * L.iy2) + (fzp + fzm) * L.iz2);
    if (fabs(diag) < Eps<T>::v) return self;  // a fully blocked cell
    const T off = ((fxp * xp + fxm * xm) * L.ix2 + (fyp * yp + fym * ym) * L.iy2) + (fzp * zp + fzm * zm) * L.iz2;
    return (bv - off) / diag;
}

template <typename T>
__device__ __forceinline__ T rb_value(const LevelD<T> &L, int i, int j, int k, T xp, T xm, T yp, T ym, T zp, T zm,
                                      T self, T bv) {
    if (!L.cx) {
        const T diag = T(-2) * ((L.ix2 + L.iy2) + L.iz2);
        const T off = ((xp + xm) * L.ix2 + (yp + ym) * L.iy2) + (zp + zm) * L.iz2;
        return (bv - off) / diag;
    }
    const uint32_t nx1 = L.nx + 1, ny1 = L.ny + 1;
    const T fxp = L.cx[(uint32_t)(i + 1) + nx1 * ((uint32_t)j + (uint32_t)L.ny * k)];
    const T fxm = L.cx[(uint32_t)i + nx1 * ((uint32_t)j + (uint32_t)L.ny * k)];
    const T fyp = L.cy[(uint32_t)i + (uint32_t)L.nx * ((uint32_t)(j + 1) + ny1 * k)];
    const T fym = L.cy[(uint32_t)i + (uint32_t)L.nx * ((uint32_t)j + ny1 * k)];
    const T fzp = L.cz[lidx(L, i, j, k + 1)];
    const T fzm = L.cz[lidx(L, i, j, k)];
    return rb_value_c(L, bv, fxp, fxm, fyp, fym, fzp, fzm, xp, xm, yp, ym, zp, zm, self);
}


// one colour of the red-black Gauss-Seidel sweep (_rbgs_body!, src/Multigrid.jl:307-337):
// colour c updates the cells with (i + j + k + c) even in 0-based interior
// indices (the reference's i = 2ih + ((j + k + c) & 1) in unit-halo storage).
// SMODE folds a pending mean removal φ ← φ − m (m = mptr[0], shift_kernel's
// values) into a sweep's two passes: 1, the first, reads every φ less m (its
// neighbours are the other colour, not written in this pass); 2, the second,
// whose neighbours the first wrote in the shifted frame, takes only its own
// old value less m (a blocked cell keeps it, a mirror boundary makes it its
// own neighbour); 3 is the first pass from φ = 0 (reads no φ; the pair's
// other cell is written zero). bm: b is read less bm[0] (a pending mean of b)
template <typename T, int SMODE>
__global__ void rbgs_kernel(LevelD<T> L, int colour, const double *__restrict__ mptr, const double *__restrict__ bm) {
    constexpr bool Z = SMODE == 3;
    int bxi, j, k;
    xcd_block3(bxi, j, k);
    const int ih = bxi * blockDim.x + threadIdx.x;
    const int par = (j + k + colour) & 1;
    const int i = 2 * ih + par;
    if constexpr (Z) {  // the other cell of the pair (2ih, 2ih + 1): of the other colour, zero
        const int io = 2 * ih + 1 - par;
        if (ih < (L.nx + 1) / 2 && io < L.nx) L.phi[lidx(L, io, j, k)] = T(0);
    }
    if (ih >= (L.nx + 1) / 2 || i >= L.nx) return;
    const T *f = L.phi;
    const T ms = (SMODE == 1 || SMODE == 2) ? (T)mptr[0] : T(0);
    const uint32_t cs = lidx(L, i, j, k);
    auto nb = [&](uint32_t cn) -> T {
        if constexpr (Z) return T(0);
        return (SMODE == 1 || (SMODE == 2 && cn == cs)) ? f[cn] - ms : f[cn];
    };
    const T xp = nb(lidx(L, wrapc(i + 1, L.nx, L.bcx), j, k)), xm = nb(lidx(L, wrapc(i - 1, L.nx, L.bcx), j, k));
    const T yp = nb(lidx(L, i, wrapc(j + 1, L.ny, L.bcy), k)), ym = nb(lidx(L, i, wrapc(j - 1, L.ny, L.bcy), k));
    const T zp = nb(lidx(L, i, j, wrapc(k + 1, L.nz, L.bcz))), zm = nb(lidx(L, i, j, wrapc(k - 1, L.nz, L.bcz)));
    const T self = Z ? T(0) : (SMODE != 0 ? f[cs] - ms : f[cs]);
    const T bv = bm ? L.b[cs] - (T)bm[0] : L.b[cs];
    L.phi[cs] = rb_value(L, i, j, k, xp, xm, yp, ym, zp, zm, self, bv);
}

// The terrain grid's finest-level face coefficients along a thread's column
// over a chunk of levels [k0, k1) (FP64; FP32 for the FP32 V-cycle): ρJ_x on the column's west and east
// faces and ρJ_y on its south and north faces at the cell levels, ρJG^σσ on
// its σ-faces k0 … k1 (tfw_mgcoef_kernel's expressions at the storage indices
// (i + H, j + H, k + H)), each times 1/Δ² of its axis. ρ̄ = ρ0 exp(−z/H_s) is
// evaluated by exp at the chunk's first level (and at the σ-face k1, the next
// chunk's first), and a face's coefficient is carried upwards by ρ̄'s ratio
// between levels, exp(−Δz J_f/H_s): a product per face and level in place of
// an exp, with the level-independent factors folded into the carried value.
// The chunks are the same for all columns, both colours and the residual, so
// the two cells of a face form the same products (a red-black pass steps two
// levels at once: the same to rounding). Over at most 32 levels the FP64 values
// are within 64 ulp of the stored arrays' (which still build the coarser
// levels): a level adds the product's rounding and the ratio's own (at most 32
// ulp in 1e5 random columns).
template <typename T>
struct TFChain {
    T g2, iJJ, t, dz;              // σ_x² + σ_y² over (H − σ)², 1/J²; H − σ at the current lower σ-face
    T xm, xp, ym, yp, z, z1;       // the carried values at the current level (z: its lower σ-face); z1: σ-face k1
    T qxm, qxp, qym, qyp, qz;      // their ratio between consecutive levels
    __device__ __forceinline__ void init(const TFM<T> &gm, const LevelD<T> &L, int I, int J, int K0, int K1) {
        const T Jxm = gm.Jx(I, J), Jxp = gm.Jx(I + 1, J), Jym = gm.Jy(I, J), Jyp = gm.Jy(I, J + 1);
        const T hc = gm.hp(I, J), Jc = gm.J(I, J);
        const T den = gm.Hl - hc, ax = (T)gm.hx[I + gm.sx * J] / den, ay = (T)gm.hy[I + gm.sx * J] / den;
        g2 = ax * ax + ay * ay;
        iJJ = 1 / (Jc * Jc);
        auto ratio = [&](T Jf) {
            if constexpr (sizeof(T) == 4) return __expf(-(gm.dz * Jf) * gm.iHs);
            else return exp(-(gm.dz * Jf) * gm.iHs);
        };
        const T sc = gm.sigc(K0);
        xm = gm.rho(gm.hxf(I, J) + sc * Jxm) * Jxm * L.ix2;
        xp = gm.rho(gm.hxf(I + 1, J) + sc * Jxp) * Jxp * L.ix2;
        ym = gm.rho(gm.hyf(I, J) + sc * Jym) * Jym * L.iy2;
        yp = gm.rho(gm.hyf(I, J + 1) + sc * Jyp) * Jyp * L.iy2;
        z = gm.rho(hc + gm.sigf(K0) * Jc) * Jc * L.iz2;
        z1 = gm.rho(hc + gm.sigf(K1) * Jc) * Jc * L.iz2;
        t = gm.Hl - gm.sigf(K0);
        dz = gm.dz;
        qxm = ratio(Jxm); qxp = ratio(Jxp); qym = ratio(Jym); qyp = ratio(Jyp); qz = ratio(Jc);
    }
    __device__ __forceinline__ void step() { xm *= qxm; xp *= qxp; ym *= qym; yp *= qyp; z *= qz; t -= dz; }
    // ρJG^σσ = ρ̄ J ((σ_x² + σ_y²) + 1/J²), σ_x = −(H − σ) h_x/(H − h), on the current level k's σ-faces
    // (the upper one of the chunk's last level by exp)
    static __device__ __forceinline__ T ma(T a, T b, T c) {
        if constexpr (sizeof(T) == 4) return __builtin_fmaf(a, b, c);
        else return __builtin_fma(a, b, c);
    }
    __device__ __forceinline__ T lower() const { return z * ma(t * t, g2, iJJ); }
    __device__ __forceinline__ T upper(int k, int k1, T qup) const {
        const T tu = t - dz;
        return (k + 1 < k1 ? z * qup : z1) * ma(tu * tu, g2, iJJ);
    }
    // a colour's march, every other level: from here step() takes two levels
    __device__ __forceinline__ void col(const TFM<T> &gm, const LevelD<T> &L, const double *, int i, int j, int k0, int k1) {
        init(gm, L, i + gm.H, j + gm.H, k0 + gm.H, k1 + gm.H);
    }
    __device__ __forceinline__ void skip() { step(); }  // up one level, before two()
    T q1, d1;                                           // z's ratio and t's step of one level
    __device__ __forceinline__ void two() {
        q1 = qz; d1 = dz;
        qxm *= qxm; qxp *= qxp; qym *= qym; qyp *= qyp; qz *= qz;
        dz += dz;
    }
    __device__ __forceinline__ T cxm() const { return xm; }
    __device__ __forceinline__ T cxp() const { return xp; }
    __device__ __forceinline__ T cym() const { return ym; }
    __device__ __forceinline__ T cyp() const { return yp; }
    // the lower and upper σ-face's coefficients of level k
    __device__ __forceinline__ void zfaces(int k, int k1, T &lo, T &up) {
        lo = lower();
        const T tu = t - d1;
        up = (k + 1 < k1 ? z * q1 : z1) * ma(tu * tu, g2, iJJ);
    }
};

// The same for the level below the finest (FP64): a coarse face's coefficient
// is the mean of its four fine faces' (restrict_coeff). On a lateral face
// these are two levels of two fine columns, so the sum over the levels is each
// column's lower value times 1 + ratio, carried by the ratio's square; a
// σ-face takes four fine columns at one fine level, each with its share
// of (H − σ)² and of 1. The values at each chunk's first level and the ratios
// are kept in a table (tf_table_kernel), read once per chunk, since the 24 exps
// of a thread cost as much as half its cells (128×68×44: 12.6 us a pass with
// the exps, 7.8 from the table).
constexpr int TFC_Q = 8, TFC_V = 12;  // planes of ratios, of values per chunk
constexpr size_t TFC_MIN = 3 << 19;   // least cells of the level (mg_set_terrain_coef)
struct TFChain2 {
    double x[4], y[4], qx[4], qy[4];  // west, west, east, east; south, south, north, north
    double zg[4], zi[4], qz[4], t, dz;                // t: H − σ at the current lower σ-face
    __device__ __forceinline__ void col(const TFM<double> &gm, const LevelD<double> &L, const double *tab, int i, int j, int k0, int) {
        // the planes, each (nx + 1) × (ny + 1)
        const uint32_t w = (uint32_t)L.nx + 1, n = w * ((uint32_t)L.ny + 1), c = (uint32_t)i + w * (uint32_t)j;
        const double *v = tab + (size_t)n * (TFC_Q + TFC_V * blockIdx.z);
#pragma unroll
        for (int o = 0; o < 2; o++) {
            x[o] = v[o * n + c]; x[2 + o] = v[o * n + c + 1];
            y[o] = v[(2 + o) * n + c]; y[2 + o] = v[(2 + o) * n + c + w];
            qx[o] = tab[o * n + c]; qx[2 + o] = tab[o * n + c + 1];
            qy[o] = tab[(2 + o) * n + c]; qy[2 + o] = tab[(2 + o) * n + c + w];
        }
#pragma unroll
        for (int o = 0; o < 4; o++) {
            qz[o] = tab[(4 + o) * n + c];
            zg[o] = v[(4 + o) * n + c];
            zi[o] = v[(8 + o) * n + c];
        }
        dz = 2.0 * gm.dz;
        t = gm.Hl - k0 * dz;
    }
    __device__ __forceinline__ double zf() const {
        return __builtin_fma(t * t, (zg[0] + zg[1]) + (zg[2] + zg[3]), (zi[0] + zi[1]) + (zi[2] + zi[3]));
    }
    // σ's part goes up with each face taken, two a cell
    __device__ __forceinline__ void zfaces(int, int, double &lo, double &up) {
        lo = zf();
        zstep();
        up = zf();
        zstep();
    }
    __device__ __forceinline__ void zstep() {
#pragma unroll
        for (int c = 0; c < 4; c++) { zg[c] *= qz[c]; zi[c] *= qz[c]; }
        t -= dz;
    }
    __device__ __forceinline__ void step() {
#pragma unroll
        for (int c = 0; c < 4; c++) { x[c] *= qx[c]; y[c] *= qy[c]; }
    }
    __device__ __forceinline__ void skip() { step(); zstep(); }
    __device__ __forceinline__ void two() {
#pragma unroll
        for (int c = 0; c < 4; c++) { qx[c] *= qx[c]; qy[c] *= qy[c]; }
    }
    __device__ __forceinline__ double cxm() const { return x[0] + x[1]; }
    __device__ __forceinline__ double cxp() const { return x[2] + x[3]; }
    __device__ __forceinline__ double cym() const { return y[0] + y[1]; }
    __device__ __forceinline__ double cyp() const { return y[2] + y[3]; }
};

// TFChain2's table: thread (i, j) of (nx + 1) × (ny + 1), chunk blockIdx.z
__global__ void tf_table_kernel(double *__restrict__ tab, TFM<double> gm, int nx, int ny, int kc, double ix2, double iy2,
                                double iz2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
    if (i > nx) return;
    const uint32_t w = (uint32_t)nx + 1, n = w * ((uint32_t)ny + 1), c = (uint32_t)i + w * (uint32_t)j;
    double *v = tab + (size_t)n * (TFC_Q + TFC_V * blockIdx.z);
    const int I = 2 * i + gm.H, J = 2 * j + gm.H, K = 2 * kc * (int)blockIdx.z + gm.H;
    const double sc = gm.sigc(K);
    for (int o = 0; o < 2; o++) {
        // (the last column and row have no faces beyond their first)
        const int jo = j < ny ? J + o : J, io = i < nx ? I + o : I;
        const double Jx = gm.Jx(I, jo), Jy = gm.Jy(io, J);
        const double rx = exp(-(gm.dz * Jx) * gm.iHs), ry = exp(-(gm.dz * Jy) * gm.iHs);
        v[o * n + c] = gm.rho(gm.hxf(I, jo) + sc * Jx) * Jx * (1.0 + rx) * (0.25 * ix2);
        v[(2 + o) * n + c] = gm.rho(gm.hyf(io, J) + sc * Jy) * Jy * (1.0 + ry) * (0.25 * iy2);
        tab[o * n + c] = rx * rx;
        tab[(2 + o) * n + c] = ry * ry;
    }
    for (int o = 0; o < 4; o++) {
        const int a = i < nx ? I + (o & 1) : I, b = j < ny ? J + (o >> 1) : J;
        const double hc = gm.hp(a, b), Jc = gm.J(a, b), den = gm.Hl - hc;
        const double ax = gm.hx[a + gm.sx * b] / den, ay = gm.hy[a + gm.sx * b] / den;
        const double z = gm.rho(hc + gm.sigf(K) * Jc) * Jc * (0.25 * iz2);
        v[(4 + o) * n + c] = z * (ax * ax + ay * ay);
        v[(8 + o) * n + c] = z / (Jc * Jc);
        tab[(4 + o) * n + c] = exp(-2.0 * (gm.dz * Jc) * gm.iHs);
    }
}

// One colour of the red-black sweep on the terrain grid's finest level
// (FP64), with the face coefficients evaluated from the Gal-Chen metrics
// (TFChain) instead of read from the stored arrays. Thread (i, j) marches its
// column over a chunk of levels, updating the colour's cells (every other
// level) and carrying the z-neighbour shared by consecutive cells. φ and b
// are colour-split (SplitMap), so a pass reads the other colour's half of φ
// and its own half of b and writes its own half of φ: 3 × 4 bytes per cell.
// A cell's own old value is read only where the diagonal vanishes.
// FROM0, a cycle's first pass (colour 0): φ is zero, so no φ is read and
// b/diag written; the other colour's half is not needed before the next pass
// has written it, except where a mirror boundary makes a cell its own
// neighbour, and there that pass takes zero (first).
// SUM, a cycle's last pass: the block sums of b·φ, φ and b (what the CG needs
// of z = φ), of the updated cells and of the other colour's, whose φ the pass
// reads as z-neighbours.
// Measured at 512×512×256: 257 us and 1.22 GB per pass with every cell's old
// value read → 221 us and 1.01 GB (4.6 TB/s; 0.81 GB is the least, the rest
// the neighbouring strips' lines). It is bound by memory: half the VALU work
// per cell, the next cell's loads issued ahead, 4 rows or 64 levels per block
// all stay within 2 %; blocks in XCD-contiguous rows are 5 % slower. From
// zero 170 → 108 us. The pass with the three sums 261 us, where a mean pass
// (100 us) and a pass over φ and r (183 us) read them before.
constexpr int RBC_BY = 2;   // rows per block
constexpr int RBC_KC = 32;  // most levels per chunk
constexpr int RBC_FILL = 2048;  // blocks a round (chunk_levels); 96×96×48 step 22.1 ms with 32 levels, 18.8 to 19.2 with 1024 or 2048 blocks
template <bool FROM0, bool SUM, class CH>
__global__ void __launch_bounds__(64 * RBC_BY) rbgs_tf_kernel(LevelD<double> L, TFM<double> gm,
                                                              const double *__restrict__ tab, int colour, int kc,
                                                              int first, double *__restrict__ partials, int npb,
                                                              uint32_t half) {
    static_assert(!(FROM0 && SUM), "the from-zero pass is a sweep's first");
    const int i0 = blockIdx.x * 64 + threadIdx.x, j0 = blockIdx.y * RBC_BY + threadIdx.y;
    const bool ok = i0 < L.nx && j0 < L.ny;
    if (!SUM && !ok) return;
    const int i = ok ? i0 : 0, j = ok ? j0 : 0;
    const int k0 = blockIdx.z * kc, k1 = min(k0 + kc, L.nz);
    double srz = 0.0, sz = 0.0, sr = 0.0;
    CH q;
    q.col(gm, L, tab, i, j, k0, k1);
    const double *f = L.phi;
    // a neighbour cn of cell cs (cn == cs: a mirror boundary)
    auto nb = [&](uint32_t cn, uint32_t cs) {
        if constexpr (FROM0) return 0.0;
        return first && cn == cs ? 0.0 : f[cn];
    };
    const int ixp = wrapc(i + 1, L.nx, L.bcx), ixm = wrapc(i - 1, L.nx, L.bcx);
    const int jyp = wrapc(j + 1, L.ny, L.bcy), jym = wrapc(j - 1, L.ny, L.bcy);
    auto pi = [&](int ii, int jj, int kk) { return split_at(half, ii, jj, kk, lidx(L, ii, jj, kk)); };  // the index of φ and b
    int k = k0 + ((i + j + k0 + colour) & 1);
    if (k > k0) q.skip();
    double zm = 0.0;
    if (ok && k < k1) {
        const uint32_t cb = pi(i, j, wrapc(k - 1, L.nz, L.bcz));
        zm = nb(cb, pi(i, j, k));
        if (SUM && k - 1 >= k0) {  // the chunk's first level, of the other colour
            const double bo = L.b[cb];
            srz += bo * zm; sz += zm; sr += bo;
        }
    } else if (SUM && ok) {  // a chunk with none of this colour (one level)
        for (int kk = k0; kk < k1; kk++) {
            const uint32_t co = pi(i, j, kk);
            const double bo = L.b[co], vo = f[co];
            srz += bo * vo; sz += vo; sr += bo;
        }
    }
    // the column's index offsets, in either layout: a neighbour on the cell's
    // level is the cell's index plus a constant of the column, the level
    // above inside the grid likewise, the next cell of the colour two levels
    // up too (in the split layout the lateral and vertical neighbours lie in
    // the other colour's half, dbase away; nx even)
    const uint32_t nxy = (uint32_t)L.nx * (uint32_t)L.ny;
    const bool spl = half != 0;
    const uint32_t dbase = spl ? (colour ? 0u - half : half) : 0u;
    auto lat = [&](int ni, int nj) -> uint32_t {
        const int d = (ni - i) + (nj - j) * L.nx;
        if (!spl) return (uint32_t)d;
        return (uint32_t)(((i & 1) + d) >> 1) + ((((ni - i) + (nj - j)) & 1) ? dbase : 0u);
    };
    const uint32_t oxp = lat(ixp, j), oxm = lat(ixm, j), oyp = lat(i, jyp), oym = lat(i, jym);
    const uint32_t ozp = spl ? dbase + (nxy >> 1) : nxy, sstep = spl ? nxy : 2 * nxy;
    uint32_t cs = pi(i, j, k);  // the cell's index
    q.two();
    for (; ok && k < k1; k += 2, cs += sstep) {
        const double xp = nb(cs + oxp, cs), xm = nb(cs + oxm, cs);
        const double yp = nb(cs + oyp, cs), ym = nb(cs + oym, cs);
        const uint32_t cu = k + 1 < L.nz ? cs + ozp : pi(i, j, wrapc(k + 1, L.nz, L.bcz));
        const double zp = nb(cu, cs);
        double fzm, fzp;
        q.zfaces(k, k1, fzm, fzp);
        const double fxm = q.cxm(), fxp = q.cxp(), fym = q.cym(), fyp = q.cyp();
        const double bv = L.b[cs];
        const double diag = ((fxp + fxm) + (fyp + fym)) + (fzp + fzm);  // −diag of A
        double vnew;
        if (diag < Eps<double>::v) {
            vnew = FROM0 || first ? 0.0 : f[cs];
        } else {
            const double ox = __builtin_fma(fxp, xp, fxm * xm), oy = __builtin_fma(fyp, yp, fym * ym);
            const double oz = __builtin_fma(fzp, zp, __builtin_fma(fzm, zm, -bv));
            vnew = qdiv<double>((ox + oy) + oz, diag);
        }
        L.phi[cs] = vnew;
        if (SUM) {
            srz += bv * vnew; sz += vnew; sr += bv;
            if (k + 1 < k1) {  // the level above, of the other colour, in the chunk
                const double bo = L.b[cu];
                srz += bo * zp; sz += zp; sr += bo;
            }
        }
        zm = zp;  // the next cell's lower neighbour (k + 1, not updated in this colour)
        q.step();
    }
    if constexpr (SUM) {
        __shared__ double sh[RBC_BY][3];
        for (int off = 32; off > 0; off >>= 1) {
            srz += __shfl_down(srz, off, 64);
            sz += __shfl_down(sz, off, 64);
            sr += __shfl_down(sr, off, 64);
        }
        if (threadIdx.x == 0) { sh[threadIdx.y][0] = srz; sh[threadIdx.y][1] = sz; sh[threadIdx.y][2] = sr; }
        __syncthreads();
        if (threadIdx.x < 3 && threadIdx.y == 0) {
            double t = 0.0;
            for (int w = 0; w < RBC_BY; w++) t += sh[w][threadIdx.x];
            partials[threadIdx.x * npb + blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)] = t;
        }
    }
}

// The residual of the terrain grid's finest level restricted to the coarse
// right-hand side (the mean of the 8 fine values), after a smoothing whose
// last pass updated colour 1: those cells' equations then hold, so only the
// colour-0 cells' residuals (4 of a coarse cell's 8) are formed, and r is
// never stored. A cell with a mirror boundary is the exception, since its
// update took its own old value for the missing neighbour: the colour-1 cells
// of the bottom and top level are formed too (the lateral axes are periodic).
// A wave is 32 pairs of columns (2I, 2I + 1) × the two rows of a coarse cell;
// a thread marches its pair of columns over a chunk of levels, in column A on
// the chunk's even levels and in B on the odd ones (each the colour-0 cell of
// its level), with a TFChain of each column. Of a pair, the split layout has
// both colours at one index, so the colour-1 value of the pair on levels
// k − 1, k, k + 1 is the lower neighbour, the x neighbour inside the pair and
// the upper neighbour: per level it loads six values. The rows' and levels'
// sums meet in a lane exchange.
// With partials, the block sums of the coarse values (for their mean).
// Bound: memory, φ and half of b read, 13 B per fine cell. At 512×512×256:
// residual 470 us + restriction 111 us → 210 us.
constexpr int RRC_BW = 4;  // waves per block
__global__ void __launch_bounds__(64 * RRC_BW) residual_restrict_tf_kernel(LevelD<double> L, LevelD<double> C,
                                                                           TFM<double> gm, int kc,
                                                                           double *__restrict__ partials,
                                                                           uint32_t half, uint32_t halfc) {
    __shared__ double sh[RRC_BW];
    const int lane = threadIdx.x, wv = threadIdx.y;
    const int ci = blockIdx.x * 32 + (lane & 31), cj = blockIdx.y * RRC_BW + wv;
    const bool ok = ci < C.nx && cj < C.ny;
    const int pr = ok ? ci : 0, j = ok ? 2 * cj + (lane >> 5) : 0;
    const int k0 = blockIdx.z * kc, k1 = min(k0 + kc, L.nz);  // even
    const uint32_t hx = (uint32_t)L.nx >> 1, pl = hx * (uint32_t)L.ny;  // pairs per row, per level
    const int sA = j & 1;                                               // column A is 2·pr + sA (k0 even)
    const int iA = 2 * pr + sA, iB = 2 * pr + 1 - sA;
    TFChain<double> A, B;
    A.init(gm, L, iA + gm.H, j + gm.H, k0 + gm.H, k1 + gm.H);
    B.init(gm, L, iB + gm.H, j + gm.H, k0 + gm.H, k1 + gm.H);
    // "xp" of a chain: the face towards the pair's other column
    auto swapx = [](TFChain<double> &q) {
        const double a = q.xm, c = q.qxm;
        q.xm = q.xp; q.qxm = q.qxp;
        q.xp = a; q.qxp = c;
    };
    if (sA) swapx(A); else swapx(B);
    const int left = wrapc(2 * pr - 1, L.nx, L.bcx) >> 1, right = wrapc(2 * pr + 2, L.nx, L.bcx) >> 1;
    const uint32_t oA = sA ? right : left, oB = sA ? left : right;  // the pair beyond the outer x face
    const uint32_t jp = wrapc(j + 1, L.ny, L.bcy), jm = wrapc(j - 1, L.ny, L.bcy);
    const double *f0 = L.phi, *f1 = L.phi + half, *b0 = L.b, *b1 = L.b + half;
    // b − A φ of a cell of level k: its value c, the pair's other value xi, the
    // outer x value xo, the y values, the z values
    auto res = [&](const TFChain<double> &q, int k, double bv, double c, double xi, double xo, double yp, double ym,
                   double zp, double zm) {
        const double fzp = q.upper(k, k1, q.qz), fzm = q.lower();
        const double ax = __builtin_fma(q.xp, xi - c, q.xm * (xo - c)), ay = __builtin_fma(q.yp, yp - c, q.ym * (ym - c));
        const double az = __builtin_fma(fzp, zp - c, __builtin_fma(fzm, zm - c, -bv));
        return -((ax + ay) + az);
    };
    const uint32_t row = hx * (uint32_t)j, rowp = hx * jp, rowm = hx * jm;
    uint32_t base = pl * (uint32_t)k0;
    // the pair's colour-1 value below, on and above the level (mirrored ends: unused)
    double m0 = k0 > 0 ? f1[base - pl + row + pr] : (L.bcz == BC_PERIODIC ? f1[pl * (uint32_t)(L.nz - 1) + row + pr] : 0.0);
    double m1 = f1[base + row + pr];
    double cprev = 0.0, total = 0.0;
    for (int k = k0; k < k1; k += 2) {
        double r = 0.0;
        auto level = [&](const TFChain<double> &q, const TFChain<double> &qo, uint32_t outer, uint32_t outer1, int kk) {
            const uint32_t s = base + row + pr;
            const double c = f0[s], bv = b0[s];
            const bool top = kk + 1 == L.nz, per = L.bcz == BC_PERIODIC;
            const double m2 = !top ? f1[s + pl] : (per ? f1[row + pr] : c);
            const double xo = f1[base + row + outer];
            const double yp = f1[base + rowp + pr], ym = f1[base + rowm + pr];
            const bool bottom = kk == 0 && !per;
            r += res(q, kk, bv, c, m1, xo, yp, ym, m2, bottom ? c : m0);
            if (!per && (kk == 0 || top)) {
                // the pair's colour-1 cell on a mirror boundary
                const double xo1 = f0[base + row + outer1], yp1 = f0[base + rowp + pr], ym1 = f0[base + rowm + pr];
                const double up = top ? m1 : f0[s + pl], dn = kk == 0 ? m1 : cprev;
                r += res(qo, kk, b1[s], m1, c, xo1, yp1, ym1, up, dn);
            }
            m0 = m1;
            m1 = m2;
            cprev = c;
            base += pl;
        };
        if (ok) level(A, B, oA, oB, k);
        A.step();
        B.step();
        if (ok) level(B, A, oB, oA, k + 1);
        A.step();
        B.step();
        r += __shfl_xor(r, 32, 64);
        const double bc = r * 0.125;
        if (ok && lane < 32) {
            C.b[split_at(halfc, ci, cj, k >> 1, lidx(C, ci, cj, k >> 1))] = bc;
            total += bc;
        }
    }
    if (partials) {
        for (int off = 16; off > 0; off >>= 1) total += __shfl_down(total, off, 64);
        if (lane == 0) sh[wv] = total;
        __syncthreads();
        if (lane == 0 && wv == 0) {
            double t = 0.0;
            for (int w = 0; w < RRC_BW; w++) t += sh[w];
            partials[blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)] = t;
        }
    }
}

// φ += the trilinear correction (prolong_kernel's weights) on the terrain
// grid's finest level, before a smoothing whose first pass updates colour 0:
// that pass reads no colour-0 value, so only the colour-1 cells are
// corrected. On a mirror boundary a cell is its own neighbour: both colours
// of the bottom and top level are corrected.
// A thread marches a pair of columns; its row's parity is the wave's, so
// which column holds colour 1 on a level is uniform. The x-y part of the
// weights is summed once per coarse level, for the pair's left and right
// column, and kept for three coarse levels.
// both: no smoothing follows, and every cell is corrected.
// Bound: memory, half of φ read and written, 9 B per fine cell. At
// 512×512×256: 258 us (both colours, one column per thread) → 155 us (142
// before the coarse φ was colour-split).
constexpr int PRC_BY = 4;   // rows per block
constexpr int PRC_KC = 16;  // most fine levels per chunk (even)
constexpr int PRC_FILL = 1024;  // blocks a round (chunk_levels)
__global__ void __launch_bounds__(64 * PRC_BY) prolong_tf_kernel(LevelD<double> F, LevelD<double> C, int kc,
                                                                 uint32_t half, uint32_t halfc, int both) {
    const int pr = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * PRC_BY + __builtin_amdgcn_readfirstlane(threadIdx.y);
    if (pr >= C.nx || j >= F.ny) return;
    const int k0 = blockIdx.z * kc, k1 = min(k0 + kc, F.nz);
    const int xl = wrapc(pr - 1, C.nx, C.bcx), xr = wrapc(pr + 1, C.nx, C.bcx);
    const int J = j >> 1, jy = wrapc(J + ((j & 1) ? 1 : -1), C.ny, C.bcy);
    // the x-y sums of coarse level m for the pair's columns 2·pr (l) and 2·pr + 1 (r)
    auto plane = [&](int m, double &l, double &r) {
        const int mm = wrapc(m, C.nz, C.bcz);
        auto at = [&](int i, int jc) { return C.phi[split_at(halfc, i, jc, mm, lidx(C, i, jc, mm))]; };
        const double near = 0.75 * at(pr, J) + 0.25 * at(pr, jy);
        const double nl = 0.75 * at(xl, J) + 0.25 * at(xl, jy), nr = 0.75 * at(xr, J) + 0.25 * at(xr, jy);
        l = 0.75 * near + 0.25 * nl;
        r = 0.75 * near + 0.25 * nr;
    };
    double l0, r0, l1, r1, l2, r2;
    plane((k0 >> 1) - 1, l0, r0);
    plane(k0 >> 1, l1, r1);
    const uint32_t hx = (uint32_t)F.nx >> 1, pl = hx * (uint32_t)F.ny;
    uint32_t s = hx * (uint32_t)j + pr + pl * (uint32_t)k0;
    double *f0 = F.phi, *f1 = F.phi + half;
    const bool mirror = F.bcz != BC_PERIODIC;
    const int odd = j & 1;  // on an even level colour 1 is the pair's right column in an even row
    for (int k = k0; k < k1; k += 2) {
        plane((k >> 1) + 1, l2, r2);
        const double le = 0.75 * l1 + 0.25 * l0, re = 0.75 * r1 + 0.25 * r0;
        const double lo = 0.75 * l1 + 0.25 * l2, ro = 0.75 * r1 + 0.25 * r2;
        f1[s] += odd ? le : re;
        if (both || (mirror && k == 0)) f0[s] += odd ? re : le;
        f1[s + pl] += odd ? ro : lo;
        if (both || (mirror && k + 2 == F.nz)) f0[s + pl] += odd ? lo : ro;
        s += 2 * pl;
        l0 = l1; r0 = r1; l1 = l2; r1 = r2;
    }
}


// damped Jacobi from `src` into `dst`: φ ← φ + ω (b − Aφ)/diag (a fully blocked cell keeps φ)
// (src null: φ = 0, the first sweep of a cycle from zero: ω b/diag, the
// same arithmetic as 0 + ω (b − A0)/diag without reading or clearing φ)
template <typename T>
__global__ void jacobi_kernel(LevelD<T> L, const T *__restrict__ src, T *__restrict__ dst, T omega) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y, k = blockIdx.z;
    if (i >= L.nx) return;
    const uint32_t c = lidx(L, i, j, k);
    const T d = diagA(L, i, j, k);
    const T x = src ? src[c] : T(0);
    if (fabs(d) < Eps<T>::v) { dst[c] = x; return; }
    const T r = src ? L.b[c] - applyA(L, src, i, j, k) : L.b[c];
    dst[c] = x + omega * (r / d);
}

// The FP32 V-cycle's finest level on the terrain grid: damped Jacobi
// (jacobi_kernel's arithmetic) and the residual (residual_kernel's, without
// the block sums) with the face coefficients evaluated in FP32 from the
// Gal-Chen metrics (TFChain<float>: ρ̄ by __expf at a chunk's first level
// and carried up by its FP32 ratio between levels, the column's 1/(H − h)
// once, the update's division by v_rcp_f32) instead of read: φ, b and the
// result per cell, no coefficient arrays. The values are an FP32
// evaluation, not the FP64 coefficients rounded, so the preconditioner
// differs from the stored-array one at FP32 rounding; every face is
// evaluated by one sequence of operations wherever it is needed, so the
// operator stays symmetric. A thread marches its column over a chunk of
// levels; its bottom face is the level below's top face (carried).
// (the fast form's step on one box: 4 rows × 32 levels 114.0 ms, × 16 115.0;
// 2 × 32 115.8, 2 × 16 115.4; FP32 ρ̄ carried over 32 levels)
constexpr int JTF_BY = 4;   // rows per block
constexpr int JTF_KC = 32;  // levels per chunk

// MODE 0: dst = src + ω (b − A src)/diag (src null: the zero start); MODE 1: dst = b − A src
template <int MODE>
__global__ void __launch_bounds__(64 * JTF_BY) jacobi_tf_kernel(LevelD<float> L, TFM<float> gm,
                                                                 const float *__restrict__ src, float *__restrict__ dst,
                                                                 float omega, int kc) {
    const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * JTF_BY + threadIdx.y;
    const bool ok = i < L.nx && j < L.ny;
    const int k0 = blockIdx.z * kc, k1 = min(k0 + kc, L.nz);
    const int ic = ok ? i : 0, jc = ok ? j : 0;
    const int I = ic + gm.H, J = jc + gm.H;
    TFChain<float> q;
    q.init(gm, L, I, J, k0 + gm.H, k1 + gm.H);
    const uint32_t ixp = wrapc(ic + 1, L.nx, L.bcx), ixm = wrapc(ic - 1, L.nx, L.bcx);
    const uint32_t jyp = wrapc(jc + 1, L.ny, L.bcy), jym = wrapc(jc - 1, L.ny, L.bcy);
    float fzm = q.lower();
    float c = 0.f, zm = 0.f;
    if (src && ok) {
        c = src[lidx(L, ic, jc, k0)];
        zm = src[lidx(L, ic, jc, wrapc(k0 - 1, L.nz, L.bcz))];
    }
    for (int k = k0; k < k1; k++) {
        const float fzp = q.upper(k, k1, q.qz);
        float zp = 0.f;
        if (src && ok) zp = src[lidx(L, ic, jc, wrapc(k + 1, L.nz, L.bcz))];
        if (ok) {
            const uint32_t cc = lidx(L, i, j, k);
            float Ax = 0.f;
            if (src) {
                const float xp = src[lidx(L, ixp, j, k)], xm = src[lidx(L, ixm, j, k)];
                const float yp = src[lidx(L, i, jyp, k)], ym = src[lidx(L, i, jym, k)];
                Ax = (__builtin_fmaf(q.xp, xp - c, q.xm * (xm - c)) + __builtin_fmaf(q.yp, yp - c, q.ym * (ym - c))) +
                     __builtin_fmaf(fzp, zp - c, fzm * (zm - c));
            }
            if constexpr (MODE == 1) {
                dst[cc] = L.b[cc] - Ax;
            } else {
                const float d = -(((q.xp + q.xm) + (q.yp + q.ym)) + (fzp + fzm));
                if (fabsf(d) < Eps<float>::v) {
                    dst[cc] = c;
                } else {
                    const float r = src ? L.b[cc] - Ax : L.b[cc];
                    dst[cc] = c + omega * qdiv<float>(r, d);
                }
            }
        }
        fzm = fzp;
        zm = c;
        c = zp;
        q.step();
    }
}

// r = b − Aφ (_res_body!, src/Multigrid.jl:266-269), with the block sums of r;
// with mptr φ is read less its pending mean, with bm b less its pending mean
template <typename T>
__global__ void residual_kernel(LevelD<T> L, double *__restrict__ partials, const double *__restrict__ mptr,
                                const double *__restrict__ bm) {
    __shared__ double sh[RB / 64];
    int bxi, j, k;
    xcd_block3(bxi, j, k);
    const int i = bxi * blockDim.x + threadIdx.x;
    double v = 0.0;
    if (i < L.nx) {
        const uint32_t c = lidx(L, i, j, k);
        const T bv = bm ? L.b[c] - (T)bm[0] : L.b[c];
        const T r = bv - (mptr ? applyA<T, true>(L, L.phi, i, j, k, (T)mptr[0]) : applyA(L, L.phi, i, j, k));
        L.r[c] = r;
        v = (double)r;
    }
    double s = block_sum(v, sh);
    if (threadIdx.x == 0) partials[blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)] = s;
}

// coarse b = the mean of the 8 fine (r − m) (_restrict_body!, src/Multigrid.jl:381-392), with block sums
template <typename T>
__global__ void restrict_kernel(LevelD<T> C, LevelD<T> F, const double *__restrict__ mptr, double *__restrict__ partials) {
    __shared__ double sh[RB / 64];
    const int I = blockIdx.x * blockDim.x + threadIdx.x;
    const int J = blockIdx.y, K = blockIdx.z;
    double v = 0.0;
    if (I < C.nx) {
        const T m = mptr ? (T)mptr[0] : T(0);
        const int i = 2 * I, j = 2 * J, k = 2 * K;
        const T *r = F.r;
        T s = (((((((r[lidx(F, i, j, k)] - m) + (r[lidx(F, i + 1, j, k)] - m)) + (r[lidx(F, i, j + 1, k)] - m)) +
                   (r[lidx(F, i + 1, j + 1, k)] - m)) + (r[lidx(F, i, j, k + 1)] - m)) +
                 (r[lidx(F, i + 1, j, k + 1)] - m)) + (r[lidx(F, i, j + 1, k + 1)] - m)) +
               (r[lidx(F, i + 1, j + 1, k + 1)] - m);
        T bval = s * T(1.0 / 8);
        C.b[lidx(C, I, J, K)] = bval;
        v = (double)bval;
    }
    double s = block_sum(v, sh);
    if (threadIdx.x == 0) partials[blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)] = s;
}

// coarse b = the mean of the 8 fine residuals, where the last smoothing pass
// updated colour 1 (the colour-1 equations then hold and only colour-0 cells
// are formed, as in residual_restrict_tf_kernel; a cell on a mirror boundary
// is formed whichever its colour), with the block sums of b when asked.
// One coarse cell per work item; r is not stored.
// SPL: the fine level is colour-split (with stored coefficients)
template <typename T, bool SPL = false>
__global__ void residual_restrict_kernel(LevelD<T> C, LevelD<T> F, double *__restrict__ partials, uint32_t half = 0) {
    __shared__ double sh[RB / 64];
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    double v = 0.0;
    if (t < (uint32_t)C.nx * (uint32_t)C.ny * (uint32_t)C.nz) {
        const uint32_t JK = t / (uint32_t)C.nx, I = t - JK * (uint32_t)C.nx, K = JK / (uint32_t)C.ny, J = JK - K * (uint32_t)C.ny;
        const bool mx = F.bcx != BC_PERIODIC, my = F.bcy != BC_PERIODIC, mz = F.bcz != BC_PERIODIC;
        T s = T(0);
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int i = 2 * I + (q & 1), j = 2 * J + ((q >> 1) & 1), k = 2 * K + (q >> 2);
            const bool even = (((q & 1) + ((q >> 1) & 1) + (q >> 2)) & 1) == 0;
            if (even || (mx && (i == 0 || i == F.nx - 1)) || (my && (j == 0 || j == F.ny - 1)) ||
                (mz && (k == 0 || k == F.nz - 1)))
            {
                if constexpr (SPL) {
                    auto at = [&](int a, int b, int c) { return split_at(half, a, b, c, lidx(F, a, b, c)); };
                    const uint32_t nx1 = F.nx + 1, ny1 = F.ny + 1, row = (uint32_t)j + (uint32_t)F.ny * k;
                    const T c = F.phi[at(i, j, k)];
                    const T dxp = F.phi[at(wrapc(i + 1, F.nx, F.bcx), j, k)] - c, dxm = F.phi[at(wrapc(i - 1, F.nx, F.bcx), j, k)] - c;
                    const T dyp = F.phi[at(i, wrapc(j + 1, F.ny, F.bcy), k)] - c, dym = F.phi[at(i, wrapc(j - 1, F.ny, F.bcy), k)] - c;
                    const T dzp = F.phi[at(i, j, wrapc(k + 1, F.nz, F.bcz))] - c, dzm = F.phi[at(i, j, wrapc(k - 1, F.nz, F.bcz))] - c;
                    const T *cx = F.cx + ((uint32_t)i + nx1 * row), *cy = F.cy + ((uint32_t)i + (uint32_t)F.nx * ((uint32_t)j + ny1 * k));
                    const T *cz = F.cz + lidx(F, i, j, k);
                    const T ax = (cx[1] * dxp + cx[0] * dxm) * F.ix2, ay = (cy[F.nx] * dyp + cy[0] * dym) * F.iy2;
                    const T az = (cz[(uint32_t)F.nx * (uint32_t)F.ny] * dzp + cz[0] * dzm) * F.iz2;
                    s += F.b[at(i, j, k)] - ((ax + ay) + az);
                } else {
                    s += F.b[lidx(F, i, j, k)] - applyA(F, F.phi, i, j, k);
                }
            }
        }
        const T bval = s * T(1.0 / 8);
        C.b[t] = bval;
        v = (double)bval;
    }
    if (partials) {
        const double sb = block_sum(v, sh);
        if (threadIdx.x == 0) partials[blockIdx.x] = sb;
    }
}

// coarse b = the mean of the 8 fine b, the residual of φ = 0, with its block
// sums when asked (FP64 terrain cycle without pre-smoothing; half, halfc: the
// levels' colour split, 0 natural)
__global__ void restrict_rhs_kernel(LevelD<double> C, LevelD<double> F, double *__restrict__ partials, uint32_t half,
                                    uint32_t halfc) {
    __shared__ double sh[RB / 64];
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    double v = 0.0;
    if (t < (uint32_t)C.nx * (uint32_t)C.ny * (uint32_t)C.nz) {
        const uint32_t JK = t / (uint32_t)C.nx, I = t - JK * (uint32_t)C.nx, K = JK / (uint32_t)C.ny, J = JK - K * (uint32_t)C.ny;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int i = 2 * I + (q & 1), j = 2 * J + ((q >> 1) & 1), k = 2 * K + (q >> 2);
            v += F.b[split_at(half, i, j, k, lidx(F, i, j, k))];
        }
        v *= 0.125;
        C.b[split_at(halfc, I, J, K, t)] = v;
    }
    if (partials) {
        const double sb = block_sum(v, sh);
        if (threadIdx.x == 0) partials[blockIdx.x] = sb;
    }
}

// φ += trilinear correction (_prolong_body!, src/Multigrid.jl:415-432), with block sums of φ
// with mcptr the coarse φ is read less its pending mean
template <typename T>
__global__ void prolong_kernel(LevelD<T> F, LevelD<T> C, double *__restrict__ partials, const double *__restrict__ mptr,
                               const double *__restrict__ mcptr) {
    __shared__ double sh[RB / 64];
    int bxi, j, k;
    xcd_block3(bxi, j, k);
    const int i = bxi * blockDim.x + threadIdx.x;
    double v = 0.0;
    if (i < F.nx) {
        // 1-based fine index i+1: coarse cell (i+1+1)>>1 (1-based) and the far neighbour
        const int Ih = (i >> 1), Ix = Ih + (((i + 1) & 1) ? -1 : 1);
        const int Jh = (j >> 1), Jy = Jh + (((j + 1) & 1) ? -1 : 1);
        const int Kh = (k >> 1), Kz = Kh + (((k + 1) & 1) ? -1 : 1);
        const int ix = wrapc(Ix, C.nx, C.bcx), jy = wrapc(Jy, C.ny, C.bcy), kz = wrapc(Kz, C.nz, C.bcz);
        const T n = T(3) / T(4), f = T(1) / T(4);
        const T mcv = mcptr ? (T)mcptr[0] : T(0);
        auto P = [&](uint32_t q) -> T { return mcptr ? C.phi[q] - mcv : C.phi[q]; };
        T acc = T(0);
        acc += (n * n * n) * P(lidx(C, Ih, Jh, Kh));
        acc += (f * n * n) * P(lidx(C, ix, Jh, Kh));
        acc += (n * f * n) * P(lidx(C, Ih, jy, Kh));
        acc += (f * f * n) * P(lidx(C, ix, jy, Kh));
        acc += (n * n * f) * P(lidx(C, Ih, Jh, kz));
        acc += (f * n * f) * P(lidx(C, ix, Jh, kz));
        acc += (n * f * f) * P(lidx(C, Ih, jy, kz));
        acc += (f * f * f) * P(lidx(C, ix, jy, kz));
        const uint32_t c = lidx(F, i, j, k);
        // with mptr, the fine φ first loses its mean (shift_kernel's value)
        const T val = (mptr ? F.phi[c] - (T)mptr[0] : F.phi[c]) + acc;
        F.phi[c] = val;
        v = (double)val;
    }
    double s = block_sum(v, sh);
    if (threadIdx.x == 0) partials[blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)] = s;
}

// prolong_kernel marching fine columns (the finest level, even extents):
// thread (i, j) walks a chunk of fine levels; the coarse values of its four
// coarse columns (Ih or its far neighbour × Jh or its far neighbour) over
// the coarse levels m − 1, m, m + 1 are kept in registers and shifted one
// coarse level per two fine levels, so each fine cell's eight coarse terms
// are summed in prolong_kernel's order from registers. The block sums of φ
// add each column's levels in order, then the block's columns.
template <typename T>
__global__ void __launch_bounds__(64 * PRC_BY) prolong_col_kernel(LevelD<T> F, LevelD<T> C, int kc,
                                                                  double *__restrict__ partials,
                                                                  const double *__restrict__ mptr,
                                                                  const double *__restrict__ mcptr) {
    __shared__ double sh[PRC_BY];
    const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * PRC_BY + threadIdx.y;
    const bool ok = i < F.nx && j < F.ny;
    const int k0 = blockIdx.z * kc, k1 = min(k0 + kc, F.nz);
    double sum = 0.0;
    if (ok) {
        const int Ih = i >> 1, ix = wrapc(Ih + (((i + 1) & 1) ? -1 : 1), C.nx, C.bcx);
        const int Jh = j >> 1, jy = wrapc(Jh + (((j + 1) & 1) ? -1 : 1), C.ny, C.bcy);
        const T n = T(3) / T(4), f = T(1) / T(4);
        const T *P = C.phi;
        const T m = mptr ? (T)mptr[0] : T(0);
        const T mcv = mcptr ? (T)mcptr[0] : T(0);  // the coarse φ's pending mean
        // w[q][s]: coarse column q (0: Ih Jh, 1: ix Jh, 2: Ih jy, 3: ix jy) at coarse level mc − 1 + s
        auto ld = [&](int q, int lev) -> T {
            const int kk = wrapc(lev, C.nz, C.bcz);
            const T v = P[lidx(C, (q & 1) ? ix : Ih, (q & 2) ? jy : Jh, kk)];
            return mcptr ? v - mcv : v;
        };
        int mc = k0 >> 1;
        T w[4][3];
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int s2 = 0; s2 < 3; s2++) w[q][s2] = ld(q, mc - 1 + s2);
        for (int k = k0; k < k1; k++) {
            // the far coarse level: below for an even fine level, above for an odd one
            const int far = (k & 1) ? 2 : 0;
            T acc = T(0);
            acc += (n * n * n) * w[0][1];
            acc += (f * n * n) * w[1][1];
            acc += (n * f * n) * w[2][1];
            acc += (f * f * n) * w[3][1];
            acc += (n * n * f) * (far ? w[0][2] : w[0][0]);
            acc += (f * n * f) * (far ? w[1][2] : w[1][0]);
            acc += (n * f * f) * (far ? w[2][2] : w[2][0]);
            acc += (f * f * f) * (far ? w[3][2] : w[3][0]);
            const uint32_t c = lidx(F, i, j, k);
            const T val = (mptr ? F.phi[c] - m : F.phi[c]) + acc;
            F.phi[c] = val;
            sum += (double)val;
            if ((k & 1) && k + 1 < k1) {  // the next coarse level
                mc++;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    w[q][0] = w[q][1];
                    w[q][1] = w[q][2];
                    w[q][2] = ld(q, mc + 1);
                }
            }
        }
    }
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
    if (threadIdx.x == 0) sh[threadIdx.y] = sum;
    __syncthreads();
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        double t = 0.0;
        for (int q = 0; q < PRC_BY; q++) t += sh[q];
        partials[blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)] = t;
    }
}

// a ← a − m (m on the device), with the block sums of the result when asked
template <typename T>
__global__ void shift_kernel(T *__restrict__ a, int n, const double *__restrict__ mptr) {
    const T m = (T)mptr[0];
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) a[t] = a[t] - m;
}

// dst = src in the colour-split layout
__global__ void split_copy_kernel(double *__restrict__ dst, const double *__restrict__ src, int n, SplitMap sm) {
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) dst[split_t(sm, t)] = src[t];
}

// block sums of an array (for a mean)
template <typename T>
__global__ void sum_kernel(const T *__restrict__ a, int n, double *__restrict__ partials) {
    __shared__ double sh[RB / 64];
    double v = 0.0;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) v += (double)a[t];
    double s = block_sum(v, sh);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

template <typename T>
__global__ void sumsq_kernel(const T *__restrict__ a, int n, double *__restrict__ partials) {
    __shared__ double sh[RB / 64];
    double v = 0.0;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) v += (double)a[t] * (double)a[t];
    double s = block_sum(v, sh);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

template <typename T>
__global__ void copyout_kernel(double *__restrict__ out, T *__restrict__ phi, int n, const double *__restrict__ mptr) {
    const double m = mptr[0];
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        const T v = (T)((double)phi[t] - m);
        phi[t] = v;
        out[t] = (double)v;
    }
}

template <typename T>
__global__ void zero_kernel(T *__restrict__ a, int n) {
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) a[t] = T(0);
}

// The coarsest level in one workgroup: 50 red-black sweeps with φ in LDS,
// then the mean projection (_solve_coarsest!, src/Multigrid.jl:685-689).
//
// It is bound by the latency of 100 dependent half-sweeps, so a half-sweep
// must be short. A thread owns S slots of each colour (slot s: row s / h,
// the s % h-th cell of the colour in it, h = ⌈nx/2⌉) and keeps for each, in
// registers, the six neighbours' LDS indices, the six face weights divided
// by the diagonal and b over the diagonal: a half-sweep is six LDS reads,
// six multiply-adds, one LDS write and the barrier. S = 0, for levels of up to
// 4096 cells with more slots than the registers hold (coarsest_slots: 3 per
// thread in FP64, 4 in FP32): the cell's weights are formed from the arrays at
// every visit (one division per cell), b read from memory.
// Measured per launch against the form that read the coefficients and
// divided the linear index by the extents at every visit: 12×12×6 FP64
// 183 → 24 us, 16×16×6 FP32 211 → 27 us.
template <typename T, int S>
__global__ void __launch_bounds__(1024) coarsest_kernel(LevelD<T> L, int nsweeps, int singular,
                                                        const double *__restrict__ bm, int zero_start) {
    extern __shared__ unsigned char smem_raw[];
    T *sphi = reinterpret_cast<T *>(smem_raw);
    const int n = L.nx * L.ny * L.nz;
    __shared__ double sh[1024 / 64];
    // bm: b's pending mean; zero_start: φ enters as zero (not read)
    const T bmv = bm ? (T)bm[0] : T(0);
    for (int t = threadIdx.x; t < n; t += blockDim.x) sphi[t] = zero_start ? T(0) : L.phi[t];
    const int h = (L.nx + 1) / 2, slots = h * L.ny * L.nz;
    // the slot's cell (−1: none, or a fully blocked cell, which keeps φ), its
    // neighbours and weights
    struct Slot {
        int c;
        uint32_t q[3];  // the neighbours of an axis, 16 bits each
        T w[6], b;
    };
    auto make = [&](int s, int colour) {
        Slot o;
        o.c = -1;
        if (s >= slots) return o;
        const int ih = s % h, jk = s / h, j = jk % L.ny, k = jk / L.ny;
        const int i = 2 * ih + ((j + k + colour) & 1);
        if (i >= L.nx) return o;
        T w[6];
        if (L.cx) {
            const uint32_t nx1 = L.nx + 1, ny1 = L.ny + 1;
            w[0] = L.cx[(uint32_t)(i + 1) + nx1 * ((uint32_t)j + (uint32_t)L.ny * k)] * L.ix2;
            w[1] = L.cx[(uint32_t)i + nx1 * ((uint32_t)j + (uint32_t)L.ny * k)] * L.ix2;
            w[2] = L.cy[(uint32_t)i + (uint32_t)L.nx * ((uint32_t)(j + 1) + ny1 * k)] * L.iy2;
            w[3] = L.cy[(uint32_t)i + (uint32_t)L.nx * ((uint32_t)j + ny1 * k)] * L.iy2;
            w[4] = L.cz[lidx(L, i, j, k + 1)] * L.iz2;
            w[5] = L.cz[lidx(L, i, j, k)] * L.iz2;
        } else {
            w[0] = w[1] = L.ix2;
            w[2] = w[3] = L.iy2;
            w[4] = w[5] = L.iz2;
        }
        const T d = -(((w[0] + w[1]) + (w[2] + w[3])) + (w[4] + w[5]));
        if (L.cx && fabs(d) < Eps<T>::v) return o;
        const T id = T(1) / d;
        o.c = (int)lidx(L, i, j, k);
        o.q[0] = lidx(L, wrapc(i + 1, L.nx, L.bcx), j, k) | lidx(L, wrapc(i - 1, L.nx, L.bcx), j, k) << 16;
        o.q[1] = lidx(L, i, wrapc(j + 1, L.ny, L.bcy), k) | lidx(L, i, wrapc(j - 1, L.ny, L.bcy), k) << 16;
        o.q[2] = lidx(L, i, j, wrapc(k + 1, L.nz, L.bcz)) | lidx(L, i, j, wrapc(k - 1, L.nz, L.bcz)) << 16;
#pragma unroll
        for (int m = 0; m < 6; m++) o.w[m] = w[m] * id;
        o.b = (L.b[o.c] - bmv) * id;
        return o;
    };
    auto update = [&](const Slot &o) {
        if (o.c < 0) return;
        const T u = o.w[0] * sphi[o.q[0] & 0xffffu] + o.w[1] * sphi[o.q[0] >> 16];
        const T v = o.w[2] * sphi[o.q[1] & 0xffffu] + o.w[3] * sphi[o.q[1] >> 16];
        const T w = o.w[4] * sphi[o.q[2] & 0xffffu] + o.w[5] * sphi[o.q[2] >> 16];
        sphi[o.c] = o.b - ((u + v) + w);
    };
    if constexpr (S > 0) {
        Slot own[2][S];
#pragma unroll
        for (int colour = 0; colour <= 1; colour++)
#pragma unroll
            for (int q = 0; q < S; q++) own[colour][q] = make((int)threadIdx.x + q * (int)blockDim.x, colour);
        __syncthreads();
        for (int sw = 0; sw < nsweeps; sw++) {
#pragma unroll
            for (int colour = 0; colour <= 1; colour++) {
#pragma unroll
                for (int q = 0; q < S; q++) update(own[colour][q]);
                __syncthreads();
            }
        }
    } else {
        __syncthreads();
        for (int sw = 0; sw < nsweeps; sw++)
            for (int colour = 0; colour <= 1; colour++) {
                for (int s = threadIdx.x; s < slots; s += blockDim.x) update(make(s, colour));
                __syncthreads();
            }
    }
    if (singular) {
        double v = 0.0;
        for (int t = threadIdx.x; t < n; t += blockDim.x) v += (double)sphi[t];
        double s = block_sum(v, sh);
        __shared__ T mean;
        if (threadIdx.x == 0) mean = (T)(s / n);
        __syncthreads();
        for (int t = threadIdx.x; t < n; t += blockDim.x) sphi[t] = sphi[t] - mean;
        __syncthreads();
    }
    for (int t = threadIdx.x; t < n; t += blockDim.x) L.phi[t] = sphi[t];
}

// Slots per thread of coarsest_kernel (0: from memory), or −1 where the level
// takes a launch per half-sweep instead. 1024 threads hold 3 slots of each
// colour in FP64 (4 in FP32) in their 128 registers: 25×17×11 FP64 in
// 104 us against 100 launches of about 4.5 us. Past that the form from
// memory loses to the launches (27×25×19 FP64 1055 us), so it serves only
// levels of up to 4096 cells whose rows are so short that half the slots are
// empty.
static int coarsest_slots(int nx, int ny, int nz, int esz) {
    const int slots = (nx + 1) / 2 * ny * nz, s = (slots + 1023) / 1024;
    if (s <= (esz == 8 ? 3 : 4)) return s;
    return nx * ny * nz <= 4096 ? 0 : -1;
}

// ---- the outer FP64 CG kernels (pcg!, src/Backends.jl:1526-1589) ------------
// Ap = A p on the fine level (FP64), with the block sums of p·Ap
__global__ void cg_apply_kernel(LevelD<double> L, const double *__restrict__ p, double *__restrict__ Ap,
                                double *__restrict__ partials) {
    __shared__ double sh[RB / 64];
    int bxi, j, k;
    xcd_block3(bxi, j, k);
    const int i = bxi * blockDim.x + threadIdx.x;
    double v = 0.0;
    if (i < L.nx) {
        const uint32_t c = lidx(L, i, j, k);
        const double a = applyA(L, p, i, j, k);
        Ap[c] = a;
        v = p[c] * a;
    }
    double s = block_sum(v, sh);
    if (threadIdx.x == 0) partials[blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)] = s;
}

// r −= αAp, block sums of (r², r)  (α from the device); sm: r is colour-split,
// Ap natural
__global__ void cg_update_kernel(double *__restrict__ r, const double *__restrict__ Ap,
                                 const double *__restrict__ aptr, int n, double *__restrict__ partials, int nblk,
                                 SplitMap sm) {
    __shared__ double sh[RB / 64];
    const double alpha = aptr[0];
    double s2 = 0.0, s1 = 0.0;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        const uint32_t q = split_t(sm, t);
        const double rv = r[q] - alpha * Ap[t];
        r[q] = rv;
        s2 += rv * rv;
        s1 += rv;
    }
    double a = block_sum(s2, sh);
    double b = block_sum(s1, sh);
    if (threadIdx.x == 0) { partials[blockIdx.x] = a; partials[nblk + blockIdx.x] = b; }
}

// the preconditioner's right-hand side: level-0 b = T(r − mean r)  (_load_rhs!, src/Multigrid.jl:764-775)
template <typename T>
__global__ void load_rhs_kernel(T *__restrict__ b, const double *__restrict__ r, int n, const double *__restrict__ mptr) {
    const double m = mptr ? mptr[0] : 0.0;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) b[t] = (T)(r[t] - m);
}

// z = φ − mean φ (_store_solution!, :789-793), stored when z is given, and the
// block sums of (r·z, z, r)
template <typename T>
__global__ void store_rz_kernel(double *__restrict__ z, const T *__restrict__ phi, const double *__restrict__ r, int n,
                                const double *__restrict__ mptr, double *__restrict__ partials, int nblk) {
    __shared__ double sh[RB / 64];
    const double m = mptr ? mptr[0] : 0.0;
    double srz = 0.0, sz = 0.0, sr = 0.0;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        const double zv = (double)phi[t] - m;
        if (z) z[t] = zv;
        srz += r[t] * zv;
        sz += zv;
        sr += r[t];
    }
    double a = block_sum(srz, sh), b = block_sum(sz, sh), c = block_sum(sr, sh);
    if (threadIdx.x == 0) {
        partials[blockIdx.x] = a; partials[nblk + blockIdx.x] = b; partials[2 * nblk + blockIdx.x] = c;
    }
}

// the CG's scalars live on the device (slots of the plan's scal array), so
// an iteration reads one block of them on the host: ‖r‖² and the breakdown
// flag. The arithmetic is pcg!'s, in FP64 (src/Backends.jl:1461-1591).
constexpr int S_PAP = 11, S_R2 = 12, S_RZ = 16, S_ALPHA = 17, S_BETA = 18, S_M = 19, S_BREAK = 20;
// slots 32 + 2l and 33 + 2l: level l's pending means of b and of φ after its
// pre-smoothing (the FP64 red-black cycle's coarse levels)
constexpr int MG_NSCAL = 32 + 2 * 24;

// after the first preconditioning: m = Σz/n, rz = r·z − m Σr
__global__ void cg_init_scalars_kernel(double *scal, double dn) {
    const double m = scal[1] / dn;
    double rz = scal[0];
    rz -= m * scal[2];
    scal[S_RZ] = rz; scal[S_M] = m; scal[S_BETA] = 0.0; scal[S_ALPHA] = 0.0; scal[S_BREAK] = 0.0;
}
// α = rz/pAp, or the breakdown flag (|pAp| ≤ ε|rz|) with α = 0
__global__ void cg_alpha_kernel(double *scal) {
    const double pAp = scal[S_PAP], rz = scal[S_RZ];
    const bool ok = fabs(pAp) > DBL_EPSILON * fabs(rz);
    scal[S_BREAK] = ok ? 0.0 : 1.0;
    scal[S_ALPHA] = ok ? rz / pAp : 0.0;
}
// after a preconditioning: m, the new rz and β (pcg!'s rz'/rz, or with an
// FP32 V-cycle the flexible (Polak–Ribière) β = −ẑ'·Ap/pAp)
__global__ void cg_beta_kernel(double *scal, double dn, int flexible) {
    const double m = scal[1] / dn;
    double rzn = scal[0];
    rzn -= m * scal[2];
    scal[S_BETA] = flexible ? -scal[3] / scal[S_PAP] : rzn / scal[S_RZ];
    scal[S_M] = m;
    scal[S_RZ] = rzn;
}

// p = (z − m) + βp  (_pcg_dir_body!, src/Backends.jl:1413-1417); first:
// p = z − m. z is formed from the cycle's φ as store_rz_kernel forms it
// (z = φ − m2, m2 nullable), so that z is never stored; not first, x += αp
// from the p it replaces (the update of x deferred to the pass that reads p
// anyway)
template <typename T>
__global__ void cg_dir_phi_kernel(double *__restrict__ p, const T *__restrict__ phi, int n,
                                  const double *__restrict__ scal, int first, const double *__restrict__ m2ptr,
                                  double *__restrict__ x, SplitMap sm) {
    const double m = scal[S_M], beta = scal[S_BETA], m2 = m2ptr ? m2ptr[0] : 0.0, alpha = scal[S_ALPHA];
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        const double z = (double)phi[split_t(sm, t)] - m2;
        if (first) {
            p[t] = z - m;
        } else {
            const double pv = p[t];
            x[t] = x[t] + alpha * pv;
            p[t] = (z - m) + beta * pv;
        }
    }
}

// the FP32 V-cycle's fused CG sweeps: r −= αAp with the cycle's FP32
// right-hand side written in the same pass (and the sums of r², r); the
// sums of (r·z, z, r, z·Ap) read z = φ of the cycle without storing it; then
// x += αp (deferred from the update) and p = (φ − m) + βp in one pass
template <typename T>
__global__ void cg_update_rhs_kernel(double *__restrict__ r, const double *__restrict__ Ap, T *__restrict__ b,
                                     const double *__restrict__ scal, int n, double *__restrict__ partials, int nblk) {
    __shared__ double sh[RB / 64];
    const double alpha = scal[S_ALPHA];
    double s2 = 0.0, s1 = 0.0;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        const double rv = r[t] - alpha * Ap[t];
        r[t] = rv;
        b[t] = (T)rv;
        s2 += rv * rv;
        s1 += rv;
    }
    double a = block_sum(s2, sh);
    double c = block_sum(s1, sh);
    if (threadIdx.x == 0) { partials[blockIdx.x] = a; partials[nblk + blockIdx.x] = c; }
}
template <typename T>
__global__ void rz_sums_kernel(const T *__restrict__ phi, const double *__restrict__ r, const double *__restrict__ ap,
                               int n, double *__restrict__ partials, int nblk) {
    __shared__ double sh[RB / 64];
    double srz = 0.0, sz = 0.0, sr = 0.0, szap = 0.0;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        const double zv = (double)phi[t];
        srz += r[t] * zv;
        sz += zv;
        sr += r[t];
        if (ap) szap += zv * ap[t];
    }
    double a = block_sum(srz, sh), b = block_sum(sz, sh), c = block_sum(sr, sh);
    double d = ap ? block_sum(szap, sh) : 0.0;
    if (threadIdx.x == 0) {
        partials[blockIdx.x] = a; partials[nblk + blockIdx.x] = b; partials[2 * nblk + blockIdx.x] = c;
        partials[3 * nblk + blockIdx.x] = d;
    }
}
template <typename T>
__global__ void cg_dir_x_kernel(double *__restrict__ x, double *__restrict__ p, const T *__restrict__ phi, int n,
                                const double *__restrict__ scal, int first) {
    const double m = scal[S_M], beta = scal[S_BETA], alpha = scal[S_ALPHA];
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        const double zv = (double)phi[t] - m;
        if (first) {
            p[t] = zv;
        } else {
            const double pv = p[t];
            x[t] = x[t] + alpha * pv;
            p[t] = zv + beta * pv;
        }
    }
}
// block partial sums of a·b (flat grid-stride; nblk blocks)
__global__ void dot_kernel(const double *__restrict__ a, const double *__restrict__ b, int n,
                           double *__restrict__ partials) {
    __shared__ double sh[RB / 64];
    double s = 0.0;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) s += a[t] * b[t];
    const double v = block_sum(s, sh);
    if (threadIdx.x == 0) partials[blockIdx.x] = v;
}
// r = r − Ax (the initial residual of a warm start)
__global__ void sub_kernel(double *__restrict__ r, const double *__restrict__ ax, int n) {
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) r[t] = r[t] - ax[t];
}

__global__ void cg_axpy_kernel(double *__restrict__ x, const double *__restrict__ p, int n,
                               const double *__restrict__ scal) {
    const double alpha = scal[S_ALPHA];
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) x[t] = x[t] + alpha * p[t];
}

__global__ void scale_rows_kernel(double *__restrict__ a, const double *__restrict__ sc, int nxy, int n) {
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) a[t] = a[t] * sc[t / nxy];
}

__global__ void fill_kernel(double *__restrict__ a, int n, double v) {
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) a[t] = v;
}
__global__ void shift_copy_kernel(double *__restrict__ out, const double *__restrict__ x, int n, double m) {
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) out[t] = x[t] - m;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct MGLevelH {
    int nx, ny, nz;
    double dx, dy, dz;
    void *phi = nullptr, *b = nullptr, *r = nullptr, *tmp = nullptr;
    void *cx = nullptr, *cy = nullptr, *cz = nullptr;
};

struct MGPlan {
    int nlev = 0;
    bool gen0 = false;  // the finest level's coefficients from the terrain metrics (FP64 red-black)
    int kc0 = RBC_KC;   // levels per chunk of its kernels
    bool gen1 = false;  // the level below likewise
    int kc1 = RBC_KC;
    double *tab1 = nullptr;  // TFChain2's
    TFM<double> gm{};
    bool gen0f = false;  // likewise in FP32 (FP32 Jacobi V-cycle)
    TFM<float> gmf{};
    MGLevelH L[24];
    // the pending mean of a coarse level's b in a red-black cycle (set by the
    // level above for the cycle's visit, null otherwise)
    const double *bmL[24] = {};
    // the colour split of the finest φ and b and, with gen1, of the next level's
    // (SplitMap::half; 0: natural), on during an FP64 terrain PCG solve
    uint32_t half0 = 0, half1 = 0;
    // every cell of every level has a non-vanishing diagonal
    bool open = false;
    int bcx, bcy, bcz, nu1, nu2, smoother, prec;  // prec 0 double, 1 float
    int wcycle = 0, fmg = 0;  // cycle = :W (two coarse recursions); the nested-iteration start
    double omega;
    bool coeff = false;
    // FP64 fine operator for the CG
    double *cx64 = nullptr, *cy64 = nullptr, *cz64 = nullptr;
    double *rhs_scale = nullptr;
    // CG arrays and reduction scratch
    double *x = nullptr, *r = nullptr, *p = nullptr, *Ap = nullptr;
    double *part = nullptr, *scal = nullptr;  // scal: device scalars
    double *part2 = nullptr;                  // the block sums of a long partial list (≤ 2048)
    int npart = 0;
};

static int ilog2c(int n) { int l = 0; while ((1 << l) < n) l++; return l; }

template <typename T>
static LevelD<T> devlevel(const MGPlan *P, int l) {
    const MGLevelH &h = P->L[l];
    LevelD<T> L;
    L.nx = h.nx; L.ny = h.ny; L.nz = h.nz;
    L.ix2 = T(1.0 / (h.dx * h.dx)); L.iy2 = T(1.0 / (h.dy * h.dy)); L.iz2 = T(1.0 / (h.dz * h.dz));
    L.phi = (T *)h.phi; L.b = (T *)h.b; L.r = (T *)h.r; L.tmp = (T *)h.tmp;
    L.cx = (const T *)h.cx; L.cy = (const T *)h.cy; L.cz = (const T *)h.cz;
    L.bcx = P->bcx; L.bcy = P->bcy; L.bcz = P->bcz;
    return L;
}

static LevelD<double> finelevel64(const MGPlan *P) {
    const MGLevelH &h = P->L[0];
    LevelD<double> L;
    L.nx = h.nx; L.ny = h.ny; L.nz = h.nz;
    L.ix2 = 1.0 / (h.dx * h.dx); L.iy2 = 1.0 / (h.dy * h.dy); L.iz2 = 1.0 / (h.dz * h.dz);
    L.phi = L.b = L.r = L.tmp = nullptr;
    L.cx = P->cx64; L.cy = P->cy64; L.cz = P->cz64;
    L.bcx = P->bcx; L.bcy = P->bcy; L.bcz = P->bcz;
    return L;
}

static dim3 grid3(int nx, int ny, int nz) { return dim3((nx + RB - 1) / RB, ny, nz); }
static int nblocks3(int nx, int ny, int nz) { return ((nx + RB - 1) / RB) * ny * nz; }
// the vector kernels' loops stride by the grid, so any grid is correct.
// Those that also sum take at most 2048 blocks (few partials to fold; the
// per-block sum is amortised); the plain streaming ones take one element
// per work item, on MI355X ≈ 20 % faster than a capped grid walking the
// array in strides. A list of partial sums is folded by ≤ 2048 blocks.
static int flat_blocks(int n) { int b = (n + RB - 1) / RB; return b < 2048 ? b : 2048; }
static int stream_blocks(int n) { return (n + RB - 1) / RB; }
static int fold_blocks(int n) { return flat_blocks(n); }

// out = scale · Σ part[0..n): one block for a short list; a long one (the
// per-row partials of a fine level) is first folded into ≤ 2048 block sums,
// so no single block walks hundreds of thousands of values. Fixed order.
static void finalize_to(MGPlan *P, hipStream_t st, double *out, const double *part, int n, double scale) {
    if (n <= 4096) {
        hipLaunchKernelGGL(finalize_kernel, dim3(1), dim3(RB), 0, st, out, part, n, scale);
        return;
    }
    const int nb = fold_blocks(n);
    hipLaunchKernelGGL(sum_kernel<double>, dim3(nb), dim3(RB), 0, st, part, n, P->part2);
    hipLaunchKernelGGL(finalize_kernel, dim3(1), dim3(RB), 0, st, out, P->part2, nb, scale);
}

// out[c] = Σ part[c·n .. (c+1)·n) for c < ncomp, fixed order: one block
// for short lists, else 64 segment sums per component first
static void finalize_multi_to(MGPlan *P, hipStream_t st, double *out, const double *part, int n, int ncomp) {
    if (n <= 4096) {
        hipLaunchKernelGGL(finalize_multi_kernel, dim3(1), dim3(RB), 0, st, out, part, n, ncomp);
        return;
    }
    hipLaunchKernelGGL(fold_multi_kernel, dim3(ncomp, 64), dim3(RB), 0, st, P->part2, part, n);
    hipLaunchKernelGGL(finalize_multi_kernel, dim3(1), dim3(RB), 0, st, out, (const double *)P->part2, 64, ncomp);
}

// the mean of the interior of `a` (level l) into scal[slot], via partials
template <typename T>
static void mean_to(MGPlan *P, hipStream_t st, const T *a, int n, int slot) {
    int nb = flat_blocks(n);
    hipLaunchKernelGGL(sum_kernel<T>, dim3(nb), dim3(RB), 0, st, a, n, P->part);
    finalize_to(P, st, P->scal + slot, P->part, nb, 1.0 / n);
}

template <typename T>
static void project_mean(MGPlan *P, hipStream_t st, int l) {
    const MGLevelH &h = P->L[l];
    int n = h.nx * h.ny * h.nz;
    mean_to<T>(P, st, (const T *)h.phi, n, 4);
    hipLaunchKernelGGL(shift_kernel<T>, dim3(stream_blocks(n)), dim3(RB), 0, st, (T *)h.phi, n, P->scal + 4);
}

// a cycle's first Jacobi sweep on a level can read its zero start as zero
// (no clearing pass); the coarsest level's solve and red-black sweeps read φ
static bool jacobi_from_zero(const MGPlan *P) { return P->smoother == 1 && P->nu1 >= 1; }
// the finest φ's layout for a kernel of precision T that reads it
template <typename T>
static SplitMap split0(const MGPlan *P) {
    const int nx = P->L[0].nx, ny = P->L[0].ny;
    auto lg = [](int v) { int e = 0; while ((1 << e) < v) e++; return (1 << e) == v ? e : -1; };
    const int sx = lg(nx), sy = lg(ny);
    const bool pow2 = sx >= 0 && sy >= 0;
    return SplitMap{sizeof(T) == 8 ? P->half0 : 0u, nx, ny, pow2 ? sx : -1, pow2 ? sy : -1};
}
// A red-black cycle on an open operator (no fully blocked cell) with
// smoothing on both sides of the coarse correction, or on the terrain grid
// with any, leaves out what changes no iterate of the CG beyond rounding:
//  - the mean removals inside the cycle: a constant is in the kernel of every
//    level's operator, changes no residual and prolongs to a constant, and the
//    residual and its restriction have the mean of b, which the CG keeps zero.
//    Only the coarsest right-hand side's rounding is removed, which 50 sweeps
//    would let drift. (With blocked cells the constant is not the whole
//    kernel: a removal moves the fluid against the blocked cells' values.)
//  - the residual of the colour the last pass updated, and the correction of
//    the colour the next pass overwrites (residual_restrict_kernel,
//    prolong_tf_kernel);
//  - the clearing of φ: a cycle's first sweep starts from zero.
// Without post-smoothing every cell is corrected; without pre-smoothing φ is
// zero (the terrain's cycles are V-cycles from zero) and b is restricted.
// A CG iteration at 512×512×256 with sweeps (2, 0), (1, 0), (0, 2): 8.5, 6.7
// and 8.5 ms through the full cycle and its stored coefficients → 3.7, 3.0, 3.4.
static bool rb_cycle(const MGPlan *P) {
    return P->smoother == 0 && P->open && ((P->nu1 >= 1 && P->nu2 >= 1) || (P->gen0 && !P->wcycle));
}

// m_first: a mean removal of φ still pending, folded into the first sweep
// sums (FP64 terrain finest level): the last pass also writes the block sums
// of b·φ, φ and b to P->part; their count goes to *sum_nb
template <typename T>
static void smooth(MGPlan *P, hipStream_t st, int l, int nsweeps, bool from_zero = false,
                   const double *m_first = nullptr, int *sum_nb = nullptr) {
    MGLevelH &h = P->L[l];
    LevelD<T> L = devlevel<T>(P, l);
    // the finest level's launches are booked one by one when profiling
    const char *tag = l != 0 ? nullptr
                             : (P->smoother == 0 ? (sizeof(T) == 8 ? "mg_rbgs_f64_l0" : "mg_rbgs_f32_l0")
                                                 : (sizeof(T) == 8 ? "mg_jacobi_f64_l0" : "mg_jacobi_f32_l0"));
    if (P->smoother == 0) {
        dim3 g(((h.nx + 1) / 2 + RB - 1) / RB, h.ny, h.nz);
        const bool gen = sizeof(T) == 8 && l == 0 && P->gen0;
        const bool gen1 = sizeof(T) == 8 && l == 1 && P->half1;
        for (int s = 0; s < nsweeps; s++)
            for (int colour = 0; colour <= 1; colour++) {
                ProfScope ps(tag);
                if (gen || gen1) {
                    const int kc = gen ? P->kc0 : P->kc1;
                    const dim3 gr((h.nx + 63) / 64, (h.ny + RBC_BY - 1) / RBC_BY, (h.nz + kc - 1) / kc);
                    const int nb = (int)(gr.x * gr.y * gr.z);
                    const bool zero = from_zero && s == 0;
                    const bool sums = sum_nb && s == nsweeps - 1 && colour == 1;
                    auto launch = [&](auto kern) {
                        hipLaunchKernelGGL(kern, gr, dim3(64, RBC_BY), 0, st, devlevel<double>(P, l), P->gm, (const double *)P->tab1, colour, kc,
                                           (int)(zero && colour == 1), P->part, nb, gen ? P->half0 : P->half1);
                    };
                    if (gen1) {
                        if (zero && colour == 0) launch(rbgs_tf_kernel<true, false, TFChain2>);
                        else launch(rbgs_tf_kernel<false, false, TFChain2>);
                    } else if (sums) {
                        *sum_nb = nb;
                        launch(rbgs_tf_kernel<false, true, TFChain<double>>);
                    } else if (zero && colour == 0) {
                        launch(rbgs_tf_kernel<true, false, TFChain<double>>);
                    } else {
                        launch(rbgs_tf_kernel<false, false, TFChain<double>>);
                    }
                } else {
                    // the generic sweep: a pending b mean (bmL), the first pass
                    // from zero, a pending φ mean folded into the first sweep
                    const double *bm = P->bmL[l];
                    if (from_zero && s == 0 && colour == 0)
                        hipLaunchKernelGGL((rbgs_kernel<T, 3>), g, dim3(RB), 0, st, L, colour, m_first, bm);
                    else if (m_first && s == 0 && colour == 0)
                        hipLaunchKernelGGL((rbgs_kernel<T, 1>), g, dim3(RB), 0, st, L, colour, m_first, bm);
                    else if (m_first && s == 0)
                        hipLaunchKernelGGL((rbgs_kernel<T, 2>), g, dim3(RB), 0, st, L, colour, m_first, bm);
                    else
                        hipLaunchKernelGGL((rbgs_kernel<T, 0>), g, dim3(RB), 0, st, L, colour, m_first, bm);
                }
            }
    } else {
        const bool gen = sizeof(T) == 4 && l == 0 && P->gen0f;
        const int kc = h.nz < JTF_KC ? h.nz : JTF_KC;
        for (int s = 0; s < nsweeps; s++) {
            ProfScope ps(tag);
            const T *src = (from_zero && s == 0) ? (const T *)nullptr : (const T *)h.phi;
            if (gen)
                hipLaunchKernelGGL(jacobi_tf_kernel<0>, dim3((h.nx + 63) / 64, (h.ny + JTF_BY - 1) / JTF_BY,
                                                             (h.nz + kc - 1) / kc),
                                   dim3(64, JTF_BY), 0, st, devlevel<float>(P, 0), P->gmf, (const float *)src,
                                   (float *)h.tmp, (float)P->omega, kc);
            else
                hipLaunchKernelGGL(jacobi_kernel<T>, grid3(h.nx, h.ny, h.nz), dim3(RB), 0, st, L, src, (T *)h.tmp,
                                   (T)P->omega);
            std::swap(h.phi, h.tmp);
            L = devlevel<T>(P, l);
        }
    }
}

// the FP64 red-black cycle on a coarse level l ≥ 1 folds its mean removals
// into the kernels that read the values next (the same values as the
// explicit shifts): b's (the restricted residual's mean) into every kernel
// that reads b; φ's after the pre-smoothing into the residual and the
// prolongation; after the prolongation into the first post-smoothing
// sweep; after the post-smoothing into the level above's prolongation. The
// cycle's first sweep starts from zero (no clearing pass). Not for the
// W-cycle, whose second visit starts from the first one's φ.
template <typename T>
static bool coarse_fold(const MGPlan *P, int l) {
    return sizeof(T) == 8 && P->prec == 0 && !rb_cycle(P) && !P->wcycle && P->smoother == 0 && l >= 1 && 33 + 2 * l < MG_NSCAL;
}

int chunk_tf_prolong(int nx, int ny, int nz) {
    return chunk_levels(((nx + 63) / 64) * ((ny + PRC_BY - 1) / PRC_BY), nz, PRC_KC, PRC_FILL, 2, 2);
}
int chunk_tf_smooth(int nx, int ny, int nz) {
    return chunk_levels(((nx + 63) / 64) * ((ny + RBC_BY - 1) / RBC_BY), nz, RBC_KC, RBC_FILL, 3, 2);
}
static int prolong_chunk(const MGLevelH &h) { return chunk_tf_prolong(h.nx, h.ny, h.nz); }

// φ of level l += the prolongation of the coarse φ, with the block sums of
// the result in P->part; returns their count. pre_m, mc: pending means of the
// fine and the coarse φ
template <typename T>
static int prolong(MGPlan *P, hipStream_t st, int l, const double *pre_m, const double *mc) {
    const MGLevelH &h = P->L[l];
    const LevelD<T> L = devlevel<T>(P, l), C = devlevel<T>(P, l + 1);
    if (l == 0 && h.nx % 2 == 0 && h.ny % 2 == 0 && h.nz % 2 == 0) {
        const int kc = prolong_chunk(h);
        const dim3 gp((h.nx + 63) / 64, (h.ny + PRC_BY - 1) / PRC_BY, (h.nz + kc - 1) / kc);
        hipLaunchKernelGGL(prolong_col_kernel<T>, gp, dim3(64, PRC_BY), 0, st, L, C, kc, P->part, pre_m, mc);
        return (int)(gp.x * gp.y * gp.z);
    }
    hipLaunchKernelGGL(prolong_kernel<T>, grid3(h.nx, h.ny, h.nz), dim3(RB), 0, st, L, C, P->part, pre_m, mc);
    return nblocks3(h.nx, h.ny, h.nz);
}
// zero_start: φ of level l enters as zero (a preconditioner's cycle or the
// first visit of a coarse level), so a Jacobi smoother's first sweep can
// read it as zero without a clearing pass. defer_final: leave the
// post-smoothing's mean removal pending, its mean in slot 4 (for the folded
// coarse levels); returns whether it was left pending. sum_nb: smooth's, for
// the finest level's last pass
template <typename T>
static bool vcycle(MGPlan *P, hipStream_t st, int l, bool zero_start, bool defer_final = false, int *sum_nb = nullptr) {
    MGLevelH &h = P->L[l];
    const int n = h.nx * h.ny * h.nz;
    const bool cf = coarse_fold<T>(P, l);
    const bool rb = rb_cycle(P) && P->nlev > 1 && (P->nu1 >= 1 || zero_start);
    if (l == P->nlev - 1) {
        const int own = coarsest_slots(h.nx, h.ny, h.nz, sizeof(T));
        if (own >= 0) {
            // as few waves as hold the slots of one colour (a barrier of fewer waves is shorter)
            const int slots = (h.nx + 1) / 2 * h.ny * h.nz, bt = slots >= 1024 ? 1024 : (slots + 63) / 64 * 64;
            auto launch = [&](auto kern) {
                hipLaunchKernelGGL(kern, dim3(1), dim3(bt), sizeof(T) * (size_t)n, st, devlevel<T>(P, l), 50, 1,
                                   cf || rb ? P->bmL[l] : (const double *)nullptr, (int)((cf || rb) && zero_start));
            };
            if (own == 1) launch(coarsest_kernel<T, 1>);
            else if (own == 2) launch(coarsest_kernel<T, 2>);
            else if (own == 3) launch(coarsest_kernel<T, 3>);
            else if (own == 4) launch(coarsest_kernel<T, sizeof(T) == 4 ? 4 : 3>);
            else launch(coarsest_kernel<T, 0>);
        } else {
            int sm = P->smoother;
            P->smoother = 0;
            smooth<T>(P, st, l, 50, (cf || rb) && zero_start);
            P->smoother = sm;
            if (rb) return false;
            if (cf && defer_final) {
                mean_to<T>(P, st, (const T *)h.phi, n, 4);
                return true;
            }
            project_mean<T>(P, st, l);
        }
        return false;
    }
    MGLevelH &c = P->L[l + 1];
    const int nc = c.nx * c.ny * c.nz;
    if (rb) {
        if (P->nu1 >= 1) smooth<T>(P, st, l, P->nu1, zero_start);
        else hipLaunchKernelGGL(zero_kernel<T>, dim3(stream_blocks(n)), dim3(RB), 0, st, (T *)h.phi, n);
        const bool last = l + 1 == P->nlev - 1;  // the coarsest right-hand side: its mean is left out
        const LevelD<T> L = devlevel<T>(P, l), C = devlevel<T>(P, l + 1);
        double *part = last ? P->part : nullptr;
        // the colour split of the levels (the finest one's transfers by the metrics take it)
        const uint32_t half = l == 0 ? P->half0 : l == 1 ? P->half1 : 0u, halfc = l == 0 ? P->half1 : 0u;
        const bool gen = sizeof(T) == 8 && l == 0 && half;
        int nb;
        if (P->nu1 == 0) {
            nb = stream_blocks(nc);
            hipLaunchKernelGGL(restrict_rhs_kernel, dim3(nb), dim3(RB), 0, st, devlevel<double>(P, l + 1),
                               devlevel<double>(P, l), part, half, halfc);
        } else if (gen) {
            const dim3 gr((c.nx + 31) / 32, (c.ny + RRC_BW - 1) / RRC_BW, (h.nz + P->kc0 - 1) / P->kc0);
            nb = (int)(gr.x * gr.y * gr.z);
            hipLaunchKernelGGL(residual_restrict_tf_kernel, gr, dim3(64, RRC_BW), 0, st, devlevel<double>(P, 0),
                               devlevel<double>(P, 1), P->gm, P->kc0, part, half, halfc);
        } else {
            nb = stream_blocks(nc);
            if (half)
                hipLaunchKernelGGL((residual_restrict_kernel<T, true>), dim3(nb), dim3(RB), 0, st, C, L, part, half);
            else
                hipLaunchKernelGGL((residual_restrict_kernel<T>), dim3(nb), dim3(RB), 0, st, C, L, part, 0u);
        }
        if (last) {
            P->bmL[l + 1] = P->scal + 32 + 2 * (l + 1);
            finalize_to(P, st, P->scal + 32 + 2 * (l + 1), P->part, nb, 1.0 / nc);
        }
        for (int rec = 0; rec < (P->wcycle ? 2 : 1); rec++) vcycle<T>(P, st, l + 1, rec == 0);
        P->bmL[l + 1] = nullptr;
        if (half) {
            const int kc = prolong_chunk(h);
            hipLaunchKernelGGL(prolong_tf_kernel, dim3((c.nx + 63) / 64, (h.ny + PRC_BY - 1) / PRC_BY, (h.nz + kc - 1) / kc),
                               dim3(64, PRC_BY), 0, st, devlevel<double>(P, l), devlevel<double>(P, l + 1), kc, half, halfc,
                               (int)(P->nu2 == 0));
        } else {
            prolong<T>(P, st, l, nullptr, nullptr);
        }
        smooth<T>(P, st, l, P->nu2, false, nullptr, sum_nb);
        return false;
    }
    // the FP32 V-cycle keeps only the projection that makes the coarsest
    // problem consistent (the restricted residual's mean): a constant in φ
    // is in the operator's kernel, changes no residual, and the CG removes
    // z's mean when it forms the direction
    const bool lean = P->prec != 0;
    const double *bm = cf ? P->bmL[l] : nullptr;  // b's pending mean
    smooth<T>(P, st, l, P->nu1, zero_start && (jacobi_from_zero(P) || (cf && P->nu1 >= 1)));
    const double *pre_m = nullptr;  // φ's pending mean after the pre-smoothing
    if (cf) {
        mean_to<T>(P, st, (const T *)h.phi, n, 33 + 2 * l);
        pre_m = P->scal + 33 + 2 * l;
    } else if (!lean) {
        project_mean<T>(P, st, l);
    }
    // residual, its mean, and the restriction of (r − m)
    LevelD<T> L = devlevel<T>(P, l), C = devlevel<T>(P, l + 1);
    int nb = nblocks3(h.nx, h.ny, h.nz);
    // (the FP32 cycle makes only the coarsest problem consistent: a mean in
    // an intermediate level's right-hand side drifts that level's φ by a
    // constant, which the next consistent level and the CG ignore)
    const bool consistent = !lean || l + 1 == P->nlev - 1;
    if (sizeof(T) == 4 && l == 0 && P->gen0f && !consistent) {
        const int kc = h.nz < JTF_KC ? h.nz : JTF_KC;
        hipLaunchKernelGGL(jacobi_tf_kernel<1>, dim3((h.nx + 63) / 64, (h.ny + JTF_BY - 1) / JTF_BY, (h.nz + kc - 1) / kc),
                           dim3(64, JTF_BY), 0, st, devlevel<float>(P, 0), P->gmf, (const float *)h.phi,
                           (float *)h.r, 0.f, kc);
    } else {
        hipLaunchKernelGGL(residual_kernel<T>, grid3(h.nx, h.ny, h.nz), dim3(RB), 0, st, L, P->part, pre_m, bm);
    }
    if (consistent) finalize_to(P, st, P->scal + 5, P->part, nb, 1.0 / n);
    int nbc = nblocks3(c.nx, c.ny, c.nz);
    hipLaunchKernelGGL(restrict_kernel<T>, grid3(c.nx, c.ny, c.nz), dim3(RB), 0, st, C, L,
                       consistent ? (const double *)(P->scal + 5) : (const double *)nullptr, P->part);
    // the coarse level's b mean: removed here, or left pending for its kernels
    const bool ccf = coarse_fold<T>(P, l + 1);
    if (consistent) {
        if (ccf) {
            finalize_to(P, st, P->scal + 32 + 2 * (l + 1), P->part, nbc, 1.0 / nc);
            P->bmL[l + 1] = P->scal + 32 + 2 * (l + 1);
        } else {
            finalize_to(P, st, P->scal + 6, P->part, nbc, 1.0 / nc);
            hipLaunchKernelGGL(shift_kernel<T>, dim3(stream_blocks(nc)), dim3(RB), 0, st, (T *)c.b, nc, P->scal + 6);
        }
    }
    // the coarse φ is cleared here unless its first sweep starts from zero
    const bool child_fz = ccf && (l + 1 == P->nlev - 1 || P->nu1 >= 1);
    const bool skip_zero = (jacobi_from_zero(P) && l + 1 < P->nlev - 1) || child_fz;
    if (!skip_zero) hipLaunchKernelGGL(zero_kernel<T>, dim3(stream_blocks(nc)), dim3(RB), 0, st, (T *)c.phi, nc);
    bool child_def = false;
    for (int rec = 0; rec < (P->wcycle ? 2 : 1); rec++) child_def = vcycle<T>(P, st, l + 1, rec == 0, ccf);
    P->bmL[l + 1] = nullptr;
    // prolong and correct (with the sum of the corrected φ), project
    const int nb_p = prolong<T>(P, st, l, pre_m, child_def ? (const double *)(P->scal + 4) : (const double *)nullptr);
    // the corrected φ's mean: folded into the first post-smoothing sweep
    const bool post_fold = cf && P->nu2 >= 1;
    if (!lean) {
        finalize_to(P, st, P->scal + 4, P->part, nb_p, 1.0 / n);
        if (!post_fold)
            hipLaunchKernelGGL(shift_kernel<T>, dim3(stream_blocks(n)), dim3(RB), 0, st, (T *)h.phi, n, P->scal + 4);
    }
    smooth<T>(P, st, l, P->nu2, false, post_fold ? (const double *)(P->scal + 4) : (const double *)nullptr);
    if (cf && defer_final) {
        mean_to<T>(P, st, (const T *)h.phi, n, 4);
        return true;
    }
    if (!lean) project_mean<T>(P, st, l);
    return false;
}

// coefficient coarsening, _restrict_coeff (src/Multigrid.jl:465-496), on the host in FP64
static void restrict_coeff(const std::vector<double> &cx, const std::vector<double> &cy, const std::vector<double> &cz,
                           int fnx, int fny, int fnz, std::vector<double> &Cx, std::vector<double> &Cy,
                           std::vector<double> &Cz, int cnx, int cny, int cnz) {
    auto FX = [&](int i, int j, int k) { return cx[(size_t)(i - 1) + (size_t)(fnx + 1) * ((j - 1) + (size_t)fny * (k - 1))]; };
    auto FY = [&](int i, int j, int k) { return cy[(size_t)(i - 1) + (size_t)fnx * ((j - 1) + (size_t)(fny + 1) * (k - 1))]; };
    auto FZ = [&](int i, int j, int k) { return cz[(size_t)(i - 1) + (size_t)fnx * ((j - 1) + (size_t)fny * (k - 1))]; };
    Cx.assign((size_t)(cnx + 1) * cny * cnz, 0);
    Cy.assign((size_t)cnx * (cny + 1) * cnz, 0);
    Cz.assign((size_t)cnx * cny * (cnz + 1), 0);
    const double quarter = 1.0 / 4;
    auto mn = [](int a, int b) { return a < b ? a : b; };
    for (int K = 1; K <= cnz; K++)
        for (int J = 1; J <= cny; J++)
            for (int I = 1; I <= cnx + 1; I++) {
                int i = 2 * I - 1;
                double s = 0;
                for (int dk = 0; dk <= 1; dk++)
                    for (int dj = 0; dj <= 1; dj++) s += FX(mn(i, fnx + 1), mn(2 * J - 1 + dj, fny), mn(2 * K - 1 + dk, fnz));
                Cx[(size_t)(I - 1) + (size_t)(cnx + 1) * ((J - 1) + (size_t)cny * (K - 1))] = s * quarter;
            }
    for (int K = 1; K <= cnz; K++)
        for (int J = 1; J <= cny + 1; J++)
            for (int I = 1; I <= cnx; I++) {
                int j = 2 * J - 1;
                double s = 0;
                for (int dk = 0; dk <= 1; dk++)
                    for (int di = 0; di <= 1; di++) s += FY(mn(2 * I - 1 + di, fnx), mn(j, fny + 1), mn(2 * K - 1 + dk, fnz));
                Cy[(size_t)(I - 1) + (size_t)cnx * ((J - 1) + (size_t)(cny + 1) * (K - 1))] = s * quarter;
            }
    for (int K = 1; K <= cnz + 1; K++)
        for (int J = 1; J <= cny; J++)
            for (int I = 1; I <= cnx; I++) {
                int k = 2 * K - 1;
                double s = 0;
                for (int dj = 0; dj <= 1; dj++)
                    for (int di = 0; di <= 1; di++) s += FZ(mn(2 * I - 1 + di, fnx), mn(2 * J - 1 + dj, fny), mn(k, fnz + 1));
                Cz[(size_t)(I - 1) + (size_t)cnx * ((J - 1) + (size_t)cny * (K - 1))] = s * quarter;
            }
}

template <typename T>
static hipError_t upload_as(void **dst, const std::vector<double> &h) {
    std::vector<T> t(h.begin(), h.end());
    hipError_t e = hipMalloc(dst, sizeof(T) * t.size());
    if (e != hipSuccess) return e;
    return upload_dev(*dst, t.data(), sizeof(T) * t.size());
}

MGPlan *mg_create(int nx, int ny, int nz, double dx, double dy, double dz, int bcx, int bcy, int bcz, const double *cx,
                  const double *cy, const double *cz, const double *rhs_scale, int nu1, int nu2, int smoother,
                  double omega, int prec, int min_size, char *err, size_t errlen) {
    auto fail = [&](const char *m) { snprintf(err, errlen, "%s", m); return (MGPlan *)nullptr; };
    MGPlan *P = new MGPlan();
    P->bcx = bcx; P->bcy = bcy; P->bcz = bcz; P->nu1 = nu1; P->nu2 = nu2; P->smoother = smoother;
    P->omega = omega; P->prec = prec;
    P->coeff = cx != nullptr;
    P->open = !P->coeff;
    const size_t esz = prec == 0 ? 8 : 4;
    std::vector<double> hx, hy, hz;
    if (P->coeff) {
        hx.assign(cx, cx + (size_t)(nx + 1) * ny * nz);
        hy.assign(cy, cy + (size_t)nx * (ny + 1) * nz);
        hz.assign(cz, cz + (size_t)nx * ny * (nz + 1));
        if (upload_as<double>((void **)&P->cx64, hx) || upload_as<double>((void **)&P->cy64, hy) ||
            upload_as<double>((void **)&P->cz64, hz))
            return fail("mg: allocation failed");
    }
    int lx = nx, ly = ny, lz = nz;
    double ddx = dx, ddy = dy, ddz = dz;
    while (true) {
        MGLevelH &h = P->L[P->nlev];
        h.nx = lx; h.ny = ly; h.nz = lz; h.dx = ddx; h.dy = ddy; h.dz = ddz;
        size_t n = (size_t)lx * ly * lz;
        void **arrs[4] = {&h.phi, &h.b, &h.r, &h.tmp};
        for (auto a : arrs) {
            if (hipMalloc(a, esz * n) != hipSuccess) return fail("mg: allocation failed");
            zero_dev(*a, esz * n);
        }
        if (P->coeff) {
            hipError_t e1 = prec == 0 ? upload_as<double>(&h.cx, hx) : upload_as<float>(&h.cx, hx);
            hipError_t e2 = prec == 0 ? upload_as<double>(&h.cy, hy) : upload_as<float>(&h.cy, hy);
            hipError_t e3 = prec == 0 ? upload_as<double>(&h.cz, hz) : upload_as<float>(&h.cz, hz);
            if (e1 || e2 || e3) return fail("mg: allocation failed");
        }
        P->nlev++;
        // the coarsening rule, src/Multigrid.jl:576-590
        bool cxo = lx % 2 == 0 && lx / 2 >= min_size, cyo = ly % 2 == 0 && ly / 2 >= min_size,
             czo = lz % 2 == 0 && lz / 2 >= min_size;
        if (!(cxo && cyo && czo) || P->nlev >= 24) break;
        int nlx = lx / 2, nly = ly / 2, nlz = lz / 2;
        if (P->coeff) {
            std::vector<double> Cx, Cy, Cz;
            restrict_coeff(hx, hy, hz, lx, ly, lz, Cx, Cy, Cz, nlx, nly, nlz);
            hx.swap(Cx); hy.swap(Cy); hz.swap(Cz);
        }
        lx = nlx; ly = nly; lz = nlz;
        ddx *= 2; ddy *= 2; ddz *= 2;
    }
    size_t n0 = (size_t)nx * ny * nz;
    double **cg[4] = {&P->x, &P->r, &P->p, &P->Ap};
    for (auto a : cg) {
        if (hipMalloc(a, 8 * n0) != hipSuccess) return fail("mg: allocation failed");
        zero_dev(*a, 8 * n0);
    }
    // partial sums: the fine level's row blocks, or four per streaming block
    P->npart = nblocks3(nx, ny, nz);
    if (P->npart < 4 * flat_blocks((int)n0)) P->npart = 4 * flat_blocks((int)n0);
    if (P->npart < 4 * 2048) P->npart = 4 * 2048;
    // three sums per block of the terrain finest level's last pass (two levels a chunk at least)
    const int npt = 3 * ((nx + 63) / 64) * ((ny + RBC_BY - 1) / RBC_BY) * ((nz + 1) / 2);
    if (P->coeff && prec == 0 && P->npart < npt) P->npart = npt;
    if (hipMalloc(&P->part, sizeof(double) * P->npart) != hipSuccess) return fail("mg: allocation failed");
    if (hipMalloc(&P->part2, sizeof(double) * 2048) != hipSuccess) return fail("mg: allocation failed");
    if (hipMalloc(&P->scal, sizeof(double) * MG_NSCAL) != hipSuccess) return fail("mg: allocation failed");
    zero_dev(P->scal, sizeof(double) * MG_NSCAL);
    if (rhs_scale) {
        std::vector<double> rs(rhs_scale, rhs_scale + nz);
        if (upload_as<double>((void **)&P->rhs_scale, rs)) return fail("mg: allocation failed");
    }
    hipDeviceSynchronize();
    return P;
}

void mg_destroy(MGPlan *P) {
    if (!P) return;
    for (int l = 0; l < P->nlev; l++) {
        MGLevelH &h = P->L[l];
        hipFree(h.phi); hipFree(h.b); hipFree(h.r); hipFree(h.tmp); hipFree(h.cx); hipFree(h.cy); hipFree(h.cz);
    }
    hipFree(P->cx64); hipFree(P->cy64); hipFree(P->cz64); hipFree(P->rhs_scale);
    hipFree(P->x); hipFree(P->r); hipFree(P->p); hipFree(P->Ap);
    hipFree(P->part); hipFree(P->part2); hipFree(P->scal); hipFree(P->tab1);
    delete P;
}

int mg_levels(const MGPlan *P) { return P->nlev; }

// z = M⁻¹ r: one V-cycle from zero, the reference's _mg_precond! (src/Multigrid.jl:922-932);
// returns with the block sums of (r·z, z, r) finalised into scal[0..2]. z is
// stored when given (not aliased with r); the CG forms it again from φ with
// cg_dir_phi_kernel. The FP32 V-cycle neither removes r's mean (r is mean-free in a
// consistent CG to its rounding) nor z's: the CG subtracts Σz/n when it
// forms the direction (the sums above carry what it needs). A red-black
// cycle on an open operator leaves z's mean in likewise.
// rsum_in_part: P->part[fb .. 2fb) holds the block sums of r in sum_kernel's
// layout (cg_update_kernel's second component), so r's mean needs no pass
template <typename T>
static void precond(MGPlan *P, hipStream_t st, const double *r, double *z = nullptr, bool rsum_in_part = false) {
    MGLevelH &h = P->L[0];
    const int n = h.nx * h.ny * h.nz;
    const int fb = flat_blocks(n);
    const bool lean = P->prec != 0;
    const bool rb = rb_cycle(P) && P->nlev > 1;
    // the mean of r, then b = r − m
    if (!lean && rsum_in_part) finalize_to(P, st, P->scal + 7, P->part + fb, fb, 1.0 / n);
    else if (!lean) mean_to<double>(P, st, r, n, 7);
    hipLaunchKernelGGL(load_rhs_kernel<T>, dim3(stream_blocks(n)), dim3(RB), 0, st, (T *)h.b, r, n,
                       lean ? (const double *)nullptr : (const double *)(P->scal + 7));
    if (!(jacobi_from_zero(P) && P->nlev > 1) && !rb)
        hipLaunchKernelGGL(zero_kernel<T>, dim3(stream_blocks(n)), dim3(RB), 0, st, (T *)h.phi, n);
    vcycle<T>(P, st, 0, true);
    const double *m2 = nullptr;
    if (!lean && !rb) {
        mean_to<T>(P, st, (const T *)h.phi, n, 8);
        m2 = P->scal + 8;
    }
    hipLaunchKernelGGL(store_rz_kernel<T>, dim3(fb), dim3(RB), 0, st, z, (const T *)h.phi, r, n, m2, P->part, fb);
    finalize_multi_to(P, st, P->scal, P->part, fb, 3);
}

// the FP64 terrain cycle inside the CG: r in place as the finest right-hand
// side (colour-split), the sums of (r·z, z, r), z = φ, from the last pass, if there is one
static void precond_split(MGPlan *P, hipStream_t st) {
    int nb = 0;
    vcycle<double>(P, st, 0, true, false, &nb);
    if (nb == 0) {  // no post-smoothing
        const MGLevelH &h = P->L[0];
        const int n = h.nx * h.ny * h.nz;
        nb = flat_blocks(n);
        hipLaunchKernelGGL(store_rz_kernel<double>, dim3(nb), dim3(RB), 0, st, (double *)nullptr, (const double *)h.phi,
                           (const double *)h.b, n, (const double *)nullptr, P->part, nb);
    }
    finalize_multi_to(P, st, P->scal, P->part, nb, 3);
}

// the FP32 V-cycle's preconditioning inside the fused CG: the level-0
// right-hand side is already in place (written by the update sweep); the
// sums of (r·z, z, r[, z·Ap]) from the cycle's φ into scal[0..3]
template <typename T>
static void precond_fused(MGPlan *P, hipStream_t st, const double *ap) {
    MGLevelH &h = P->L[0];
    const int n = h.nx * h.ny * h.nz;
    const int fb = flat_blocks(n);
    if (!(jacobi_from_zero(P) && P->nlev > 1) && !(rb_cycle(P) && P->nlev > 1))
        hipLaunchKernelGGL(zero_kernel<T>, dim3(stream_blocks(n)), dim3(RB), 0, st, (T *)h.phi, n);
    vcycle<T>(P, st, 0, true);
    hipLaunchKernelGGL(rz_sums_kernel<T>, dim3(fb), dim3(RB), 0, st, (const T *)h.phi, (const double *)P->r, ap, n,
                       P->part, fb);
    finalize_multi_to(P, st, P->scal, P->part, fb, ap ? 4 : 3);
}

static double read_scal(hipStream_t st, const double *d) {
    double v = 0;
    hipMemcpyAsync(&v, d, sizeof(double), hipMemcpyDeviceToHost, st);
    hipStreamSynchronize(st);
    return v;
}
static void read_scals(hipStream_t st, const double *d, double *h, int n) {
    hipMemcpyAsync(h, d, sizeof(double) * n, hipMemcpyDeviceToHost, st);
    hipStreamSynchronize(st);
}

// pcg!'s iteration (src/Backends.jl:1461-1591) from P->x, P->r (‖r‖ =
// *rnorm): preconditioned by the plan's V-cycle, A the caller's operator or
// (op null) the plan's fine one. One host read per iteration (‖r‖² and the
// breakdown flag); α, β, m live on the device. x += αp is deferred to the
// direction update, which reads p anyway (a last axpy on convergence). An
// FP32 V-cycle takes the fused sweeps (r and the cycle's FP32 right-hand
// side in one pass, z never stored) and the flexible β.
static int pcg_run(MGPlan *P, hipStream_t st, const FCGOp *op, double tol, double bnorm, int maxit, int *iters_out,
                   double *rnorm_io) {
    MGLevelH &h = P->L[0];
    const int n = h.nx * h.ny * h.nz;
    const int fb = flat_blocks(n), sb = stream_blocks(n);
    const double dn = (double)n;
    const bool fused = P->prec != 0;
    const bool split = !fused && P->half0 != 0;  // the FP64 terrain cycle: r lives in the finest b, colour-split
    // the FP64 cycle's z = φ − m2
    const double *m2 = !split && !(rb_cycle(P) && P->nlev > 1) ? (const double *)(P->scal + 8) : (const double *)nullptr;
    double rnorm = *rnorm_io;
    int iters = 0, status = rnorm <= tol * bnorm ? 0 : 1;
    if (status != 0 && split)
        hipLaunchKernelGGL(split_copy_kernel, dim3(sb), dim3(RB), 0, st, (double *)h.b, (const double *)P->r, n,
                           split0<double>(P));
    if (status != 0) {
        if (fused) {
            hipLaunchKernelGGL(load_rhs_kernel<float>, dim3(sb), dim3(RB), 0, st, (float *)h.b, (const double *)P->r,
                               n, (const double *)nullptr);
            precond_fused<float>(P, st, nullptr);
        } else if (split) {
            precond_split(P, st);
        } else {
            precond<double>(P, st, P->r);
        }
        hipLaunchKernelGGL(cg_init_scalars_kernel, dim3(1), dim3(1), 0, st, P->scal, dn);
        if (fused)
            hipLaunchKernelGGL(cg_dir_x_kernel<float>, dim3(sb), dim3(RB), 0, st, P->x, P->p, (const float *)h.phi, n,
                               (const double *)P->scal, 1);
        else
            hipLaunchKernelGGL(cg_dir_phi_kernel<double>, dim3(sb), dim3(RB), 0, st, P->p, (const double *)h.phi, n,
                               (const double *)P->scal, 1, m2, (double *)nullptr, split0<double>(P));
    }
    const int nb3 = nblocks3(h.nx, h.ny, h.nz);
    while (status != 0 && iters < maxit) {
        // Ap and p·Ap into scal[S_PAP]
        int np = -1;
        if (!op) {
            hipLaunchKernelGGL(cg_apply_kernel, grid3(h.nx, h.ny, h.nz), dim3(RB), 0, st, finelevel64(P),
                               (const double *)P->p, P->Ap, P->part);
            finalize_to(P, st, P->scal + S_PAP, P->part, nb3, 1.0);
        } else {
            if (op->apply_dot) np = op->apply_dot(op->ctx, st, P->Ap, P->p, P->part, P->npart);
            else op->apply(op->ctx, st, P->Ap, P->p);
            if (np > 0) {
                finalize_to(P, st, P->scal + S_PAP, P->part, np, 1.0);
            } else {
                hipLaunchKernelGGL(dot_kernel, dim3(fb), dim3(RB), 0, st, (const double *)P->p, (const double *)P->Ap,
                                   n, P->part);
                finalize_to(P, st, P->scal + S_PAP, P->part, fb, 1.0);
            }
        }
        hipLaunchKernelGGL(cg_alpha_kernel, dim3(1), dim3(1), 0, st, P->scal);
        if (fused)
            hipLaunchKernelGGL(cg_update_rhs_kernel<float>, dim3(fb), dim3(RB), 0, st, P->r, (const double *)P->Ap,
                               (float *)h.b, (const double *)P->scal, n, P->part, fb);
        else
            hipLaunchKernelGGL(cg_update_kernel, dim3(fb), dim3(RB), 0, st, split ? (double *)h.b : P->r,
                               (const double *)P->Ap, (const double *)(P->scal + S_ALPHA), n, P->part, fb,
                               split0<double>(P));
        finalize_multi_to(P, st, P->scal + S_R2, P->part, fb, 2);
        double sc[S_BREAK - S_R2 + 1];
        read_scals(st, P->scal + S_R2, sc, S_BREAK - S_R2 + 1);
        if (sc[S_BREAK - S_R2] != 0.0) { status = 2; break; }  // α was 0: nothing moved
        iters++;
        rnorm = sqrt(sc[0]);
        if (rnorm <= tol * bnorm) {
            hipLaunchKernelGGL(cg_axpy_kernel, dim3(sb), dim3(RB), 0, st, P->x, (const double *)P->p, n,
                               (const double *)P->scal);
            status = 0;
            break;
        }
        if (fused) precond_fused<float>(P, st, P->Ap);
        else if (split) precond_split(P, st);
        else precond<double>(P, st, P->r, nullptr, true);
        hipLaunchKernelGGL(cg_beta_kernel, dim3(1), dim3(1), 0, st, P->scal, dn, (int)fused);
        if (fused)
            hipLaunchKernelGGL(cg_dir_x_kernel<float>, dim3(sb), dim3(RB), 0, st, P->x, P->p, (const float *)h.phi, n,
                               (const double *)P->scal, 0);
        else
            hipLaunchKernelGGL(cg_dir_phi_kernel<double>, dim3(sb), dim3(RB), 0, st, P->p, (const double *)h.phi, n,
                               (const double *)P->scal, 0, m2, P->x, split0<double>(P));
    }
    *iters_out = iters;
    *rnorm_io = rnorm;
    return status;
}

// MGPreconditionedCG solve!: pcg! with project_mean, definite = :negative,
// zero guess; b is the FP64 interior-sized source (scaled rows when rhs_scale)
int mg_pcg_solve(MGPlan *P, hipStream_t st, double *xout, const double *bin, double tol, int maxit, int *iters_out,
                 double *resid_out, double *bnorm_out) {
    MGLevelH &h = P->L[0];
    const int n = h.nx * h.ny * h.nz;
    const int fb = flat_blocks(n);
    double *b = P->Ap;  // the scaled source lives in Ap until the first apply
    hipMemcpyAsync(b, bin, sizeof(double) * n, hipMemcpyDeviceToDevice, st);
    if (P->rhs_scale)
        hipLaunchKernelGGL(scale_rows_kernel, dim3(stream_blocks(n)), dim3(RB), 0, st, b, (const double *)P->rhs_scale, h.nx * h.ny, n);
    // mb = mean(b); r = b − mb; x = 0; ‖b − mb‖
    mean_to<double>(P, st, b, n, 9);
    double mb = read_scal(st, P->scal + 9);
    hipLaunchKernelGGL(shift_copy_kernel, dim3(stream_blocks(n)), dim3(RB), 0, st, P->r, (const double *)b, n, mb);
    hipLaunchKernelGGL(fill_kernel, dim3(stream_blocks(n)), dim3(RB), 0, st, P->x, n, 0.0);
    hipLaunchKernelGGL(dot_kernel, dim3(fb), dim3(RB), 0, st, (const double *)P->r, (const double *)P->r, n, P->part);
    finalize_to(P, st, P->scal + 12, P->part, fb, 1.0);
    double b2 = read_scal(st, P->scal + 12);
    double bnorm = sqrt(b2);
    *bnorm_out = bnorm;
    if (bnorm == 0) {
        hipLaunchKernelGGL(fill_kernel, dim3(stream_blocks(n)), dim3(RB), 0, st, xout, n, 0.0);
        *iters_out = 0;
        *resid_out = 0;
        return 3;
    }
    double rnorm = sqrt(b2);
    int iters = 0;
    const int status = pcg_run(P, st, nullptr, tol, bnorm, maxit, &iters, &rnorm);
    // the solution's mean removed
    mean_to<double>(P, st, P->x, n, 13);
    double mx = read_scal(st, P->scal + 13);
    hipLaunchKernelGGL(shift_copy_kernel, dim3(stream_blocks(n)), dim3(RB), 0, st, xout, (const double *)P->x, n, mx);
    *iters_out = iters;
    *resid_out = rnorm;
    return status;
}

// pcg! (src/Backends.jl:1461-1591) with a caller's FP64 operator A in place of
// the plan's fine operator, the plan's V-cycle (FP64 or FP32 levels) as the
// preconditioner M, project_mean, definite = :negative, and the warm start of
// zero_guess = false (:1514, 1532-1536) when x0 is given. On return
// *resid_out is ‖r‖ of the recursion; with true_resid, *true_resid holds
// ‖(b − mean b) − A x‖ recomputed from the solution in FP64.
int mg_pcg_solve_op(MGPlan *P, hipStream_t st, const FCGOp &op, double *xout, const double *bin, const double *x0,
                    double tol, int maxit, int *iters_out, double *resid_out, double *bnorm_out, double *true_resid,
                    double *r0_out) {
    MGLevelH &h = P->L[0];
    const int n = h.nx * h.ny * h.nz;
    const int fb = flat_blocks(n);
    double *b = P->Ap;  // the source's copy lives in Ap until the first apply
    hipMemcpyAsync(b, bin, sizeof(double) * n, hipMemcpyDeviceToDevice, st);
    mean_to<double>(P, st, b, n, 9);
    const double mb = read_scal(st, P->scal + 9);
    hipLaunchKernelGGL(shift_copy_kernel, dim3(stream_blocks(n)), dim3(RB), 0, st, P->r, (const double *)b, n, mb);
    hipLaunchKernelGGL(dot_kernel, dim3(fb), dim3(RB), 0, st, (const double *)P->r, (const double *)P->r, n, P->part);
    finalize_to(P, st, P->scal + 12, P->part, fb, 1.0);
    const double bnorm = sqrt(read_scal(st, P->scal + 12));
    *bnorm_out = bnorm;
    if (bnorm == 0) {
        hipLaunchKernelGGL(fill_kernel, dim3(stream_blocks(n)), dim3(RB), 0, st, xout, n, 0.0);
        *iters_out = 0;
        *resid_out = 0;
        if (true_resid) *true_resid = 0;
        return 3;
    }
    if (x0) {
        hipMemcpyAsync(P->x, x0, sizeof(double) * n, hipMemcpyDeviceToDevice, st);
        op.apply(op.ctx, st, P->Ap, P->x);
        hipLaunchKernelGGL(sub_kernel, dim3(stream_blocks(n)), dim3(RB), 0, st, P->r, (const double *)P->Ap, n);
    } else {
        hipLaunchKernelGGL(fill_kernel, dim3(stream_blocks(n)), dim3(RB), 0, st, P->x, n, 0.0);
    }
    hipLaunchKernelGGL(dot_kernel, dim3(fb), dim3(RB), 0, st, (const double *)P->r, (const double *)P->r, n, P->part);
    finalize_to(P, st, P->scal + 12, P->part, fb, 1.0);
    double rnorm = sqrt(read_scal(st, P->scal + 12));
    if (r0_out) *r0_out = rnorm;
    int iters = 0;
    // the FP64 terrain preconditioner keeps its finest φ and b colour-split for
    // the solve (a level with a coarser one has even extents)
    P->half0 = P->gen0 && rb_cycle(P) && P->nlev > 1 ? (uint32_t)(n / 2) : 0u;
    P->half1 = P->half0 && P->gen1 ? (uint32_t)((size_t)P->L[1].nx * P->L[1].ny * P->L[1].nz / 2) : 0u;
    const int status = pcg_run(P, st, &op, tol, bnorm, maxit, &iters, &rnorm);
    P->half0 = P->half1 = 0;
    mean_to<double>(P, st, P->x, n, 13);
    const double mx = read_scal(st, P->scal + 13);
    hipLaunchKernelGGL(shift_copy_kernel, dim3(stream_blocks(n)), dim3(RB), 0, st, xout, (const double *)P->x, n, mx);
    if (true_resid) {
        // ‖(b − mb) − A x‖ from the returned x (FP64); b is re-read from bin
        op.apply(op.ctx, st, P->Ap, xout);
        hipLaunchKernelGGL(shift_copy_kernel, dim3(stream_blocks(n)), dim3(RB), 0, st, P->r, bin, n, mb);
        hipLaunchKernelGGL(sub_kernel, dim3(stream_blocks(n)), dim3(RB), 0, st, P->r, (const double *)P->Ap, n);
        hipLaunchKernelGGL(dot_kernel, dim3(fb), dim3(RB), 0, st, (const double *)P->r, (const double *)P->r, n,
                           P->part);
        finalize_to(P, st, P->scal + 12, P->part, fb, 1.0);
        *true_resid = sqrt(read_scal(st, P->scal + 12));
    }
    *iters_out = iters;
    *resid_out = rnorm;
    return status;
}

// plain multigrid cycles (mg_solve!, src/Multigrid.jl:801-845) with FP64 levels
// cycle = :V / :W and fmg of MultigridPoissonSolver (src/Multigrid.jl:559-570)
void mg_set_cycle(MGPlan *P, int wcycle, int fmg) {
    P->wcycle = wcycle;
    P->fmg = fmg;
}

void mg_set_terrain_coef(MGPlan *P, const TFWView &v) {
    const bool dims = P->coeff && P->L[0].nx == v.Nx && P->L[0].ny == v.Ny && P->L[0].nz == v.Nz;
    P->gm = make_tfm<double>(v);
    P->gmf = make_tfm<float>(v);
    // ρ̄ > 0 and J > 0 on every face, so every diagonal is negative
    P->open = P->open || dims;
    P->gen0 = dims && P->prec == 0 && P->smoother == 0;
    P->kc0 = chunk_tf_smooth(v.Nx, v.Ny, v.Nz);
    // the next level's sweeps likewise, with its φ and b colour-split, where
    // its coefficients, φ and b (40 B a cell) would stream from memory. A pass
    // at 256×256×128 (336 MB, past the 256 MB of the Infinity Cache): 86 us with
    // the stored coefficients, 36 from the metrics (and the transfers
    // below it 133 → 87 us); at 160×128×80 (66 MB) 14.4 and 13.9; at 108×100×76
    // (33 MB) 8.4 and 10.6, where the chunks' table costs more than it saves.
    const int nx1 = v.Nx / 2, ny1 = v.Ny / 2, nz1 = v.Nz / 2;
    P->gen1 = false;
    hipFree(P->tab1);
    P->tab1 = nullptr;
    if (P->gen0 && rb_cycle(P) && P->nlev > 2 && (size_t)nx1 * ny1 * nz1 >= TFC_MIN) {
        P->kc1 = chunk_tf_smooth(nx1, ny1, nz1);
        const int nch = (nz1 + P->kc1 - 1) / P->kc1;
        const size_t n = (size_t)(nx1 + 1) * (ny1 + 1) * (TFC_Q + TFC_V * (size_t)nch);
        if (hipMalloc(&P->tab1, sizeof(double) * n) == hipSuccess) {
            const LevelD<double> L = devlevel<double>(P, 1);
            hipLaunchKernelGGL(tf_table_kernel, dim3((nx1 + 64) / 64, ny1 + 1, nch), dim3(64), 0, 0, P->tab1, P->gm, nx1,
                               ny1, P->kc1, L.ix2, L.iy2, L.iz2);
            P->gen1 = hipDeviceSynchronize() == hipSuccess;
        } else {
            P->tab1 = nullptr;
            (void)hipGetLastError();
        }
    }
    P->gen0f = dims && P->prec == 1 && P->smoother == 1;
}

// _fmg_start! (src/Multigrid.jl:743-760), FP64 levels: the right-hand side
// restricted to every level (mean projected), the coarsest level solved,
// then at each finer level φ = prolongation of the coarse φ and one cycle
static void fmg_start(MGPlan *P, hipStream_t st) {
    for (int l = 0; l < P->nlev - 1; l++) {
        MGLevelH &h = P->L[l], &c = P->L[l + 1];
        const int n = h.nx * h.ny * h.nz, nc = c.nx * c.ny * c.nz;
        hipMemcpyAsync(h.r, h.b, sizeof(double) * n, hipMemcpyDeviceToDevice, st);
        LevelD<double> L = devlevel<double>(P, l), C = devlevel<double>(P, l + 1);
        const int nbc = nblocks3(c.nx, c.ny, c.nz);
        hipLaunchKernelGGL(restrict_kernel<double>, grid3(c.nx, c.ny, c.nz), dim3(RB), 0, st, C, L,
                           (const double *)nullptr, P->part);
        finalize_to(P, st, P->scal + 6, P->part, nbc, 1.0 / nc);
        hipLaunchKernelGGL(shift_kernel<double>, dim3(stream_blocks(nc)), dim3(RB), 0, st, (double *)c.b, nc,
                           P->scal + 6);
    }
    {
        MGLevelH &c = P->L[P->nlev - 1];
        const int nc = c.nx * c.ny * c.nz;
        hipLaunchKernelGGL(zero_kernel<double>, dim3(stream_blocks(nc)), dim3(RB), 0, st, (double *)c.phi, nc);
        vcycle<double>(P, st, P->nlev - 1, false);  // the coarsest level: _solve_coarsest!
    }
    for (int l = P->nlev - 2; l >= 0; l--) {
        MGLevelH &h = P->L[l];
        const int n = h.nx * h.ny * h.nz;
        hipLaunchKernelGGL(zero_kernel<double>, dim3(stream_blocks(n)), dim3(RB), 0, st, (double *)h.phi, n);
        LevelD<double> L = devlevel<double>(P, l), C = devlevel<double>(P, l + 1);
        hipLaunchKernelGGL(prolong_kernel<double>, grid3(h.nx, h.ny, h.nz), dim3(RB), 0, st, L, C, P->part,
                           (const double *)nullptr, (const double *)nullptr);
        vcycle<double>(P, st, l, false);
    }
}

int mg_cycles_solve(MGPlan *P, hipStream_t st, double *xout, const double *bin, double tol, int maxcycles,
                    int *cycles_out, double *rel_out) {
    if (P->prec != 0) return -1;
    MGLevelH &h = P->L[0];
    const int n = h.nx * h.ny * h.nz;
    const int fb = flat_blocks(n);
    hipMemcpyAsync(P->r, bin, sizeof(double) * n, hipMemcpyDeviceToDevice, st);
    if (P->rhs_scale)
        hipLaunchKernelGGL(scale_rows_kernel, dim3(stream_blocks(n)), dim3(RB), 0, st, P->r, (const double *)P->rhs_scale, h.nx * h.ny, n);
    // _load_rhs!: b = rhs − mean(rhs); φ = 0; ‖b‖
    mean_to<double>(P, st, P->r, n, 7);
    hipLaunchKernelGGL(load_rhs_kernel<double>, dim3(stream_blocks(n)), dim3(RB), 0, st, (double *)h.b, (const double *)P->r, n,
                       P->scal + 7);
    hipLaunchKernelGGL(zero_kernel<double>, dim3(stream_blocks(n)), dim3(RB), 0, st, (double *)h.phi, n);
    hipLaunchKernelGGL(sumsq_kernel<double>, dim3(fb), dim3(RB), 0, st, (const double *)h.b, n, P->part);
    finalize_to(P, st, P->scal, P->part, fb, 1.0);
    const double bn = sqrt(read_scal(st, P->scal));
    if (bn == 0) {
        hipLaunchKernelGGL(fill_kernel, dim3(stream_blocks(n)), dim3(RB), 0, st, xout, n, 0.0);
        *cycles_out = 0;
        *rel_out = 0;
        return 0;
    }
    if (P->fmg) fmg_start(P, st);
    double rel = 1;
    int ncyc = 0;
    const int nb3 = nblocks3(h.nx, h.ny, h.nz);
    for (int cyc = 1; cyc <= maxcycles; cyc++) {
        vcycle<double>(P, st, 0, false);
        // _residual_norm!: r, its mean removed, ‖r‖
        LevelD<double> L = devlevel<double>(P, 0);
        hipLaunchKernelGGL(residual_kernel<double>, grid3(h.nx, h.ny, h.nz), dim3(RB), 0, st, L, P->part,
                           (const double *)nullptr, (const double *)nullptr);
        finalize_to(P, st, P->scal + 5, P->part, nb3, 1.0 / n);
        hipLaunchKernelGGL(shift_kernel<double>, dim3(stream_blocks(n)), dim3(RB), 0, st, (double *)h.r, n, P->scal + 5);
        hipLaunchKernelGGL(sumsq_kernel<double>, dim3(fb), dim3(RB), 0, st, (const double *)h.r, n, P->part);
        finalize_to(P, st, P->scal, P->part, fb, 1.0);
        rel = sqrt(read_scal(st, P->scal)) / bn;
        ncyc = cyc;
        if (rel < tol) break;
    }
    // _store_solution!
    mean_to<double>(P, st, (const double *)h.phi, n, 8);
    hipLaunchKernelGGL(copyout_kernel<double>, dim3(fb), dim3(RB), 0, st, xout, (double *)h.phi, n, P->scal + 8);
    *cycles_out = ncyc;
    *rel_out = rel;
    return rel < tol ? 0 : 1;
}

// one V-cycle of the preconditioner on r (its mean removed first), z its
// mean-free result (_mg_precond!, src/Multigrid.jl:922-932); r and z may alias
void mg_precond_apply(MGPlan *P, hipStream_t st, double *z, const double *r) {
    MGLevelH &h = P->L[0];
    const int n = h.nx * h.ny * h.nz;
    if (r == z) {  // aliased: r is read after z is written, so it goes through the plan's r
        hipMemcpyAsync(P->r, r, sizeof(double) * n, hipMemcpyDeviceToDevice, st);
        r = P->r;
    }
    if (P->prec == 0) precond<double>(P, st, r, z); else precond<float>(P, st, r, z);
    if (P->prec != 0 || (rb_cycle(P) && P->nlev > 1)) {  // the cycle leaves z's mean in: remove it here
        mean_to<double>(P, st, z, n, 8);
        hipLaunchKernelGGL(shift_kernel<double>, dim3(stream_blocks(n)), dim3(RB), 0, st, z, n, P->scal + 8);
    }
}

// apply the fine FP64 operator (_apply_fine!, src/Multigrid.jl:911-917)
void mg_apply(MGPlan *P, hipStream_t st, double *out, const double *x) {
    MGLevelH &h = P->L[0];
    hipLaunchKernelGGL(cg_apply_kernel, grid3(h.nx, h.ny, h.nz), dim3(RB), 0, st, finelevel64(P), x, out, P->part);
}

}  // namespace aeo
