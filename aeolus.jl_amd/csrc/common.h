// Shared definitions of the gfx950 kernels of libaeolus_hip.
//
// Storage layout: the reference's (src/Grids.jl:98-140), a field is a
// column-major (Nx+2H) x (Ny+2H) x (Nz+2H) array, x fastest. Device code
// uses 0-based storage indices; the interior is H .. H+N-1 on every axis.
// Metric vectors are indexed by the 0-based storage level (the reference's
// 1-based level k is entry k-1 here).
#pragma once
#include <hip/hip_runtime.h>
#include <cfloat>
#include <cstdint>
#include <cstddef>

namespace aeo {

enum Loc { LOC_CC = 0, LOC_FX = 1, LOC_FY = 2, LOC_FZ = 3 };
enum Bc { BC_PERIODIC = 0, BC_NOFLUX = 1, BC_WALL = 2 };
enum Scheme {
    SCH_CENTERED = 0,  // Centered2 (advect_centered! / momentum_advect!)
    SCH_UPWIND1 = 1,   // _UpwindFirst
    SCH_WENO5 = 2,     // FiniteVolume._weno5_left (classic WENO-5, :weno5)
    SCH_WENO_JS5 = 3,  // weno_js5_left
    SCH_WENO_Z5 = 4,   // _weno_z5_left
    SCH_WENO_Z7 = 5,   // _weno_z7_left
    SCH_TENO5 = 6,     // _teno5_left (q = 6)
    SCH_TENO8 = 7,     // _teno8_left (q = 6)
    SCH_VARCONS = 8    // advect_variance_conserving! (not a reconstruction)
};

template <typename T> struct Eps;
template <> struct Eps<double> { static constexpr double v = DBL_EPSILON; };
template <> struct Eps<float> { static constexpr float v = FLT_EPSILON; };

// Grid metrics of one precision (src/FiniteVolume.jl:36-186).
template <typename T>
struct Metrics {
    int Nx, Ny, Nz, H;
    int sx, sy, sz;  // storage extents
    T idx, idy, idx2, idy2;
    int stretched;
    T idz, idz2;  // UniformZ
    T teno_ct;    // TENO cut-off C_T of the reconstructions that use one
    const T *idzc, *idzf, *wlo, *whi, *alo, *ahi;  // LevelZ (device)
    __device__ __forceinline__ T m_idz(int k) const { return stretched ? idzc[k] : idz; }
    __device__ __forceinline__ T m_idzf(int k) const { return stretched ? idzf[k] : idz; }
    __device__ __forceinline__ T m_zface(int k, T lo, T hi) const {
        return stretched ? wlo[k] * lo + whi[k] * hi : T(0.5) * (lo + hi);
    }
    __device__ __forceinline__ T m_zflux(int k, T lo, T hi) const {
        return stretched ? alo[k] * lo + ahi[k] * hi : T(0.5) * (lo + hi);
    }
    // the vertical term of the conservative Laplacian, _lapz (src/FiniteVolume.jl:166,177-181)
    __device__ __forceinline__ T m_lapz(int loc, int k, T fm, T c, T fp) const {
        if (!stretched) return ((fp - T(2) * c) + fm) * idz2;
        if (loc == LOC_FZ) return ((fp - c) * idzc[k] - (c - fm) * idzc[k - 1]) * idzf[k];
        return ((fp - c) * idzf[k + 1] - (c - fm) * idzf[k]) * idzc[k];
    }
};

// 32-bit element offsets: every storage array of the library holds fewer
// than 2^31 bytes (checked when a grid is created), so loads take the form
// uniform base pointer + 32-bit per-lane offset.
// XCD-aware block order for a 3-D grid whose blocks read their z-neighbours'
// data: MI355X hands workgroups to its 8 XCDs (each with its own L2) in turn
// by linear id, so neighbouring-z blocks of one tile would land on different
// L2s. With nb % 8 == 0 the linear id is remapped so that XCD x takes the
// contiguous logical range [x·nb/8, (x+1)·nb/8), ordered z fastest, then x,
// then y: the blocks that share a tile's planes run together on one L2.
// Writes the logical (bx, by, bz); otherwise the hardware's own.
__device__ __forceinline__ void xcd_block3(int &bx, int &by, int &bz) {
    const uint32_t gx = gridDim.x, gy = gridDim.y, gz = gridDim.z;
    const uint32_t nb = gx * gy * gz;
    const uint32_t id = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    if (nb % 8 != 0) {
        bx = blockIdx.x; by = blockIdx.y; bz = blockIdx.z;
        return;
    }
    const uint32_t l = (id % 8) * (nb / 8) + id / 8;
    bz = (int)(l % gz);
    bx = (int)((l / gz) % gx);
    by = (int)(l / (gz * gx));
}

// Levels per chunk of a kernel whose blocks march `tiles` columns of nz
// levels: a block costs its kc levels and about `start` more (the first
// level's windows and faces), and the chip takes `fill` blocks a round. On a
// large grid that is the longest chunk, kmax; on a small one, chunks short
// enough to occupy the chip. The length is a multiple of `step`, or nz.
inline int chunk_levels(int tiles, int nz, int kmax, int fill, int start, int step = 1) {
    int best = nz;
    long long cost = -1;
    for (int kc = step; kc <= kmax && kc <= nz; kc += step) {
        const long long blocks = (long long)tiles * ((nz + kc - 1) / kc);
        const long long c = (blocks + fill - 1) / fill * (kc + start);
        if (cost < 0 || c <= cost) { cost = c; best = kc; }
    }
    return best;
}

__device__ __forceinline__ uint32_t lin(int i, int j, int k, int sx, int sy) {
    return (uint32_t)i + (uint32_t)sx * ((uint32_t)j + (uint32_t)sy * (uint32_t)k);
}

// ---------------------------------------------------------------------------
// Reconstructions, in the reference's evaluation order (WENO-Z5 and Z7
// excepted: their own form below). The library is built
// with -ffp-contract=off; the reconstructions (and the tendency kernel, which
// turns the same pragma on for its file) let the compiler fuse a multiply and
// an add into one FMA: each fused pair rounds once instead of twice (at most
// an ulp from the unfused value; the FP64 parity bound is 1e-12), and the
// FP64 WENO-Z kernel issues 15 % fewer FP64 instructions. Sums of squares
// stay non-negative: fma(a, a, x) with x ≥ 0 is ≥ 0.
#pragma clang fp contract(fast)
// ---------------------------------------------------------------------------
// RN(x/3) without a division: q = RN(x·r), r = RN(1/3); the remainder
// x − 3q is exact in one FMA and RN(q + (x − 3q)·r) is RN(x/3). x/3 is never
// a rounding midpoint and lies at least ulp/6 from one, while the corrected
// sum is within ~2^-54 ulp of x/3, so the final rounding is the correct one
// (finite x above the subnormal range). x/6, x/12, x/24 are this times an
// exact power of two.
template <typename T> __device__ __forceinline__ T div3(T x) {
    const T r = T(1.0 / 3.0);
    T q = x * r;
    T e = fma(T(-3), q, x);
    return fma(e, r, q);
}
template <typename T> __device__ __forceinline__ T div6(T x) { return div3<T>(x) * T(0.5); }
template <typename T> __device__ __forceinline__ T div12(T x) { return div3<T>(x) * T(0.25); }
template <typename T> __device__ __forceinline__ T div24(T x) { return div3<T>(x) * T(0.125); }

template <typename T> __device__ __forceinline__ T beta3(T a1, T a2) { return a1 * a1 + T(13.0 / 3.0) * (a2 * a2); }
template <typename T> __device__ __forceinline__ T beta4(T a1, T a2, T a3) {
    return ((a1 * a1 + T(1.0 / 2.0) * (a1 * a3)) + T(13.0 / 3.0) * (a2 * a2)) + T(3129.0 / 80.0) * (a3 * a3);
}
template <typename T> __device__ __forceinline__ T b3_m2(T v1, T v2, T v3) {
    return beta3<T>(((v1 - T(4) * v2) + T(3) * v3) / T(2), ((v1 - T(2) * v2) + v3) / T(2));
}
template <typename T> __device__ __forceinline__ T b3_m1(T v1, T v2, T v3) {
    return beta3<T>((v3 - v1) / T(2), ((v1 - T(2) * v2) + v3) / T(2));
}
template <typename T> __device__ __forceinline__ T b3_p0(T v1, T v2, T v3) {
    return beta3<T>(((T(-3) * v1 + T(4) * v2) - v3) / T(2), ((v1 - T(2) * v2) + v3) / T(2));
}
template <typename T> __device__ __forceinline__ T b4_m3(T v1, T v2, T v3, T v4) {
    return beta4<T>(div24<T>(((T(-7) * v1 + T(33) * v2) - T(69) * v3) + T(43) * v4),
                    (((-v1 + T(4) * v2) - T(5) * v3) + T(2) * v4) / T(2), div6<T>(((-v1 + T(3) * v2) - T(3) * v3) + v4));
}
template <typename T> __device__ __forceinline__ T b4_p0(T v1, T v2, T v3, T v4) {
    return beta4<T>(div24<T>(((T(-43) * v1 + T(69) * v2) - T(33) * v3) + T(7) * v4),
                    (((T(2) * v1 - T(5) * v2) + T(4) * v3) - v4) / T(2), div6<T>(((-v1 + T(3) * v2) - T(3) * v3) + v4));
}
// General divisions of the nonlinear weights. The divisors are β + ε ≥ ε > 0
// or sums of positive weights: positive, normal and finite.
//  FP64: a · (1/b) with 1/b from v_rcp_f64 refined by one third-order step
//        (e = 1 − b·r, r ← r + r·(e + e²)): within 1.49 ulp of the correctly
//        rounded quotient, as with two Newton steps of one instruction more
//        (checked on 2e7 random pairs with the initial reciprocal perturbed
//        by up to 2^-22: e³ = 2^-66); the tests hold the kernels to 1e-12.
//  FP32: a · v_rcp_f32(b) (≤ 1 ulp of 1/b), stated against the FP64 oracle.
template <typename T> __device__ __forceinline__ T qdiv(T a, T b);
template <> __device__ __forceinline__ double qdiv<double>(double a, double b) {
    double r = __builtin_amdgcn_rcp(b);
    const double e = __builtin_fma(-b, r, 1.0);
    r = __builtin_fma(__builtin_fma(e, e, e), r, r);
    return a * r;
}
template <> __device__ __forceinline__ float qdiv<float>(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }

template <int P, typename T> __device__ __forceinline__ T ipow(T x) {
    if constexpr (P == 2) return x * x;
    else if constexpr (P == 6) {  // _ipow(x, Val(6)): x³·x³
        const T x3 = (x * x) * x;
        return x3 * x3;
    } else return x;
}

template <typename T> __device__ __forceinline__ T beta5(T a1, T a2, T a3, T a4) {
    return ((((a1 * a1 + T(1.0 / 2.0) * (a1 * a3)) + T(13.0 / 3.0) * (a2 * a2)) + T(21.0 / 5.0) * (a2 * a4)) +
            T(3129.0 / 80.0) * (a3 * a3)) +
           T(87617.0 / 140.0) * (a4 * a4);
}
// _b5_m4, src/AdvectionSchemes.jl:143-147 ({i-4, …, i}); x/48 = (x/3)/16, x/16 exact
template <typename T> __device__ __forceinline__ T b5_m4(T v1, T v2, T v3, T v4, T v5) {
    return beta5<T>(div3<T>((((T(9) * v1 - T(50) * v2) + T(120) * v3) - T(174) * v4) + T(95) * v5) * T(1.0 / 16.0),
                    ((((T(7) * v1 - T(36) * v2) + T(74) * v3) - T(68) * v4) + T(23) * v5) / T(16),
                    div12<T>((((T(3) * v1 - T(14) * v2) + T(24) * v3) - T(18) * v4) + T(5) * v5),
                    div24<T>((((v1 - T(4) * v2) + T(6) * v3) - T(4) * v4) + v5));
}

// 2^(K − e) from the high word of a double m·2^e, 1 ≤ m < 2 (positive, below 2^1022)
template <int K> __device__ __forceinline__ double pow2_over(int hi) {
    return __hiloint2double(0x7fe00000 + (K << 20) - (hi & 0x7ff00000), 0);
}

// _weno_z5_left, src/AdvectionSchemes.jl:240-255, from the differences
// e_m = v_{m+1} − v_m: the smoothness indicators (times 4, with ε² times 4)
// and the candidates less v3 (times 6) depend on nothing else, and the face is
// v3 + Σ a_k (6 (q_k − v3)) / (6 Σ a_k); it rounds relative to the variation,
// not the value.
// FP64: the weights a_k = g_k (1 + (τ/b_k)²) times (b0 b1 b2)², so that only
// the face divides. Such a product of indicators would end at variations of
// 1e51, so they are first scaled to 2^80 by the larger of b0 and b2 (b1 is at
// most 5.4 times it), and no sum passes 1e151. Where one is so small that the
// product vanishes, τ is either at least 2^-53 of the larger one, and the
// weight of the small one, without the product, is what counts, or zero, and
// the weights are the linear ones (w = 1). The range is that of one division
// per ratio: ratios whose square is finite. FP32: three hardware reciprocals.
// The reconstruction bounds the advection kernels. 256×256×128 RK3 stage with
// the indicators and candidates from the values 606 us, from differences 506
// (FP32 289 → 265); the limited tracer's two passes 316 → 278. A branch from
// one reciprocal of the product to one per ratio where it overflows: 122
// registers spilled, the step 2.49 → 4.59 ms.
template <int P, typename T>
__device__ __forceinline__ T weno_z5(T v1, T v2, T v3, T v4, T v5) {
    const T e1 = v2 - v1, e2 = v3 - v2, e3 = v4 - v3, e4 = v5 - v4;
    const T s0 = e2 - e1, s1 = e3 - e2, s2 = e4 - e3;                      // second differences
    const T f0 = T(3) * e2 - e1, f1 = e2 + e3, f2 = T(3) * e3 - e4;        // twice the slopes at v3
    const T c = T(13.0 / 3.0), eps = T(4) * Eps<T>::v * Eps<T>::v;
    const T b0 = f0 * f0 + ((c * s0) * s0 + eps), b1 = f1 * f1 + ((c * s1) * s1 + eps),
            b2 = f2 * f2 + ((c * s2) * s2 + eps);
    const T p0 = T(5) * e2 - T(2) * e1, p1 = T(2) * e3 + e2, p2 = T(4) * e3 - e4;
    if constexpr (sizeof(T) == 8) {
        const T r = pow2_over<80>(max(__double2hiint(b0), __double2hiint(b2)));
        const T c0 = b0 * r, c2 = b2 * r, tau = fabs(c0 - c2), c1 = b1 * r, c02 = c0 * c2;
        T w = ipow<P>(c02 * c1);
        w = __hiloint2double(tau == T(0) ? 0x3ff00000 : __double2hiint(w), __double2loint(w));
        const T tc = tau * c1, z0 = w + ipow<P>(tc * c2), z1 = w + ipow<P>(tau * c02), z2 = w + ipow<P>(tc * c0);
        const T a1 = T(6) * z1, a2 = T(3) * z2;
        return v3 + qdiv<T>((z0 * p0 + a1 * p1) + a2 * p2, T(6) * ((z0 + a1) + a2));
    } else {
        const T tau = fabs(b0 - b2);
        const T a0 = T(1.0 / 10.0) + T(1.0 / 10.0) * ipow<P>(qdiv<T>(tau, b0));
        const T a1 = T(6.0 / 10.0) + T(6.0 / 10.0) * ipow<P>(qdiv<T>(tau, b1));
        const T a2 = T(3.0 / 10.0) + T(3.0 / 10.0) * ipow<P>(qdiv<T>(tau, b2));
        return v3 + qdiv<T>((a0 * p0 + a1 * p1) + a2 * p2, T(6) * ((a0 + a1) + a2));
    }
}
// _weno_z7_left, src/AdvectionSchemes.jl:284-303, from the differences like
// weno_z5: 36 b_k = D_k² + 39 B_k² + 39.05 C_k² with D_k six times the slope
// plus a quarter, B_k the second and C_k the third differences of the
// candidate's four cells (beta4's form with its square completed), and the
// candidates less v4 times 12. FP64: a reciprocal per two indicators, one of
// each pair and τ scaled by the larger of b0 and b2 so that their product
// stays in range; where it would vanish, 1e-307 in its place leaves the pair's
// ratio to each other, and both far above the other pair's (or τ zero). FP32:
// one reciprocal each. At 187×141×75 32.6 → 24.6 us in FP32, 62.6 → 49.7 in
// FP64 (48.6 without the scaling, finite up to 1e75 only).
template <int P, typename T>
__device__ __forceinline__ T weno_z7(T v1, T v2, T v3, T v4, T v5, T v6, T v7) {
    const T e1 = v2 - v1, e2 = v3 - v2, e3 = v4 - v3, e4 = v5 - v4, e5 = v6 - v5, e6 = v7 - v6;
    const T s1 = e2 - e1, s2 = e3 - e2, s3 = e4 - e3, s4 = e5 - e4, s5 = e6 - e5;
    const T c0 = s2 - s1, c1 = s3 - s2, c2 = s4 - s3, c3 = s5 - s4;
    const T f0 = T(2) * s2 - s1, f3 = T(2) * s4 - s5;
    const T d0 = T(11) * e3 + (T(2) * e1 - T(7) * e2), d1 = T(2) * e4 + (T(5) * e3 - e2);
    const T d2 = T(2) * e3 + (T(5) * e4 - e5), d3 = T(11) * e4 + (T(2) * e6 - T(7) * e5);
    const T g = T(39), h = T(39.05), eps = T(36) * Eps<T>::v * Eps<T>::v;
    const T m = (g * s3) * s3 + eps;
    const T b0 = d0 * d0 + ((h * c0) * c0 + ((g * f0) * f0 + eps)), b1 = d1 * d1 + ((h * c1) * c1 + m);
    const T b2 = d2 * d2 + ((h * c2) * c2 + m), b3 = d3 * d3 + ((h * c3) * c3 + ((g * f3) * f3 + eps));
    const T tau = fabs(((b0 - b1) - b2) + b3);
    T t0, t1, t2, t3;
    if constexpr (sizeof(T) == 8) {
        const T n = pow2_over<0>(max(__double2hiint(b0), __double2hiint(b2))), taun = tau * n;
        const T r = qdiv<T>(taun, fma(b0 * n, b1, T(1e-307))), q = qdiv<T>(taun, fma(b2 * n, b3, T(1e-307)));
        t0 = b1 * r; t1 = b0 * r;
        t2 = b3 * q; t3 = b2 * q;
    } else {
        t0 = qdiv<T>(tau, b0); t1 = qdiv<T>(tau, b1);
        t2 = qdiv<T>(tau, b2); t3 = qdiv<T>(tau, b3);
    }
    // the weights over 16: twelve times their sum is then below what a ratio's square reaches
    const T g0 = T(1.0 / 560.0), g1 = T(12.0 / 560.0), g2 = T(18.0 / 560.0), g3 = T(4.0 / 560.0);
    const T a0 = g0 + g0 * ipow<P>(t0), a1 = g1 + g1 * ipow<P>(t1);
    const T a2 = g2 + g2 * ipow<P>(t2), a3 = g3 + g3 * ipow<P>(t3);
    const T p0 = T(13) * e3 + (T(3) * e1 - T(10) * e2), p1 = T(3) * e4 + (T(4) * e3 - e2);
    const T p2 = T(6) * e4 + (e3 - e5), p3 = T(9) * e4 + (e6 - T(4) * e5);
    return v4 + qdiv<T>(((a0 * p0 + a1 * p1) + a2 * p2) + a3 * p3, T(12) * (((a0 + a1) + a2) + a3));
}
// _teno5_left, src/AdvectionSchemes.jl:405-427 (q = 6, cut-off ct). The
// cut-off g_k/Σg < C_T is a discrete choice of stencils: it is taken with an
// IEEE division so that the same candidates survive as in the reference.
template <typename T>
__device__ __forceinline__ T teno5(T v1, T v2, T v3, T v4, T v5, T ct) {
    T q0 = div6<T>((T(2) * v1 - T(7) * v2) + T(11) * v3);
    T q1 = div6<T>((-v2 + T(5) * v3) + T(2) * v4);
    T q2 = div6<T>((T(2) * v3 + T(5) * v4) - v5);
    T b0 = b3_m2<T>(v1, v2, v3), b1 = b3_m1<T>(v2, v3, v4), b2 = b3_p0<T>(v3, v4, v5);
    const T eps = Eps<T>::v * Eps<T>::v;
    T tau = fabs(b0 - b2);
    T g0 = ipow<6>(T(1) + qdiv<T>(tau, b0 + eps));
    T g1 = ipow<6>(T(1) + qdiv<T>(tau, b1 + eps));
    T g2 = ipow<6>(T(1) + qdiv<T>(tau, b2 + eps));
    T gs = (g0 + g1) + g2;
    T d0 = g0 / gs < ct ? T(0) : T(1.0 / 10.0);
    T d1 = g1 / gs < ct ? T(0) : T(6.0 / 10.0);
    T d2 = g2 / gs < ct ? T(0) : T(3.0 / 10.0);
    return qdiv<T>((d0 * q0 + d1 * q1) + d2 * q2, (d0 + d1) + d2);
}
// _teno8_left, src/AdvectionSchemes.jl:456-495 (q = 6, cut-off ct)
template <typename T>
__device__ __forceinline__ T teno8(T v1, T v2, T v3, T v4, T v5, T v6, T v7, T v8, T ct) {
    T q0 = div6<T>((T(2) * v3 - T(7) * v4) + T(11) * v5);
    T q1 = div6<T>((-v4 + T(5) * v5) + T(2) * v6);
    T q2 = div6<T>((T(2) * v5 + T(5) * v6) - v7);
    T q3 = div12<T>(((T(-3) * v2 + T(13) * v3) - T(23) * v4) + T(25) * v5);
    T q4 = div12<T>(((T(3) * v5 + T(13) * v6) - T(5) * v7) + v8);
    T q5 = ((((T(12) * v1 - T(63) * v2) + T(137) * v3) - T(163) * v4) + T(137) * v5) / T(60);
    T b0 = b3_m2<T>(v3, v4, v5), b1 = b3_m1<T>(v4, v5, v6), b2 = b3_p0<T>(v5, v6, v7);
    T b3 = b4_m3<T>(v2, v3, v4, v5), b4 = b4_p0<T>(v5, v6, v7, v8), b5 = b5_m4<T>(v1, v2, v3, v4, v5);
    const T eps = Eps<T>::v * Eps<T>::v;
    T tau = fabs(b5 - div6<T>((b0 + T(4) * b1) + b2));
    T g0 = ipow<6>(T(1) + qdiv<T>(tau, b0 + eps));
    T g1 = ipow<6>(T(1) + qdiv<T>(tau, b1 + eps));
    T g2 = ipow<6>(T(1) + qdiv<T>(tau, b2 + eps));
    T g3 = ipow<6>(T(1) + qdiv<T>(tau, b3 + eps));
    T g4 = ipow<6>(T(1) + qdiv<T>(tau, b4 + eps));
    T g5 = ipow<6>(T(1) + qdiv<T>(tau, b5 + eps));
    T gs = ((((g0 + g1) + g2) + g3) + g4) + g5;
    T d0 = g0 / gs < ct ? T(0) : T(3.0 / 28.0);
    T d1 = g1 / gs < ct ? T(0) : T(15.0 / 28.0);
    T d2 = g2 / gs < ct ? T(0) : T(3.0 / 14.0);
    T d3 = g3 / gs < ct ? T(0) : T(3.0 / 56.0);
    T d4 = g4 / gs < ct ? T(0) : T(1.0 / 14.0);
    T d5 = g5 / gs < ct ? T(0) : T(1.0 / 56.0);
    return qdiv<T>(((((d0 * q0 + d1 * q1) + d2 * q2) + d3 * q3) + d4 * q4) + d5 * q5,
                   ((((d0 + d1) + d2) + d3) + d4) + d5);
}
// weno_js5_left, src/AdvectionSchemes.jl:319-342 (ε = 1e-6)
template <typename T>
__device__ __forceinline__ T weno_js5(T v1, T v2, T v3, T v4, T v5) {
    T q0 = div6<T>((T(2) * v1 - T(7) * v2) + T(11) * v3);
    T q1 = div6<T>((-v2 + T(5) * v3) + T(2) * v4);
    T q2 = div6<T>((T(2) * v3 + T(5) * v4) - v5);
    T b0 = b3_m2<T>(v1, v2, v3), b1 = b3_m1<T>(v2, v3, v4), b2 = b3_p0<T>(v3, v4, v5);
    const T e = T(1e-6);
    T d0 = b0 + e, d1 = b1 + e, d2 = b2 + e;
    T a0 = qdiv<T>(T(1.0 / 10.0), d0 * d0), a1 = qdiv<T>(T(6.0 / 10.0), d1 * d1), a2 = qdiv<T>(T(3.0 / 10.0), d2 * d2);
    return qdiv<T>((a0 * q0 + a1 * q1) + a2 * q2, (a0 + a1) + a2);
}
// FiniteVolume._weno5_left, src/FiniteVolume.jl:1582-1596
template <typename T>
__device__ __forceinline__ T weno5_classic(T fm2, T fm1, T fc, T fp1, T fp2) {
    T q0 = (T(1.0 / 3.0) * fm2 - T(7.0 / 6.0) * fm1) + T(11.0 / 6.0) * fc;
    T q1 = (T(-1.0 / 6.0) * fm1 + T(5.0 / 6.0) * fc) + T(1.0 / 3.0) * fp1;
    T q2 = (T(1.0 / 3.0) * fc + T(5.0 / 6.0) * fp1) - T(1.0 / 6.0) * fp2;
    T t0 = (fm2 - T(2) * fm1) + fc, s0 = (fm2 - T(4) * fm1) + T(3) * fc;
    T t1 = (fm1 - T(2) * fc) + fp1, s1 = fm1 - fp1;
    T t2 = (fc - T(2) * fp1) + fp2, s2 = (T(3) * fc - T(4) * fp1) + fp2;
    T b0 = T(13.0 / 12.0) * (t0 * t0) + T(1.0 / 4.0) * (s0 * s0);
    T b1 = T(13.0 / 12.0) * (t1 * t1) + T(1.0 / 4.0) * (s1 * s1);
    T b2 = T(13.0 / 12.0) * (t2 * t2) + T(1.0 / 4.0) * (s2 * s2);
    const T e = T(1e-6);
    T d0 = b0 + e, d1 = b1 + e, d2 = b2 + e;
    T a0 = qdiv<T>(T(1.0 / 10.0), d0 * d0), a1 = qdiv<T>(T(6.0 / 10.0), d1 * d1), a2 = qdiv<T>(T(3.0 / 10.0), d2 * d2);
    T s = (a0 + a1) + a2;
    return qdiv<T>((a0 * q0 + a1 * q1) + a2 * q2, s);
}

// Stencil half-width of a scheme: the face between cells c and c+1 reads
// c-R+1 .. c+R (the union of the left- and right-biased stencils).
template <int S> struct SchemeInfo { static constexpr int R = 3; };
template <> struct SchemeInfo<SCH_CENTERED> { static constexpr int R = 1; };
template <> struct SchemeInfo<SCH_UPWIND1> { static constexpr int R = 1; };
template <> struct SchemeInfo<SCH_WENO_Z7> { static constexpr int R = 4; };
template <> struct SchemeInfo<SCH_TENO8> { static constexpr int R = 5; };

// A load at a byte offset from a field's base. Offsets are 32-bit (every
// array is below 2 GiB): with the base in SGPRs the load takes one VGPR of
// address instead of a 64-bit pointer per load site.
template <typename T> __device__ __forceinline__ T ldo(const T *__restrict__ p, uint32_t off) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + off);
}
template <typename T> __device__ __forceinline__ void sto(T *__restrict__ p, uint32_t off, T v) {
    *reinterpret_cast<T *>(reinterpret_cast<char *>(p) + off) = v;
}

// The upwinded face value at the interface between cells c and c+1 along an
// axis, read from d at byte offsets o0 + m*st, o0 being cell c-R+1 (the
// first cell of the union of the left- and right-biased stencils): the
// left-biased stencil for vel >= 0, else the mirrored right-biased one, into
// one left reconstruction (_upwind_value, src/AdvectionSchemes.jl:659-666).
template <int S, int P, typename T>
__device__ __forceinline__ T face_value(const T *__restrict__ d, uint32_t o0, uint32_t st, T vel, T ct) {
    if constexpr (S == SCH_CENTERED) {
        return (ldo(d, o0) + ldo(d, o0 + st)) / T(2);
    } else if constexpr (S == SCH_UPWIND1) {
        return vel >= T(0) ? ldo(d, o0) : ldo(d, o0 + st);
    } else {
        constexpr int R = SchemeInfo<S>::R;
        const bool up = vel >= T(0);
        // the left-biased stencil (vel >= 0) or the mirrored right-biased one,
        // selected pair by pair (t[m] = up ? a[m] : a[2R-1-m])
        T t[2 * R - 1];
        if constexpr (R == 3) {
            const T a0 = ldo(d, o0), a1 = ldo(d, o0 + st), a2 = ldo(d, o0 + 2 * st), a3 = ldo(d, o0 + 3 * st),
                    a4 = ldo(d, o0 + 4 * st), a5 = ldo(d, o0 + 5 * st);
            t[0] = up ? a0 : a5; t[1] = up ? a1 : a4; t[2] = up ? a2 : a3; t[3] = up ? a3 : a2; t[4] = up ? a4 : a1;
        } else if constexpr (R == 4) {
            const T a0 = ldo(d, o0), a1 = ldo(d, o0 + st), a2 = ldo(d, o0 + 2 * st), a3 = ldo(d, o0 + 3 * st),
                    a4 = ldo(d, o0 + 4 * st), a5 = ldo(d, o0 + 5 * st), a6 = ldo(d, o0 + 6 * st),
                    a7 = ldo(d, o0 + 7 * st);
            t[0] = up ? a0 : a7; t[1] = up ? a1 : a6; t[2] = up ? a2 : a5; t[3] = up ? a3 : a4;
            t[4] = up ? a4 : a3; t[5] = up ? a5 : a2; t[6] = up ? a6 : a1;
        } else {
            // TENO8: the left stencil is cells c-4..c+3, the mirrored right one c+5..c-2
            T a[10];
#pragma unroll
            for (int m = 0; m < 10; m++) a[m] = ldo(d, o0 + (uint32_t)m * st);
#pragma unroll
            for (int m = 0; m < 8; m++) t[m] = up ? a[m] : a[9 - m];
        }
        if constexpr (S == SCH_WENO5) return weno5_classic<T>(t[0], t[1], t[2], t[3], t[4]);
        else if constexpr (S == SCH_WENO_JS5) return weno_js5<T>(t[0], t[1], t[2], t[3], t[4]);
        else if constexpr (S == SCH_WENO_Z5) return weno_z5<P, T>(t[0], t[1], t[2], t[3], t[4]);
        else if constexpr (S == SCH_TENO5) return teno5<T>(t[0], t[1], t[2], t[3], t[4], ct);
        else if constexpr (S == SCH_TENO8) return teno8<T>(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], ct);
        else return weno_z7<P, T>(t[0], t[1], t[2], t[3], t[4], t[5], t[6]);
    }
}

// One pair of the upwind selection: the two values pass through an empty asm
// so that the select stays a per-lane choice between two registers (a select
// between two reads of one local array is otherwise folded into a read at a
// selected index, which lowers to a compare-and-select chain per value).
template <typename T> __device__ __forceinline__ T pick(bool up, T x, T y) {
    asm volatile("" : "+v"(x), "+v"(y));
    return up ? x : y;
}

// face_value from the values a[m] of cells c-R+1+m, m = 0 .. 2R-1 (registers
// or a tile in LDS), with the same selection and reconstruction
template <int S, int P, typename T>
__device__ __forceinline__ T face_of(const T *a, T vel, T ct) {
    if constexpr (S == SCH_CENTERED) {
        return (a[0] + a[1]) / T(2);
    } else if constexpr (S == SCH_UPWIND1) {
        return pick(vel >= T(0), a[0], a[1]);
    } else {
        constexpr int R = SchemeInfo<S>::R;
        const bool up = vel >= T(0);
        constexpr int NT = S == SCH_TENO8 ? 8 : 2 * R - 1;
        T t[NT];
#pragma unroll
        for (int m = 0; m < NT; m++) t[m] = pick(up, a[m], a[2 * R - 1 - m]);
        if constexpr (S == SCH_WENO5) return weno5_classic<T>(t[0], t[1], t[2], t[3], t[4]);
        else if constexpr (S == SCH_WENO_JS5) return weno_js5<T>(t[0], t[1], t[2], t[3], t[4]);
        else if constexpr (S == SCH_WENO_Z5) return weno_z5<P, T>(t[0], t[1], t[2], t[3], t[4]);
        else if constexpr (S == SCH_TENO5) return teno5<T>(t[0], t[1], t[2], t[3], t[4], ct);
        else if constexpr (S == SCH_TENO8) return teno8<T>(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], ct);
        else return weno_z7<P, T>(t[0], t[1], t[2], t[3], t[4], t[5], t[6]);
    }
}

// |∇·u| of one cell (_div_at, src/FiniteVolume.jl:312-315), shared by the
// diagnostics kernels so that every reduction of it sees the same bits
template <typename T>
__device__ __forceinline__ double cell_abs_div(const T *u, const T *v, const T *w, size_t c, size_t sx, size_t sxy,
                                               const Metrics<double> &md, int K) {
    const double du = (double)u[c + 1] - (double)u[c];
    const double dv = (double)v[c + sx] - (double)v[c];
    const double dw = (double)w[c + sxy] - (double)w[c];
    return fabs((du * md.idx + dv * md.idy) + dw * md.m_idz(K));
}

// contraction ends with the reconstructions: the sources that include this
// header keep -ffp-contract=off unless they opt in themselves
#pragma clang fp contract(off)

}  // namespace aeo
