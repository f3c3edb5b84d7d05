// Stencil kernels of the dynamical-core step (gfx950).
//
//   halo_gather      fill_halos! of one field in one launch
//   adv_march        advection tendencies (WENO-5/WENO-JS5/WENO-Z5/WENO-Z7,
//                    centred, upwind), fused with the viscous term, the
//                    buoyancy, the surface flux and the predictor
//   div_into         the Arakawa-C divergence into the solver's buffer
//   correct          the projection's correction + RK3 combination + p
//   shell_combine    the RK3 combination of the halo shell
//   reductions       max |div|, max advective rate
#include "kernels.h"

// multiply-add pairs may fuse into FMAs here (the reconstructions in common.h
// do the same); every other source keeps -ffp-contract=off
#pragma clang fp contract(fast)

namespace aeo {

// ---------------------------------------------------------------------------
// Halo fill (src/BoundaryConditions.jl:182-259; halo_kernels.jl:100-147).
// The reference fills x, then y, then z, each over the whole face slab; the
// result at any storage point is the interior value at (mx(i), my(j), mz(k))
// (periodic wrap or mirror per axis), negated about a wall for w in z, with
// the wall faces themselves zero. Every source is interior, so one gather
// launch over the halo points (and the wall plane) gives the same values.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int map_axis(int idx, int H, int N, int bc) {
    if (idx < H) return bc == BC_PERIODIC ? idx + N : 2 * H - 1 - idx;
    if (idx >= H + N) return bc == BC_PERIODIC ? idx - N : 2 * (H + N) - 1 - idx;
    return idx;
}

template <typename T>
__device__ __forceinline__ void halo_gather_body(T *__restrict__ d, int Nx, int Ny, int Nz, int H, int bcx, int bcy,
                                                 int bcz, int wall_w) {
    const int sx = Nx + 2 * H, sy = Ny + 2 * H, sz = Nz + 2 * H;
    // enumeration: z-slabs (2H planes), then y-slabs, then x-slabs, then the
    // w wall plane k = H (interior) when wall_w
    const uint32_t nz_slab = (uint32_t)2 * H * sx * sy;
    const uint32_t ny_slab = (uint32_t)Nz * 2 * H * sx;
    const uint32_t nx_slab = (uint32_t)Nz * Ny * 2 * H;
    const uint32_t nwall = wall_w ? (uint32_t)sx * sy : 0;
    const uint32_t total = nz_slab + ny_slab + nx_slab + nwall;
    for (uint32_t t = blockIdx.x * (uint32_t)blockDim.x + threadIdx.x; t < total; t += (uint32_t)gridDim.x * blockDim.x) {
        int i, j, k;
        if (t < nz_slab) {
            uint32_t q = t;
            i = (int)(q % sx); q /= sx;
            j = (int)(q % sy); q /= sy;
            int l = (int)q;
            k = l < H ? l : H + Nz + (l - H);
        } else if (t < nz_slab + ny_slab) {
            uint32_t q = t - nz_slab;
            i = (int)(q % sx); q /= sx;
            int l = (int)(q % (2 * H)); q /= (2 * H);
            j = l < H ? l : H + Ny + (l - H);
            k = H + (int)q;
        } else if (t < nz_slab + ny_slab + nx_slab) {
            uint32_t q = t - nz_slab - ny_slab;
            int l = (int)(q % (2 * H)); q /= (2 * H);
            i = l < H ? l : H + Nx + (l - H);
            j = H + (int)(q % Ny);
            k = H + (int)(q / Ny);
        } else {
            uint32_t q = t - nz_slab - ny_slab - nx_slab;
            i = (int)(q % sx);
            j = (int)(q / sx);
            k = H;
        }
        T val;
        if (wall_w && bcz == BC_WALL) {
            if (k == H || k == H + Nz) {
                val = T(0);
            } else {
                int kk = k;
                T sgn = T(1);
                if (k < H) { kk = 2 * H - k; sgn = T(-1); }
                else if (k > H + Nz) { kk = 2 * (H + Nz) - k; sgn = T(-1); }
                int ii = map_axis(i, H, Nx, bcx), jj = map_axis(j, H, Ny, bcy);
                val = sgn < T(0) ? -d[lin(ii, jj, kk, sx, sy)] : d[lin(ii, jj, kk, sx, sy)];
            }
        } else {
            int ii = map_axis(i, H, Nx, bcx), jj = map_axis(j, H, Ny, bcy);
            int kk = map_axis(k, H, Nz, bcz == BC_PERIODIC ? BC_PERIODIC : BC_NOFLUX);
            val = d[lin(ii, jj, kk, sx, sy)];
        }
        d[lin(i, j, k, sx, sy)] = val;
        (void)sz;
    }
}

template <typename T>
__global__ void halo_gather_kernel(T *__restrict__ d, int Nx, int Ny, int Nz, int H, int bcx, int bcy, int bcz,
                                   int wall_w) {
    halo_gather_body(d, Nx, Ny, Nz, H, bcx, bcy, bcz, wall_w);
}

// several fields of one grid in one launch (blockIdx.y = field); each gather
// reads interior values only, so the fields and their points are independent
template <typename T>
__global__ void halo_multi_kernel(HaloSet<T> hs, int Nx, int Ny, int Nz, int H) {
    const int f = blockIdx.y;
    halo_gather_body(hs.d[f], Nx, Ny, Nz, H, hs.bc[f][0], hs.bc[f][1], hs.bc[f][2], hs.wall_w[f]);
}

template <typename T>
void launch_halo(hipStream_t st, T *d, int Nx, int Ny, int Nz, int H, int loc, int bcx, int bcy, int bcz) {
    int wall_w = (loc == LOC_FZ && bcz == BC_WALL) ? 1 : 0;
    const int sx = Nx + 2 * H, sy = Ny + 2 * H;
    long total = (long)2 * H * sx * sy + (long)Nz * 2 * H * sx + (long)Nz * Ny * 2 * H + (wall_w ? (long)sx * sy : 0);
    int blocks = (int)((total + 255) / 256);
    if (blocks > 65535) blocks = 65535;
    hipLaunchKernelGGL(halo_gather_kernel<T>, dim3(blocks), dim3(256), 0, st, d, Nx, Ny, Nz, H, bcx, bcy, bcz, wall_w);
}
template void launch_halo<double>(hipStream_t, double *, int, int, int, int, int, int, int, int);
template void launch_halo<float>(hipStream_t, float *, int, int, int, int, int, int, int, int);

template <typename T>
void launch_halo_multi(hipStream_t st, const HaloSet<T> &hs, int Nx, int Ny, int Nz, int H) {
    const int sx = Nx + 2 * H, sy = Ny + 2 * H;
    const long total = (long)2 * H * sx * sy + (long)Nz * 2 * H * sx + (long)Nz * Ny * 2 * H + (long)sx * sy;
    int blocks = (int)((total + 255) / 256);
    if (blocks > 65535) blocks = 65535;
    hipLaunchKernelGGL(halo_multi_kernel<T>, dim3(blocks, hs.n), dim3(256), 0, st, hs, Nx, Ny, Nz, H);
}
template void launch_halo_multi<double>(hipStream_t, const HaloSet<double> &, int, int, int, int);
template void launch_halo_multi<float>(hipStream_t, const HaloSet<float> &, int, int, int, int);

// ---------------------------------------------------------------------------
// Face fluxes vel * face_value of each transported field, per direction, at
// the interface between c and c+1 along the axis. Transporting velocities
// as in _b_recon! (src/AdvectionSchemes.jl:685-697) and _b_mrecon_u!/_v!/_w!
// (:1203-1256); on a stretched grid the horizontal faces of a w volume take
// the volume-flux mean (_zflux), the transporting velocity of the centred
// operator (src/FiniteVolume.jl:775-797).
// ---------------------------------------------------------------------------
enum Field { F_U = 0, F_V = 1, F_W = 2, F_S = 3 };

template <typename T>
struct Fields {
    const T *__restrict__ u;
    const T *__restrict__ v;
    const T *__restrict__ w;
    const T *__restrict__ s;
};

template <int F, typename T>
__device__ __forceinline__ const T *field_ptr(const Fields<T> &f) {
    if constexpr (F == F_U) return f.u;
    else if constexpr (F == F_V) return f.v;
    else if constexpr (F == F_W) return f.w;
    else return f.s;
}

// byte strides of the storage along x, y, z
struct BStride {
    uint32_t x, y, z;
};
template <typename T>
__device__ __forceinline__ BStride bstrides(const Metrics<T> &m) {
    return BStride{(uint32_t)sizeof(T), (uint32_t)sizeof(T) * (uint32_t)m.sx,
                   (uint32_t)sizeof(T) * (uint32_t)m.sx * (uint32_t)m.sy};
}

// The flux of field F through the minus face (west, south or bottom for DIR
// = 0, 1, 2) of the cell at byte offset cb on level k.
template <int DIR, int F, int S, int P, typename T>
__device__ __forceinline__ T flux_minus(const Fields<T> &f, const Metrics<T> &m, uint32_t cb, int k,
                                        const BStride &b) {
    const uint32_t bd = DIR == 0 ? b.x : DIR == 1 ? b.y : b.z;
    const T *vp = DIR == 0 ? f.u : DIR == 1 ? f.v : f.w;  // the velocity normal to the face
    T vel;
    if constexpr (F == F_S) {
        vel = ldo(vp, cb);
    } else if constexpr (F == DIR) {
        vel = (ldo(vp, cb - bd) + ldo(vp, cb)) / T(2);
    } else {
        // the normal velocity averaged along the transported component's axis
        const uint32_t bf = F == F_U ? b.x : F == F_V ? b.y : b.z;
        const T lo = ldo(vp, cb - bf), hi = ldo(vp, cb);
        if constexpr (F == F_W) vel = m.m_zflux(k, lo, hi);
        else vel = (lo + hi) / T(2);
    }
    constexpr int R = SchemeInfo<S>::R;
    return vel * face_value<S, P, T>(field_ptr<F>(f), cb - (uint32_t)R * bd, bd, vel, m.teno_ct);
}

// _lap_at, src/FiniteVolume.jl:271-283 (f at byte offset cb, level k)
template <typename T>
__device__ __forceinline__ T lap_at(const T *__restrict__ f, const Metrics<T> &m, uint32_t cb, int k, int loc,
                                    const BStride &b) {
    const T c = ldo(f, cb);
    return (((ldo(f, cb + b.x) - T(2) * c) + ldo(f, cb - b.x)) * m.idx2 +
            ((ldo(f, cb + b.y) - T(2) * c) + ldo(f, cb - b.y)) * m.idy2) +
           m.m_lapz(loc, k, ldo(f, cb - b.z), c, ldo(f, cb + b.z));
}

// ---------------------------------------------------------------------------
// The marching advection kernel.
//
// A block is 64 x BY threads: each wave is one j-row of 64 cells along x,
// and every thread marches up a chunk of KC <= KCM levels. Each face flux is
// computed once (the reference evaluates every interior face from both of
// its cells; both evaluations are the same expression on the same values, so
// sharing one evaluation gives the same bits):
//   z: the top-face flux of level k is the bottom-face flux of level k+1
//      (carried in a register);
//   x: each lane computes its west face, the east face comes from the next
//      lane; the east faces of a wave's last cell for the chunk's levels are
//      computed before the march (lane l does level k0 + l) and kept in LDS;
//   y: each wave computes its south faces, the north face comes from the
//      next wave through LDS; the north faces of the block's top row for the
//      chunk's levels are computed before the march by all the block's
//      threads (thread (lane, ty) does levels k0 + ty, k0 + ty + BY, ...),
//      so that no wave does more face evaluations per level than the others.
// ---------------------------------------------------------------------------
enum Mode { MODE_SCALAR = 0, MODE_MOMENTUM = 1, MODE_STEP = 2 };

template <typename T>
struct MarchArgs {
    Metrics<T> m;
    Fields<T> in;
    // MODE_SCALAR: ts -= adv(s); MODE_MOMENTUM: tu, tv, tw -= adv
    T *tu, *tv, *tw, *ts;
    // MODE_STEP: predictor u* (uo, vo, wo) and the advanced scalar so
    T *uo, *vo, *wo, *so;
    const T *s0;  // step-start scalar for the stage combination
    T nu, dt, theta0, coef, fb, ft, fcor;
    T ca, cb;
    const T *spg;  // sponge vectors (rate_c, rate_f, target u, v, w), sz = Nz + 2H each
    int combine, has_visc, has_buoy, has_sflux, has_cor;
    int kc;  // levels per chunk (<= KCM)
};

constexpr int MW = 64;   // lanes per wave (gfx950)
constexpr int KCM = 8;   // levels per chunk

template <int MODE> struct ModeFields { static constexpr int lo = F_U, hi = F_S; };
template <> struct ModeFields<MODE_SCALAR> { static constexpr int lo = F_S, hi = F_S; };
template <> struct ModeFields<MODE_MOMENTUM> { static constexpr int lo = F_U, hi = F_W; };

// flux_minus with the field as a (loop-unrolled, hence constant) argument
template <int DIR, int S, int P, typename T>
__device__ __forceinline__ T flux_f(int F, const Fields<T> &f, const Metrics<T> &m, uint32_t co, int k,
                                    const BStride &b) {
    if (F == F_U) return flux_minus<DIR, F_U, S, P, T>(f, m, co, k, b);
    if (F == F_V) return flux_minus<DIR, F_V, S, P, T>(f, m, co, k, b);
    if (F == F_W) return flux_minus<DIR, F_W, S, P, T>(f, m, co, k, b);
    return flux_minus<DIR, F_S, S, P, T>(f, m, co, k, b);
}

template <int MODE, int S, int P, typename T, int BY, int STR>
__global__ void __launch_bounds__(MW *BY) adv_march_kernel(MarchArgs<T> a) {
    constexpr int F0 = ModeFields<MODE>::lo, F1 = ModeFields<MODE>::hi, NF = F1 - F0 + 1;
    constexpr uint32_t ES = sizeof(T);
    // the grid kind as a compile-time constant: the metric accessors fold to
    // UniformZ or LevelZ
    Metrics<T> m = a.m;
    m.stretched = STR;
    const BStride b = bstrides(m);
    const int H = m.H;
    const int lane = threadIdx.x, ty = threadIdx.y;
    const int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
    const int i0 = H + bx * MW;
    const int jb = H + by * BY;
    const int i = i0 + lane, j = jb + ty;
    const int k0 = H + bz * a.kc;
    const int k1 = min(k0 + a.kc, H + m.Nz);
    const int ilast = min(i0 + MW - 1, H + m.Nx - 1);  // the last cell of this wave's row
    const int jlast = min(jb + BY - 1, H + m.Ny - 1);  // the block's top row
    const bool row_ok = j < H + m.Ny;
    const bool ok = row_ok && i < H + m.Nx;

    __shared__ T xb[NF][BY][KCM];  // east boundary x-flux of each row, per level of the chunk
    __shared__ T yn[NF][KCM][MW];  // north y-flux of the top row, per level of the chunk
    __shared__ T ys[NF][BY][MW];   // south y-flux of the current level

    // batched east-boundary x-fluxes (the west faces of cell ilast + 1): lane l does level k0 + l
    if (row_ok) {
        const int kb = k0 + lane;
        if (kb < k1) {
            const uint32_t ce = lin(ilast + 1, j, kb, m.sx, m.sy) * ES;
#pragma unroll
            for (int F = F0; F <= F1; F++) {
                xb[F - F0][ty][lane] = flux_f<0, S, P, T>(F, a.in, m, ce, kb, b);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    // batched north y-fluxes of the top row (the south faces of row jlast + 1):
    // thread (lane, ty) does levels k0 + ty + BY·n
    if (i < H + m.Nx) {
        for (int kk = k0 + ty; kk < k1; kk += BY) {
            const uint32_t cn = lin(i, jlast + 1, kk, m.sx, m.sy) * ES;
#pragma unroll
            for (int F = F0; F <= F1; F++) {
                yn[F - F0][kk - k0][lane] = flux_f<1, S, P, T>(F, a.in, m, cn, kk, b);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    // bottom-face z-flux of the first level
    T fzb[NF];
    if (ok) {
        const uint32_t c0 = lin(i, j, k0, m.sx, m.sy) * ES;
#pragma unroll
        for (int F = F0; F <= F1; F++) {
            fzb[F - F0] = flux_f<2, S, P, T>(F, a.in, m, c0, k0, b);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();

    for (int k = k0; k < k1; k++) {
        // the cell's byte offset, made opaque to the compiler: otherwise loop
        // strength reduction keeps one 64-bit pointer per load site live
        // across the loop (about 100 VGPRs); every address below is this
        // offset plus a uniform stride multiple
        uint32_t co = lin(i, j, k, m.sx, m.sy) * ES;
        asm volatile("" : "+v"(co));
        // the faces of this level, one at a time: west and south fluxes to
        // LDS, the top z-flux in a register (the next level's bottom flux)
        T fzt[NF], fxw[NF];
        if (ok) {
#pragma unroll
            for (int F = F0; F <= F1; F++) {
                const int q = F - F0;
                fxw[q] = flux_f<0, S, P, T>(F, a.in, m, co, k, b);
                __builtin_amdgcn_sched_barrier(0);
                ys[q][ty][lane] = flux_f<1, S, P, T>(F, a.in, m, co, k, b);
                __builtin_amdgcn_sched_barrier(0);
                fzt[q] = flux_f<2, S, P, T>(F, a.in, m, co + b.z, k + 1, b);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
        if (ok) {
#pragma unroll
            for (int F = F0; F <= F1; F++) {
                const int q = F - F0;
                // the east x-flux is the west x-flux of the next lane (one
                // row of the tile is one wave); the row's last cell takes the
                // batched boundary flux
                const T fys = ys[q][ty][lane];
                const T fnext = __shfl_down(fxw[q], 1, MW);
                const T fxe = (i == ilast) ? xb[q][ty][k - k0] : fnext;
                const T fyn = (j < jlast) ? ys[q][ty + 1 < BY ? ty + 1 : ty][lane] : yn[q][k - k0][lane];
                const T idzF = (F == F_W) ? m.m_idzf(k) : m.m_idz(k);
                const T adv = ((fxe - fxw[q]) * m.idx + (fyn - fys) * m.idy) + (fzt[q] - fzb[q]) * idzF;
                if constexpr (MODE == MODE_SCALAR) {
                    sto(a.ts, co, ldo(a.ts, co) - adv);
                } else if constexpr (MODE == MODE_MOMENTUM) {
                    T *tp = F == F_U ? a.tu : F == F_V ? a.tv : a.tw;
                    sto(tp, co, ldo(tp, co) - adv);
                } else {
                    // the tendency from zero (+ ν∇²f), then buoyancy / surface flux
                    T t = T(0) - adv;
                    const T *fp = F == F_U ? a.in.u : F == F_V ? a.in.v : F == F_W ? a.in.w : a.in.s;
                    const int loc = F == F_U ? LOC_FX : F == F_V ? LOC_FY : F == F_W ? LOC_FZ : LOC_CC;
                    if (a.has_visc) t = t + a.nu * lap_at<T>(fp, m, co, k, loc, b);
                    if (F == F_W && a.has_buoy) {
                        const T tf = m.m_zface(k, ldo(a.in.s, co - b.z), ldo(a.in.s, co));
                        t += a.coef * (tf - a.theta0);
                    }
                    // f-plane Coriolis, _b_coriolis! (src/FiniteVolume.jl:900-911)
                    if (F == F_U && a.has_cor) {
                        const T *vp = a.in.v;
                        const T vu = T(0.25) * (((ldo(vp, co - ES) + ldo(vp, co)) + ldo(vp, co - ES + b.y)) +
                                                ldo(vp, co + b.y));
                        t += a.fcor * vu;
                    }
                    if (F == F_V && a.has_cor) {
                        const T *up = a.in.u;
                        const T uv = T(0.25) * (((ldo(up, co - b.y) + ldo(up, co + ES - b.y)) + ldo(up, co)) +
                                                ldo(up, co + ES));
                        t -= a.fcor * uv;
                    }
                    if (F == F_S && a.has_sflux) {
                        if (k == H) t += a.fb;
                        if (k == H + m.Nz - 1) t -= a.ft;
                    }
                    const T x = ldo(fp, co);
                    // Rayleigh sponge −λ(z)(f − f_target), _b_damping! (src/FiniteVolume.jl:639-647)
                    if (F != F_S && a.spg) {
                        const int sz = m.Nz + 2 * H;
                        const T lam = a.spg[(F == F_W ? sz : 0) + k];
                        const T tg = a.spg[(2 + F - F_U) * sz + k];
                        t -= lam * (x - tg);
                    }
                    if (F == F_U) sto(a.uo, co, x + a.dt * t);
                    else if (F == F_V) sto(a.vo, co, x + a.dt * t);
                    else if (F == F_W) sto(a.wo, co, x + a.dt * t);
                    else {
                        const T y = x + a.dt * t;
                        sto(a.so, co, a.combine ? a.ca * ldo(a.s0, co) + a.cb * y : y);
                    }
                }
                fzb[q] = fzt[q];
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();  // the level's fluxes are read before the next level writes them
    }
}

// ---------------------------------------------------------------------------
// The tiled advection kernel (MODE_MOMENTUM and MODE_STEP): the faces and
// terms of adv_march_kernel, with every value of the transported fields read
// from memory once per block.
//
// A block is 64 x BY threads over a column of KC levels; thread (lane, ty)
// owns cell column (i0 + lane, jb + ty).
//   - Each thread keeps its own column of every field in registers over the
//     reach of the z-stencil and the z-terms (levels k-RL .. k+R), shifted
//     up one level per step: the z-faces, the z-part of the Laplacian and the
//     buoyancy read these.
//   - At each level the block writes its x-y tile of every field with an
//     R-cell halo to LDS, the tile's cells from the registers and the halo
//     from memory (loaded a level ahead); the x- and y-faces, the Coriolis
//     averages and the x-y part of the Laplacian read the tile. w's tile is
//     held for two levels (k and k+1): the top faces of u and v are
//     transported by w at k+1 on the neighbouring columns.
//   - Each face is computed once, into LDS (x and y) or a register (z): a
//     cell's east face is the next cell's west face, its north face the next
//     row's south face, its top face the next level's bottom face. The east
//     faces of the rows' last cells and the north faces of the top row are
//     computed from the tile by one wave per field and direction (waves 0-3
//     north, 4-7 east), so that every wave evaluates 13 faces per level.
//   - Two barriers per level: after the tile is written, and after the faces
//     and the terms that read the tile; the tendencies then read only the
//     face arrays and registers, so the next level's tile writes need none.
// The arithmetic of every face and term is adv_march_kernel's on the same
// values.
// ---------------------------------------------------------------------------
template <int S> struct TileInfo {
    static constexpr int R = SchemeInfo<S>::R;
    static constexpr int RL = R > 1 ? R - 1 : 1;  // the registers hold levels k-RL .. k+R
    static constexpr int NW = RL + R + 1;
};

// the minus face (DIR 0: west, 1: south) of tile cell `at` at level k: the
// field's tile fl, the normal velocity's tile vl; wlo is the normal velocity
// at level k-1 (the lower value of a w volume's horizontal-face mean)
template <int DIR, int F, int S, int P, typename T, int TW>
__device__ __forceinline__ T tile_face(const T *fl, const T *vl, int at, T wlo, const Metrics<T> &m, int k) {
    constexpr int R = SchemeInfo<S>::R;
    constexpr int st = DIR == 0 ? 1 : TW;
    T vel;
    if constexpr (F == F_S) {
        vel = vl[at];
    } else if constexpr (F == DIR) {
        vel = (vl[at - st] + vl[at]) / T(2);
    } else if constexpr (F == F_W) {
        vel = m.m_zflux(k, wlo, vl[at]);
    } else {
        constexpr int sf = F == F_U ? 1 : TW;
        vel = (vl[at - sf] + vl[at]) / T(2);
    }
    T a[2 * R];
#pragma unroll
    for (int q = 0; q < 2 * R; q++) a[q] = fl[at + (q - R) * st];
    return vel * face_of<S, P, T>(a, vel, m.teno_ct);
}

// the top face of the level whose registers are wf (field) and ww (w): the
// minus face of the level above; wt is w's tile at the level above
template <int F, int S, int P, typename T, int TW>
__device__ __forceinline__ T win_zface(const T *wf, const T *ww, const T *wt, int at, const Metrics<T> &m) {
    constexpr int R = TileInfo<S>::R, RL = TileInfo<S>::RL;
    T vel;
    if constexpr (F == F_S) vel = ww[RL + 1];
    else if constexpr (F == F_W) vel = (ww[RL] + ww[RL + 1]) / T(2);
    else if constexpr (F == F_U) vel = (wt[at - 1] + wt[at]) / T(2);
    else vel = (wt[at - TW] + wt[at]) / T(2);
    return vel * face_of<S, P, T>(wf + (RL - R + 1), vel, m.teno_ct);
}

// Launch shape of the tiled kernel, measured at 256x256x128 (FP64 and FP32
// step): at least 4 waves per SIMD (128 VGPRs in FP64: two blocks per CU,
// against one at the unconstrained 147), the next level's values loaded a
// level ahead, blocks in XCD-contiguous order, 16 levels per chunk (8 and 32
// within 2 %).
constexpr int TILE_MINW = 4;
constexpr int TILE_KC = 16;
// Blocks a round: one per CU (a second one shares the CU's FP64 units). RK3
// step, 16 levels on every grid → by chunk_levels: 32³ periodic 507 → 164 us,
// 90×72×50 with the closure 706 → 404, 128×96×64 679 → 468, 160×160×90
// 1166 → 1014, 256×256×128 unchanged (16 levels).
constexpr int TILE_FILL = 256;

template <int MODE, int S, int P, typename T, int BY, int STR>
__global__ void __launch_bounds__(MW *BY, TILE_MINW) adv_tile_kernel(MarchArgs<T> a) {
    constexpr int F0 = ModeFields<MODE>::lo, F1 = ModeFields<MODE>::hi, NF = F1 - F0 + 1;
    static_assert(F0 == F_U && NF >= 3, "the tiled kernel transports the velocity");
    static_assert(BY == 8, "the boundary faces take one wave per field and direction");
    constexpr int R = TileInfo<S>::R, RL = TileInfo<S>::RL, NW = TileInfo<S>::NW;
    constexpr int TW = MW + 2 * R, TH = BY + 2 * R, TN = TW * TH;
    constexpr int NT = MW * BY;
    constexpr int NHALO = TN - NT;
    constexpr int NHP = (NHALO + NT - 1) / NT;  // halo cells per thread
    constexpr uint32_t ES = sizeof(T);
    // tile slots: u, v, w at even levels of the chunk, w at odd levels, s
    constexpr int SU = 0, SV = 1, SW = 2, SS = 4;
    constexpr int NSLOT = NF + 1;
    Metrics<T> m = a.m;
    m.stretched = STR;
    const BStride b = bstrides(m);
    const int H = m.H;
    const int lane = threadIdx.x, ty = threadIdx.y;
    const int tid = ty * MW + lane;
    // blocks in XCD-contiguous order: the tiles that share halos and the
    // chunks that share a column's levels run on one L2
    int bx, by, bz;
    xcd_block3(bx, by, bz);
    const int i0 = H + bx * MW;
    const int jb = H + by * BY;
    const int i = i0 + lane, j = jb + ty;
    const int k0 = H + bz * a.kc;
    const int k1 = min(k0 + a.kc, H + m.Nz);
    const int ilast = min(i0 + MW - 1, H + m.Nx - 1);
    const int jlast = min(jb + BY - 1, H + m.Ny - 1);
    const bool ok = i <= ilast && j <= jlast;                 // computes its cell
    const bool inb = i <= ilast + R && j <= jlast + R;        // its column feeds the tile
    const int at = (ty + R) * TW + lane + R;                  // its tile cell

    __shared__ T tile[NSLOT][TN];
    // the faces of the level: xs[F][row][c] the west face of cell i0 + c
    // (c = MW: the east face of a full row's last cell), ys[F][r][lane] the
    // south face of row jb + r (r = BY: the north face of a full top row)
    __shared__ T xs[NF][BY][MW + 1];
    __shared__ T ys[NF][BY + 1][MW];

    const T *fp[4] = {a.in.u, a.in.v, a.in.w, a.in.s};
    auto slot = [&](int F, int lev) { return F == F_W ? SW + ((lev - k0) & 1) : F == F_S ? SS : F; };

    // the halo cells this thread loads: bottom R rows, top R rows, then the
    // left and right R columns of the tile's rows; cells past the last
    // interior cell + R in x or y are outside what any face reads
    uint32_t hoff[NHP];
    int hat[NHP];
    bool hv[NHP];
#pragma unroll
    for (int p = 0; p < NHP; p++) {
        const int h = tid + p * NT;
        int r = 0, c = 0;
        if (h < R * TW) { r = h / TW; c = h % TW; }
        else if (h < 2 * R * TW) { const int h2 = h - R * TW; r = R + BY + h2 / TW; c = h2 % TW; }
        else { const int h3 = h - 2 * R * TW; r = R + h3 / (2 * R); const int q = h3 % (2 * R); c = q < R ? q : MW + q; }
        const int hi = i0 - R + c, hj = jb - R + r;
        hv[p] = h < NHALO && hi <= ilast + R && hj <= jlast + R;
        hat[p] = r * TW + c;
        hoff[p] = hv[p] ? lin(hi, hj, 0, m.sx, m.sy) * ES : 0u;
    }
    const uint32_t cof = inb ? lin(i, j, 0, m.sx, m.sy) * ES : 0u;  // own column at level 0

    // registers of the own column: win[F][n] = level k - RL + n at level k
    T win[NF][NW];
    T nxt[NF];       // the next level's top value
    T hal[NF][NHP];  // the next tile's halo (w one level further)
#pragma unroll
    for (int F = 0; F < NF; F++) {
        nxt[F] = T(0);
#pragma unroll
        for (int n = 0; n < NW; n++) win[F][n] = T(0);
#pragma unroll
        for (int p = 0; p < NHP; p++) hal[F][p] = T(0);
    }
    // the own column's top value and the tile's halo of level kk (w at kk+1)
    auto load_level = [&](int kk) {
        if (inb) {
#pragma unroll
            for (int F = 0; F < NF; F++) nxt[F] = ldo(fp[F], cof + (uint32_t)(kk + R) * b.z);
        }
#pragma unroll
        for (int p = 0; p < NHP; p++) {
            if (hv[p]) {
#pragma unroll
                for (int F = 0; F < NF; F++)
                    hal[F][p] = ldo(fp[F], hoff[p] + (uint32_t)(F == F_W ? kk + 1 : kk) * b.z);
            }
        }
    };
    if (inb) {
        const int kb = k0 - 1 - RL;
#pragma unroll
        for (int F = 0; F < NF; F++) {
#pragma unroll
            for (int n = RL - R + 1; n < NW; n++) win[F][n] = ldo(fp[F], cof + (uint32_t)(kb + n) * b.z);
        }
    }
    // w's tile at k0 (for the bottom face of k0)
#pragma unroll
    for (int p = 0; p < NHP; p++)
        if (hv[p]) tile[slot(F_W, k0)][hat[p]] = ldo(a.in.w, hoff[p] + (uint32_t)k0 * b.z);
    load_level(k0);
    if (inb) tile[slot(F_W, k0)][at] = win[F_W][RL + 1];
    __syncthreads();
    T fzb[NF];
#pragma unroll
    for (int F = 0; F < NF; F++) fzb[F] = T(0);
    if (ok) {
        const T *wt = tile[slot(F_W, k0)];
        fzb[F_U] = win_zface<F_U, S, P, T, TW>(win[F_U], win[F_W], wt, at, m);
        fzb[F_V] = win_zface<F_V, S, P, T, TW>(win[F_V], win[F_W], wt, at, m);
        fzb[F_W] = win_zface<F_W, S, P, T, TW>(win[F_W], win[F_W], wt, at, m);
        if constexpr (NF == 4) fzb[F_S] = win_zface<F_S, S, P, T, TW>(win[F_S], win[F_W], wt, at, m);
    }

    for (int k = k0; k < k1; k++) {
        // shift the registers up to level k and write the tiles: u, v, s at k, w at k+1
#pragma unroll
        for (int F = 0; F < NF; F++) {
#pragma unroll
            for (int n = 0; n < NW - 1; n++) win[F][n] = win[F][n + 1];
            win[F][NW - 1] = nxt[F];
        }
#pragma unroll
        for (int p = 0; p < NHP; p++) {
            if (hv[p]) {
#pragma unroll
                for (int F = 0; F < NF; F++) tile[slot(F, F == F_W ? k + 1 : k)][hat[p]] = hal[F][p];
            }
        }
        if (k + 1 < k1) load_level(k + 1);  // in flight over this level's faces
        if (inb) {
#pragma unroll
            for (int F = 0; F < NF; F++) tile[slot(F, F == F_W ? k + 1 : k)][at] = win[F][F == F_W ? RL + 1 : RL];
        }
        __syncthreads();

        const T *tu = tile[SU], *tv = tile[SV], *tw = tile[slot(F_W, k)], *twn = tile[slot(F_W, k + 1)];
        const T *ts = tu;
        if constexpr (NF == 4) ts = tile[SS];
        // the faces of the own cell: west and south to LDS, top in a register
        T fzt[NF];
#pragma unroll
        for (int F = 0; F < NF; F++) fzt[F] = T(0);
        if (ok) {
            xs[F_U][ty][lane] = tile_face<0, F_U, S, P, T, TW>(tu, tu, at, T(0), m, k);
            __builtin_amdgcn_sched_barrier(0);
            ys[F_U][ty][lane] = tile_face<1, F_U, S, P, T, TW>(tu, tv, at, T(0), m, k);
            __builtin_amdgcn_sched_barrier(0);
            fzt[F_U] = win_zface<F_U, S, P, T, TW>(win[F_U], win[F_W], twn, at, m);
            __builtin_amdgcn_sched_barrier(0);
            xs[F_V][ty][lane] = tile_face<0, F_V, S, P, T, TW>(tv, tu, at, T(0), m, k);
            __builtin_amdgcn_sched_barrier(0);
            ys[F_V][ty][lane] = tile_face<1, F_V, S, P, T, TW>(tv, tv, at, T(0), m, k);
            __builtin_amdgcn_sched_barrier(0);
            fzt[F_V] = win_zface<F_V, S, P, T, TW>(win[F_V], win[F_W], twn, at, m);
            __builtin_amdgcn_sched_barrier(0);
            xs[F_W][ty][lane] = tile_face<0, F_W, S, P, T, TW>(tw, tu, at, win[F_U][RL - 1], m, k);
            __builtin_amdgcn_sched_barrier(0);
            ys[F_W][ty][lane] = tile_face<1, F_W, S, P, T, TW>(tw, tv, at, win[F_V][RL - 1], m, k);
            __builtin_amdgcn_sched_barrier(0);
            fzt[F_W] = win_zface<F_W, S, P, T, TW>(win[F_W], win[F_W], twn, at, m);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (NF == 4) {
                xs[F_S][ty][lane] = tile_face<0, F_S, S, P, T, TW>(ts, tu, at, T(0), m, k);
                __builtin_amdgcn_sched_barrier(0);
                ys[F_S][ty][lane] = tile_face<1, F_S, S, P, T, TW>(ts, tv, at, T(0), m, k);
                __builtin_amdgcn_sched_barrier(0);
                fzt[F_S] = win_zface<F_S, S, P, T, TW>(win[F_S], win[F_W], twn, at, m);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // the boundary faces, one field per wave: wave F the north faces of
        // the top row, wave 4 + F the east faces of the rows' last cells
        // (the faces of w take the normal velocity at k-1 from memory)
        const int wv = __builtin_amdgcn_readfirstlane(ty);  // one row per wave: ty is the wave's
        if (wv < 4) {
            const int ii = i0 + lane, rb = jlast + 1 - jb;
            const int bat = (rb + R) * TW + lane + R;
            if (wv < NF && ii <= ilast) {
                if (wv == F_U) ys[F_U][rb][lane] = tile_face<1, F_U, S, P, T, TW>(tu, tv, bat, T(0), m, k);
                else if (wv == F_V) ys[F_V][rb][lane] = tile_face<1, F_V, S, P, T, TW>(tv, tv, bat, T(0), m, k);
                else if (wv == F_W) {
                    const T vlo = ldo(a.in.v, lin(ii, jlast + 1, k - 1, m.sx, m.sy) * ES);
                    ys[F_W][rb][lane] = tile_face<1, F_W, S, P, T, TW>(tw, tv, bat, vlo, m, k);
                } else if constexpr (NF == 4) {
                    ys[F_S][rb][lane] = tile_face<1, F_S, S, P, T, TW>(ts, tv, bat, T(0), m, k);
                }
            }
        } else {
            const int F = wv - 4, jj = jb + lane, cb = ilast + 1 - i0;
            const int bat = (lane + R) * TW + cb + R;
            if (F < NF && lane < BY && jj <= jlast) {
                if (F == F_U) xs[F_U][lane][cb] = tile_face<0, F_U, S, P, T, TW>(tu, tu, bat, T(0), m, k);
                else if (F == F_V) xs[F_V][lane][cb] = tile_face<0, F_V, S, P, T, TW>(tv, tu, bat, T(0), m, k);
                else if (F == F_W) {
                    const T ulo = ldo(a.in.u, lin(ilast + 1, jj, k - 1, m.sx, m.sy) * ES);
                    xs[F_W][lane][cb] = tile_face<0, F_W, S, P, T, TW>(tw, tu, bat, ulo, m, k);
                } else if constexpr (NF == 4) {
                    xs[F_S][lane][cb] = tile_face<0, F_S, S, P, T, TW>(ts, tu, bat, T(0), m, k);
                }
            }
        }
        // the terms that read the tile: the x-y part of the Laplacian and the
        // Coriolis averages (after the next barrier the tile is not read
        // again at this level, and the next level may overwrite it)
        T lapxy[NF], vcor = T(0), ucor = T(0);
#pragma unroll
        for (int F = 0; F < NF; F++) lapxy[F] = T(0);
        if constexpr (MODE == MODE_STEP) {
            if (ok && a.has_visc) {
                const T *tf[4] = {tu, tv, tw, ts};
#pragma unroll
                for (int F = 0; F < NF; F++) {
                    const T *tl = tf[F];
                    const T x = win[F][RL];
                    lapxy[F] = ((tl[at + 1] - T(2) * x) + tl[at - 1]) * m.idx2 +
                               ((tl[at + TW] - T(2) * x) + tl[at - TW]) * m.idy2;
                }
            }
            // f-plane Coriolis, _b_coriolis! (src/FiniteVolume.jl:900-911): v
            // averaged to the u point, u averaged to the v point
            if (ok && a.has_cor) {
                vcor = T(0.25) * (((tv[at - 1] + tv[at]) + tv[at - 1 + TW]) + tv[at + TW]);
                ucor = T(0.25) * (((tu[at - TW] + tu[at + 1 - TW]) + tu[at]) + tu[at + 1]);
            }
        }
        __syncthreads();

        if (ok) {
            uint32_t co = cof + (uint32_t)k * b.z;
            asm volatile("" : "+v"(co));
#pragma unroll
            for (int F = 0; F < NF; F++) {
                const T adv = ((xs[F][ty][lane + 1] - xs[F][ty][lane]) * m.idx +
                               (ys[F][ty + 1][lane] - ys[F][ty][lane]) * m.idy) +
                              (fzt[F] - fzb[F]) * ((F == F_W) ? m.m_idzf(k) : m.m_idz(k));
                if constexpr (MODE == MODE_MOMENTUM) {
                    T *tp = F == F_U ? a.tu : F == F_V ? a.tv : a.tw;
                    sto(tp, co, ldo(tp, co) - adv);
                } else {
                    const T x = win[F][RL];
                    T t = T(0) - adv;
                    if (a.has_visc) {
                        // ν∇²f, lap_at (src/FiniteVolume.jl:271-283): x and y from the tile, z from the registers
                        const int loc = F == F_U ? LOC_FX : F == F_V ? LOC_FY : F == F_W ? LOC_FZ : LOC_CC;
                        t = t + a.nu * (lapxy[F] + m.m_lapz(loc, k, win[F][RL - 1], x, win[F][RL + 1]));
                    }
                    if constexpr (NF == 4)
                        if (F == F_W && a.has_buoy) t += a.coef * (m.m_zface(k, win[F_S][RL - 1], win[F_S][RL]) - a.theta0);
                    // f-plane Coriolis, _b_coriolis! (src/FiniteVolume.jl:900-911)
                    if (F == F_U && a.has_cor) t += a.fcor * vcor;
                    if (F == F_V && a.has_cor) t -= a.fcor * ucor;
                    if (F == F_S && a.has_sflux) {
                        if (k == H) t += a.fb;
                        if (k == H + m.Nz - 1) t -= a.ft;
                    }
                    // Rayleigh sponge −λ(z)(f − f_target), _b_damping! (src/FiniteVolume.jl:639-647)
                    if (F != F_S && a.spg) {
                        const int sz = m.Nz + 2 * H;
                        const T lam = a.spg[(F == F_W ? sz : 0) + k];
                        const T tg = a.spg[(2 + F - F_U) * sz + k];
                        t -= lam * (x - tg);
                    }
                    if (F == F_U) sto(a.uo, co, x + a.dt * t);
                    else if (F == F_V) sto(a.vo, co, x + a.dt * t);
                    else if (F == F_W) sto(a.wo, co, x + a.dt * t);
                    else {
                        const T y = x + a.dt * t;
                        sto(a.so, co, a.combine ? a.ca * ldo(a.s0, co) + a.cb * y : y);
                    }
                }
                fzb[F] = fzt[F];
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // no barrier here: the next level writes the tile, which this phase
        // does not read, and its faces only after its first barrier, which
        // every wave reaches after this phase
    }
}

constexpr int MBY = 8;  // rows per block of the tile and brick kernels
int chunk_tile(int nx, int ny, int nz) {
    return chunk_levels(((nx + MW - 1) / MW) * ((ny + MBY - 1) / MBY), nz, TILE_KC, TILE_FILL, 1);
}
// the brick kernel holds several blocks per CU: shorter chunks pay only
// where KCM leaves CUs without a block (33×29×25 FP64 20.6 → 5.5 us,
// 130×70×60 WENO-Z7 35.6 → 31.9; 187×141×75 FP32 31.9, 33.3 if shortened)
int chunk_brick(int nx, int ny, int nz) {
    const int tiles = ((nx + MW - 1) / MW) * ((ny + MBY - 1) / MBY), kmax = nz < KCM ? nz : KCM;
    return tiles * ((nz + kmax - 1) / kmax) >= 256 ? kmax : chunk_levels(tiles, nz, kmax, 256, 3);
}

template <int MODE, int S, int P, typename T>
static void launch_march_sp(hipStream_t st, const MarchArgs<T> &a) {
    constexpr int BY = MBY;
    const Metrics<T> &m = a.m;
    if constexpr (MODE != MODE_SCALAR) {
        MarchArgs<T> t = a;
        t.kc = chunk_tile(m.Nx, m.Ny, m.Nz);
        dim3 grid((m.Nx + MW - 1) / MW, (m.Ny + BY - 1) / BY, (m.Nz + t.kc - 1) / t.kc);
        if (m.stretched)
            hipLaunchKernelGGL((adv_tile_kernel<MODE, S, P, T, BY, 1>), grid, dim3(MW, BY), 0, st, t);
        else
            hipLaunchKernelGGL((adv_tile_kernel<MODE, S, P, T, BY, 0>), grid, dim3(MW, BY), 0, st, t);
        return;
    }
    dim3 grid((m.Nx + MW - 1) / MW, (m.Ny + BY - 1) / BY, (m.Nz + a.kc - 1) / a.kc);
    if (m.stretched)
        hipLaunchKernelGGL((adv_march_kernel<MODE, S, P, T, BY, 1>), grid, dim3(MW, BY), 0, st, a);
    else
        hipLaunchKernelGGL((adv_march_kernel<MODE, S, P, T, BY, 0>), grid, dim3(MW, BY), 0, st, a);
}

template <int MODE, typename T>
static int launch_march_mode(hipStream_t st, const MarchArgs<T> &a, int scheme, int p) {
    switch (scheme) {
    case SCH_CENTERED: launch_march_sp<MODE, SCH_CENTERED, 0, T>(st, a); return 0;
    case SCH_UPWIND1: launch_march_sp<MODE, SCH_UPWIND1, 0, T>(st, a); return 0;
    case SCH_WENO5: launch_march_sp<MODE, SCH_WENO5, 0, T>(st, a); return 0;
    case SCH_WENO_JS5: launch_march_sp<MODE, SCH_WENO_JS5, 0, T>(st, a); return 0;
    case SCH_WENO_Z5:
        if (p == 1) launch_march_sp<MODE, SCH_WENO_Z5, 1, T>(st, a);
        else launch_march_sp<MODE, SCH_WENO_Z5, 2, T>(st, a);
        return 0;
    case SCH_WENO_Z7:
        if (p == 1) launch_march_sp<MODE, SCH_WENO_Z7, 1, T>(st, a);
        else launch_march_sp<MODE, SCH_WENO_Z7, 2, T>(st, a);
        return 0;
    case SCH_TENO5:
        if constexpr (MODE == MODE_SCALAR) {
            launch_march_sp<MODE, SCH_TENO5, 0, T>(st, a);
            return 0;
        }
        return -1;
    case SCH_TENO8:
        if constexpr (MODE == MODE_SCALAR) {
            launch_march_sp<MODE, SCH_TENO8, 0, T>(st, a);
            return 0;
        }
        return -1;
    }
    return -1;
}

// advect_variance_conserving! (src/AdvectionSchemes.jl:1428-1446), regular
// grids: tend −= (u_e ϕ_{i+1} − u_w ϕ_{i−1})/(2Δx) + (y) + (z), the skew form
// ½[∇·(uϕ) + u·∇ϕ] that conserves Σϕ² for any velocity. 1/(2Δ) = (1/Δ)/2 exactly.
template <typename T>
__global__ void __launch_bounds__(256) varcons_kernel(T *__restrict__ tend, const T *__restrict__ u,
                                                      const T *__restrict__ v, const T *__restrict__ w,
                                                      const T *__restrict__ phi, Metrics<T> m) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y * blockDim.y + threadIdx.y, k = blockIdx.z;
    if (i >= m.Nx || j >= m.Ny) return;
    const uint32_t sx = m.sx, sxy = (uint32_t)m.sx * m.sy;
    const uint32_t c = lin(i + m.H, j + m.H, k + m.H, m.sx, m.sy);
    const T h2x = m.idx * T(0.5), h2y = m.idy * T(0.5), h2z = m.idz * T(0.5);
    const T d = ((u[c + 1] * phi[c + 1] - u[c] * phi[c - 1]) * h2x + (v[c + sx] * phi[c + sx] - v[c] * phi[c - sx]) * h2y) +
                (w[c + sxy] * phi[c + sxy] - w[c] * phi[c - sxy]) * h2z;
    tend[c] = tend[c] - d;
}
template <typename T>
void launch_varcons(hipStream_t st, const Metrics<T> &m, T *tend, const T *u, const T *v, const T *w, const T *phi) {
    const dim3 blk(64, 4), grd((m.Nx + 63) / 64, (m.Ny + 3) / 4, m.Nz);
    hipLaunchKernelGGL(varcons_kernel<T>, grd, blk, 0, st, tend, u, v, w, phi, m);
}
template void launch_varcons<double>(hipStream_t, const Metrics<double> &, double *, const double *, const double *,
                                     const double *, const double *);
template void launch_varcons<float>(hipStream_t, const Metrics<float> &, float *, const float *, const float *,
                                    const float *, const float *);

template <typename T>
int launch_advect(hipStream_t st, const Metrics<T> &m, int mode, int scheme, int p, const T *u, const T *v,
                  const T *w, const T *s, T *tu, T *tv, T *tw, T *ts) {
    MarchArgs<T> a{};
    a.m = m;
    a.in = Fields<T>{u, v, w, s};
    a.tu = tu; a.tv = tv; a.tw = tw; a.ts = ts;
    a.kc = chunk_brick(m.Nx, m.Ny, m.Nz);
    if (mode == MODE_SCALAR) return launch_march_mode<MODE_SCALAR, T>(st, a, scheme, p);
    return launch_march_mode<MODE_MOMENTUM, T>(st, a, scheme, p);
}
template int launch_advect<double>(hipStream_t, const Metrics<double> &, int, int, int, const double *, const double *,
                                   const double *, const double *, double *, double *, double *, double *);
template int launch_advect<float>(hipStream_t, const Metrics<float> &, int, int, int, const float *, const float *,
                                  const float *, const float *, float *, float *, float *, float *);

template <typename T>
int launch_tendency_step(hipStream_t st, const Metrics<T> &m, int scheme, int p, const T *u, const T *v, const T *w,
                         const T *s, T *uo, T *vo, T *wo, T *so, const T *s0, const StepPhys &ph, int stage) {
    MarchArgs<T> a{};
    a.m = m;
    a.in = Fields<T>{u, v, w, s};
    a.uo = uo; a.vo = vo; a.wo = wo; a.so = so; a.s0 = s0;
    a.nu = T(ph.nu); a.dt = T(ph.dt); a.theta0 = T(ph.theta0);
    a.coef = T(ph.g_accel / ph.theta0);
    a.has_visc = ph.nu != 0;
    a.has_buoy = ph.theta0 != 0;
    a.has_sflux = ph.flux_bot != 0 || ph.flux_top != 0;
    // F_bot · 1/Δz_c at the bottom level, F_top · 1/Δz_c at the top (src/FiniteVolume.jl:431-439)
    a.fb = T(ph.flux_bot * ph.idz_bot);
    a.ft = T(ph.flux_top * ph.idz_top);
    a.fcor = T(ph.fcor);
    a.has_cor = ph.fcor != 0;
    a.spg = (const T *)ph.sponge;
    stage_coeffs(stage, &ph, &a.ca, &a.cb, &a.combine);
    return launch_march_mode<MODE_STEP, T>(st, a, scheme, p);
}
template int launch_tendency_step<double>(hipStream_t, const Metrics<double> &, int, int, const double *,
                                          const double *, const double *, const double *, double *, double *,
                                          double *, double *, const double *, const StepPhys &, int);
template int launch_tendency_step<float>(hipStream_t, const Metrics<float> &, int, int, const float *, const float *,
                                         const float *, const float *, float *, float *, float *, float *,
                                         const float *, const StepPhys &, int);

// ---------------------------------------------------------------------------
// _div_at into the interior-sized solver buffer (src/FiniteVolume.jl:312-315,
// 1869-1888), accumulated in FP64.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void div_into_kernel(double *__restrict__ buf, const T *__restrict__ u, const T *__restrict__ v,
                                const T *__restrict__ w, Metrics<double> md) {
    const int H = md.H, sx = md.sx, sy = md.sy;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y, k = blockIdx.z;
    if (i >= md.Nx) return;
    const int I = i + H, J = j + H, K = k + H;
    const size_t c = lin(I, J, K, sx, sy);
    double du = (double)u[c + 1] - (double)u[c];
    double dv = (double)v[c + sx] - (double)v[c];
    double dw = (double)w[c + (size_t)sx * sy] - (double)w[c];
    buf[(size_t)i + (size_t)md.Nx * ((size_t)j + (size_t)md.Ny * k)] = (du * md.idx + dv * md.idy) + dw * md.m_idz(K);
}

template <typename T>
void launch_div_into(hipStream_t st, double *buf, const T *u, const T *v, const T *w, const Metrics<double> &md) {
    dim3 grid((md.Nx + 255) / 256, md.Ny, md.Nz);
    hipLaunchKernelGGL(div_into_kernel<T>, grid, dim3(256), 0, st, buf, u, v, w, md);
}
template void launch_div_into<double>(hipStream_t, double *, const double *, const double *, const double *,
                                      const Metrics<double> &);
template void launch_div_into<float>(hipStream_t, double *, const float *, const float *, const float *,
                                     const Metrics<double> &);

// ---------------------------------------------------------------------------
// _b_correct! (src/FiniteVolume.jl:1823-1833) with the stage combination
// c(x, snap) = a·snap + b·x (src/Simulations.jl:1192-1194) and p = φ/Δt. φ
// is the solver's interior-sized FP64 solution; with th, θ = c(tn, th0) too. φ's halo (the velocity BCs
// at a cell centre: periodic wrap or mirror) is read through the index map.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void correct_kernel(T *uo, T *vo, T *wo,
                               const T *__restrict__ us, const T *__restrict__ vs, const T *__restrict__ ws,
                               const T *u0, const T *v0, const T *w0,
                               const double *__restrict__ phi, T *__restrict__ p, Metrics<double> md, int bcx,
                               int bcy, int bcz, double ca, double cb, int combine, double dt, T *th, const T *tn,
                               const T *th0) {
    const int H = md.H, sx = md.sx, sy = md.sy, Nx = md.Nx, Ny = md.Ny, Nz = md.Nz;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y, k = blockIdx.z;
    if (i >= Nx) return;
    auto P = [&](int ii, int jj, int kk) {
        // interior-local index map of φ's unit halo
        if (ii < 0) ii = bcx == BC_PERIODIC ? ii + Nx : -1 - ii;
        if (jj < 0) jj = bcy == BC_PERIODIC ? jj + Ny : -1 - jj;
        if (kk < 0) kk = bcz == BC_PERIODIC ? kk + Nz : -1 - kk;
        return phi[(size_t)ii + (size_t)Nx * ((size_t)jj + (size_t)Ny * kk)];
    };
    const double pc = P(i, j, k);
    const int K = k + H;
    const size_t c = lin(i + H, j + H, K, sx, sy);
    double un = (double)us[c] - (pc - P(i - 1, j, k)) * md.idx;
    double vn = (double)vs[c] - (pc - P(i, j - 1, k)) * md.idy;
    double wn = (double)ws[c] - (pc - P(i, j, k - 1)) * md.m_idzf(K);
    if (combine) {
        un = ca * (double)u0[c] + cb * un;
        vn = ca * (double)v0[c] + cb * vn;
        wn = ca * (double)w0[c] + cb * wn;
    }
    uo[c] = (T)un;
    vo[c] = (T)vn;
    wo[c] = (T)wn;
    if (p) p[c] = (T)(pc / dt);
    if (th) th[c] = combine ? (T)(ca * (double)th0[c] + cb * (double)tn[c]) : tn[c];
}

template <typename T>
void launch_correct(hipStream_t st, T *uo, T *vo, T *wo, const T *us, const T *vs, const T *ws, const T *u0,
                    const T *v0, const T *w0, const double *phi, T *p, const Metrics<double> &md, int bcx, int bcy,
                    int bcz, double ca, double cb, int combine, double dt, T *th, const T *tn, const T *th0) {
    dim3 grid((md.Nx + 255) / 256, md.Ny, md.Nz);
    hipLaunchKernelGGL(correct_kernel<T>, grid, dim3(256), 0, st, uo, vo, wo, us, vs, ws, u0, v0, w0, phi, p, md, bcx,
                       bcy, bcz, ca, cb, combine, dt, th, tn, th0);
}
template void launch_correct<double>(hipStream_t, double *, double *, double *, const double *, const double *,
                                     const double *, const double *, const double *, const double *, const double *,
                                     double *, const Metrics<double> &, int, int, int, double, double, int, double,
                                     double *, const double *, const double *);
template void launch_correct<float>(hipStream_t, float *, float *, float *, const float *, const float *,
                                    const float *, const float *, const float *, const float *, const double *,
                                    float *, const Metrics<double> &, int, int, int, double, double, int, double,
                                    float *, const float *, const float *);

// ---------------------------------------------------------------------------
// The RK3 combination of the halo shell, out = a·snap + b·x at every storage
// point outside the interior (_shell_map!, src/Simulations.jl:1249-1286).
// ---------------------------------------------------------------------------
// The halo shell of up to four fields (blockIdx.y = field) combined as the
// interior is, out = ca·snap + cb·x (ca = 0, cb = 1: a copy), visiting the
// shell's points only: the two z slabs, then the y and the x slabs of the
// interior levels (the enumeration of halo_gather_body).
template <typename T>
__global__ void shell_kernel(ShellSet<T> ss, int Nx, int Ny, int Nz, int H, double ca, double cb) {
    const int f = blockIdx.y;
    T *__restrict__ out = ss.out[f];
    const T *__restrict__ x = ss.x[f];
    const T *__restrict__ snap = ss.snap[f];
    const int sx = Nx + 2 * H, sy = Ny + 2 * H;
    const uint32_t nz_slab = (uint32_t)2 * H * sx * sy;
    const uint32_t ny_slab = (uint32_t)Nz * 2 * H * sx;
    const uint32_t nx_slab = (uint32_t)Nz * Ny * 2 * H;
    const uint32_t total = nz_slab + ny_slab + nx_slab;
    const bool copy = ca == 0.0 && cb == 1.0;
    for (uint32_t t = blockIdx.x * (uint32_t)blockDim.x + threadIdx.x; t < total; t += (uint32_t)gridDim.x * blockDim.x) {
        int i, j, k;
        if (t < nz_slab) {
            uint32_t q = t;
            i = (int)(q % sx); q /= sx;
            j = (int)(q % sy); q /= sy;
            const int l = (int)q;
            k = l < H ? l : H + Nz + (l - H);
        } else if (t < nz_slab + ny_slab) {
            uint32_t q = t - nz_slab;
            i = (int)(q % sx); q /= sx;
            const int l = (int)(q % (2 * H)); q /= (2 * H);
            j = l < H ? l : H + Ny + (l - H);
            k = H + (int)q;
        } else {
            uint32_t q = t - nz_slab - ny_slab;
            const int l = (int)(q % (2 * H)); q /= (2 * H);
            i = l < H ? l : H + Nx + (l - H);
            j = H + (int)(q % Ny);
            k = H + (int)(q / Ny);
        }
        const size_t c = lin(i, j, k, sx, sy);
        out[c] = copy ? x[c] : (T)(ca * (double)snap[c] + cb * (double)x[c]);
    }
}

template <typename T>
void launch_shell(hipStream_t st, const ShellSet<T> &ss, int Nx, int Ny, int Nz, int H, double ca, double cb) {
    const int sx = Nx + 2 * H, sy = Ny + 2 * H;
    const long total = (long)2 * H * sx * sy + (long)Nz * 2 * H * sx + (long)Nz * Ny * 2 * H;
    int blocks = (int)((total + 255) / 256);
    if (blocks > 65535) blocks = 65535;
    hipLaunchKernelGGL(shell_kernel<T>, dim3(blocks, ss.n), dim3(256), 0, st, ss, Nx, Ny, Nz, H, ca, cb);
}
template void launch_shell<double>(hipStream_t, const ShellSet<double> &, int, int, int, int, double, double);
template void launch_shell<float>(hipStream_t, const ShellSet<float> &, int, int, int, int, double, double);

// ---------------------------------------------------------------------------
// Maxima (exact in any order): max |∇·u| (max_divergence, src/Simulations.jl:
// 1045-1050) and the advective CFL rate (_adv_rate_at, src/TimeIntegration.jl:
// 172-182). Non-negative doubles order as their bit patterns, so the maximum
// is an atomicMax on the bits (NaN-propagating, as the reference's max).
// ---------------------------------------------------------------------------
// Diagnostics over the interior cells, one partial per block (grid-stride
// over the flattened interior, a tree in LDS): what = 0 max |∇·u|
// (max_divergence, src/Simulations.jl:1045-1050); 3 max of the cell field u;
// 1 max Σ|u_i|/Δx_i
// (_max_advective_rate, src/TimeIntegration.jl:164-182); 2 Σ of the kinetic
// energy density (u² + v²)·Δz_c + w²·Δz_f (kinetic_energy,
// src/Simulations.jl:992-1015; uniform grids Δz_c = Δz_f = Δz).
// max(a, b) that propagates NaN, as Julia's max does (fmax drops it)
__device__ inline double nanmax(double a, double b) { return (b > a || b != b) ? b : a; }

template <typename T>
__global__ void __launch_bounds__(256) diag_kernel(double *__restrict__ part, const T *__restrict__ u,
                                                   const T *__restrict__ v, const T *__restrict__ w,
                                                   Metrics<double> md, int what) {
    __shared__ double sh[256];
    const int H = md.H, sx = md.sx, sy = md.sy;
    // 32-bit index arithmetic: every interior is below 2^32 cells
    const uint32_t n = (uint32_t)md.Nx * md.Ny * md.Nz;
    double acc = 0.0;
    for (uint32_t e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x) {
        const int i = (int)(e % (uint32_t)md.Nx);
        const uint32_t r = e / (uint32_t)md.Nx;
        const int j = (int)(r % (uint32_t)md.Ny), k = (int)(r / (uint32_t)md.Ny);
        const int K = k + H;
        const size_t c = lin(i + H, j + H, K, sx, sy);
        double val;
        if (what == 0) {
            val = cell_abs_div(u, v, w, c, (size_t)sx, (size_t)sx * sy, md, K);
        } else if (what == 1) {
            const double au = nanmax(fabs((double)u[c]), fabs((double)u[c + 1]));
            const double av = nanmax(fabs((double)v[c]), fabs((double)v[c + sx]));
            const double aw = nanmax(fabs((double)w[c]), fabs((double)w[c + (size_t)sx * sy]));
            val = (au * md.idx + av * md.idy) + aw * md.m_idz(K);
        } else if (what == 3) {
            val = (double)u[c];  // the maximum of a cell field (the SGS coefficients' maxima)
        } else {
            const double uu = (double)u[c], vv = (double)v[c], ww = (double)w[c];
            if (md.stretched) val = (uu * uu + vv * vv) * (1.0 / md.idzc[K]) + ww * ww * (1.0 / md.idzf[K]);
            else val = (uu * uu + vv * vv) + ww * ww;
        }
        // a NaN propagates through the max (range_max, src/Backends.jl:1060-1092)
        if (what == 2) acc += val;
        else acc = (val > acc || val != val) ? val : acc;
    }
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            const double a = sh[threadIdx.x], b = sh[threadIdx.x + s];
            sh[threadIdx.x] = what == 2 ? a + b : ((b > a || b != b) ? b : a);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// per-level sums of a cell field over the interior plane (one block per
// level; a fixed-order tree): the plane means of cfl_diagnostics' N
template <typename T>
__global__ void __launch_bounds__(256) plane_sum_kernel(double *__restrict__ out, const T *__restrict__ f,
                                                        Metrics<double> md) {
    __shared__ double sh[256];
    const int K = blockIdx.x + md.H;
    double acc = 0.0;
    const int np = md.Nx * md.Ny;
    for (int e = threadIdx.x; e < np; e += blockDim.x) {
        const int j = e / md.Nx, i = e - j * md.Nx;
        acc += (double)f[lin(i + md.H, j + md.H, K, md.sx, md.sy)];
    }
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.x] = sh[0];
}
template <typename T>
void launch_plane_sum(hipStream_t st, double *out, const T *f, const Metrics<double> &md) {
    hipLaunchKernelGGL(plane_sum_kernel<T>, dim3(md.Nz), dim3(256), 0, st, out, f, md);
}
template void launch_plane_sum<double>(hipStream_t, double *, const double *, const Metrics<double> &);
template void launch_plane_sum<float>(hipStream_t, double *, const float *, const Metrics<double> &);

// The post-step checks of step_adaptive! in one sweep over the interior
// (step_guard, src/TimeIntegration.jl:673-710; the sound-proof cores'
// step_guard, src/Anelastic.jl:2333-2346). Per block three partials:
// part[3b] = 1 where some u, v, w, θ or p value is not finite (0 otherwise),
// part[3b+1] = max |∇·u| (Wc == nullptr: the stencil of max_divergence) or
// max |(1/W_c)∇·(W u)| (the constraint residual of a sound-proof core, the
// stencil of weighted_divergence!), part[3b+2] = max(|u|, |v|, |w|). The
// maxima propagate NaN, as the reference's range_max does.
template <typename T>
__global__ void __launch_bounds__(256) guard_kernel(double *__restrict__ part, const T *__restrict__ u,
                                                    const T *__restrict__ v, const T *__restrict__ w,
                                                    const T *__restrict__ th, const T *__restrict__ p,
                                                    const double *__restrict__ Wc, const double *__restrict__ Wf,
                                                    Metrics<double> md) {
    __shared__ double sh[3][256];
    const int H = md.H, sx = md.sx, sy = md.sy;
    const size_t sxy = (size_t)sx * sy;
    const uint32_t n = (uint32_t)md.Nx * md.Ny * md.Nz;
    double bad = 0.0, dmax = 0.0, smax = 0.0;
    for (uint32_t e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x) {
        const int i = (int)(e % (uint32_t)md.Nx);
        const uint32_t r = e / (uint32_t)md.Nx;
        const int j = (int)(r % (uint32_t)md.Ny), k = (int)(r / (uint32_t)md.Ny);
        const int K = k + H;
        const size_t c = lin(i + H, j + H, K, sx, sy);
        const double uc = (double)u[c], vc = (double)v[c], wc = (double)w[c];
        const bool fin = isfinite(uc) && isfinite(vc) && isfinite(wc) && isfinite((double)th[c]) &&
                         isfinite((double)p[c]);
        bad = fin ? bad : 1.0;
        const double du = (double)u[c + 1] - uc, dv = (double)v[c + sx] - vc;
        double d;
        if (Wc) {
            const double wk = Wc[K];
            d = (1 / wk) * (wk * (du * md.idx + dv * md.idy) + (Wf[K + 1] * (double)w[c + sxy] - Wf[K] * wc) * md.idz);
        } else {
            d = (du * md.idx + dv * md.idy) + ((double)w[c + sxy] - wc) * md.m_idz(K);
        }
        dmax = nanmax(dmax, fabs(d));
        smax = nanmax(smax, nanmax(nanmax(fabs(uc), fabs(vc)), fabs(wc)));
    }
    sh[0][threadIdx.x] = bad;
    sh[1][threadIdx.x] = dmax;
    sh[2][threadIdx.x] = smax;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int q = 0; q < 3; q++) sh[q][threadIdx.x] = nanmax(sh[q][threadIdx.x], sh[q][threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x < 3) part[3 * blockIdx.x + threadIdx.x] = sh[threadIdx.x][0];
}
template <typename T>
void launch_guard(hipStream_t st, double *part, int nblocks, const T *u, const T *v, const T *w, const T *th,
                  const T *p, const double *Wc, const double *Wf, const Metrics<double> &md) {
    hipLaunchKernelGGL(guard_kernel<T>, dim3(nblocks), dim3(256), 0, st, part, u, v, w, th, p, Wc, Wf, md);
}
template void launch_guard<double>(hipStream_t, double *, int, const double *, const double *, const double *,
                                   const double *, const double *, const double *, const double *,
                                   const Metrics<double> &);
template void launch_guard<float>(hipStream_t, double *, int, const float *, const float *, const float *,
                                  const float *, const float *, const double *, const double *,
                                  const Metrics<double> &);

template <typename T>
void launch_diag(hipStream_t st, double *part, int nblocks, const T *u, const T *v, const T *w,
                 const Metrics<double> &md, int what) {
    hipLaunchKernelGGL(diag_kernel<T>, dim3(nblocks), dim3(256), 0, st, part, u, v, w, md, what);
}
template void launch_diag<double>(hipStream_t, double *, int, const double *, const double *, const double *,
                                  const Metrics<double> &, int);
template void launch_diag<float>(hipStream_t, double *, int, const float *, const float *, const float *,
                                 const Metrics<double> &, int);

}  // namespace aeo
