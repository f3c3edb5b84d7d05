// The learned preconditioner: a 3-level 3-D U-Net on gfx950 MFMA, trained on
// the GPU by its own forward and backward kernels, and the flexible CG that
// uses it (no reference counterpart: the reference has no network; its
// nearest hook is src/ML.jl:40-56, and the solver it accelerates is
// MGPreconditionedCG, src/Multigrid.jl:879-972).
//
// Network (c0 = 16 channels at full resolution):
//   enc0: conv 3³ in→16, conv 16→16 (skip0)         full resolution
//   pool: 2×2×2 mean
//   enc1: conv 16→32, conv 32→32 (skip1)            1/2
//   pool
//   mid:  conv 32→64, conv 64→64                    1/4
//   up ×2 (nearest), concat [up, skip1] (96 channels)
//   dec1: conv 96→32, conv 32→32                    1/2
//   up ×2, concat [up, skip0] (48 channels)
//   dec0: conv 48→16, conv 16→16                    full
//   head: 1×1 conv 16→1 (FP32)
// every 3³ convolution has a bias and a ReLU; x and y are periodic, z is
// zero-padded. Input channels: the source scaled to unit RMS, and optionally
// the fluid mask; the output is multiplied back by the source's RMS.
//
// Arithmetic: activations and weights in BF16, FP32 accumulation
// (v_mfma_f32_16x16x32_bf16), FP32 master weights, gradients and Adam.
// Layout: channels-last [voxel][channel], voxel = x + nx·(y + ny·z); channel
// counts padded to multiples of 8 (the input to 8).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

#include "kernels.h"

namespace aeo {

typedef __bf16 bf16;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

struct Vol {
    int nx, ny, nz;
};
__device__ __forceinline__ int wrapi(int a, int n) { return a < 0 ? a + n : (a >= n ? a - n : a); }
__device__ __forceinline__ bf16x8 zero8() { return __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u}); }

constexpr int UB = 256;  // threads per block of the elementwise kernels

// ---------------------------------------------------------------------------
// 3×3×3 convolution as an implicit GEMM on MFMA:
//   out[v][ooff + n] = act(bias[n] + Σ_tap Σ_c in[nb(v, tap)][c] · W[tap][c][n])
// M = voxels (64 per wave: four 16-row tiles), N = COUT, K = 27·CIN, ordered
// k = tap·CIN + c; chunks of 32 (lane group g of 16 lanes holds k = 32·ch +
// 8g .. +7, i.e. 8 channels of one tap: one 16-byte load). Weights in the B
// layout wb[k/8][n][k%8], zero-filled up to NCH·32 rows. The same kernel with
// the flipped, transposed weights is the backward pass for the input.
// Lane layout of v_mfma_f32_16x16x32_bf16: A row = lane % 16, k = 8·(lane/16)
// .. +7; B column = lane % 16, same k; D[4·(lane/16) + i][lane % 16].
// ---------------------------------------------------------------------------
template <int CIN, int COUT>
__global__ void __launch_bounds__(256) conv3_kernel(const bf16 *__restrict__ in, const bf16 *__restrict__ wb,
                                                    const float *__restrict__ bias, bf16 *__restrict__ out, int ocs,
                                                    int ooff, Vol g, int relu) {
    constexpr int TN = COUT / 16, TM = 4;
    constexpr int NCH = (27 * CIN + 31) / 32;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nxy = g.nx * g.ny;
    const int nvox = nxy * g.nz;
    const int vbase = (blockIdx.x * 4 + wave) * 64;
    if (vbase >= nvox) return;  // no block-level synchronisation below
    const int r = lane & 15, grp = lane >> 4;
    int vx[TM], vy[TM], vz[TM];
#pragma unroll
    for (int t = 0; t < TM; t++) {
        const int v = vbase + 16 * t + r;
        vz[t] = v < nvox ? v / nxy : -1000;  // out-of-range rows read zeros
        const int rem = v - (v / nxy) * nxy;
        vy[t] = rem / g.nx;
        vx[t] = rem - vy[t] * g.nx;
    }
    f32x4 acc[TM][TN];
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
        for (int u = 0; u < TN; u++) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int ch = 0; ch < NCH; ch++) {
        const int k0 = ch * 32 + grp * 8;
        const int tap = k0 / CIN, c0 = k0 - tap * CIN;
        bf16x8 b[TN];
#pragma unroll
        for (int u = 0; u < TN; u++)
            b[u] = *reinterpret_cast<const bf16x8 *>(wb + ((size_t)(k0 >> 3) * COUT + 16 * u + r) * 8);
        bf16x8 a[TM];
        const int dx = tap % 3 - 1, dy = (tap / 3) % 3 - 1, dz = tap / 9 - 1;
#pragma unroll
        for (int t = 0; t < TM; t++) {
            const int z = vz[t] + dz;
            if (tap < 27 && z >= 0 && z < g.nz) {
                const int x = wrapi(vx[t] + dx, g.nx), y = wrapi(vy[t] + dy, g.ny);
                a[t] = *reinterpret_cast<const bf16x8 *>(in + ((size_t)(x + g.nx * (y + g.ny * z)) * CIN + c0));
            } else {
                a[t] = zero8();
            }
        }
#pragma unroll
        for (int t = 0; t < TM; t++)
#pragma unroll
            for (int u = 0; u < TN; u++) acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], b[u], acc[t][u], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
        for (int u = 0; u < TN; u++) {
            const int n = 16 * u + r;
            const float bn = bias ? bias[n] : 0.f;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int v = vbase + 16 * t + 4 * grp + i;
                if (v < nvox) {
                    float y = acc[t][u][i] + bn;
                    if (relu) y = fmaxf(y, 0.f);
                    out[(size_t)v * ocs + ooff + n] = (bf16)y;
                }
            }
        }
}

// the epilogue of the tiled convolutions: D[4·group + i][r] of tile t is the
// voxel (x0 + 16·t + 4·group + i, y, z), output channel 16·u + r
template <int TM, int TN>
__device__ __forceinline__ void tile_store(const f32x4 (&acc)[TM][TN], const float *__restrict__ bias,
                                           bf16 *__restrict__ out, int ocs, int ooff, Vol g, int relu, int x0, int y,
                                           int z, int r, int grp) {
    if (y >= g.ny) return;
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
        for (int u = 0; u < TN; u++) {
            const int n = 16 * u + r;
            const float bn = bias ? bias[n] : 0.f;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int x = x0 + 16 * t + 4 * grp + i;
                if (x < g.nx) {
                    float v = acc[t][u][i] + bn;
                    if (relu) v = fmaxf(v, 0.f);
                    out[(size_t)(x + g.nx * (y + (size_t)g.ny * z)) * ocs + ooff + n] = (bf16)v;
                }
            }
        }
}

// ---------------------------------------------------------------------------
// The same convolution with the input tile staged in LDS (CIN <= 32). A block
// is 32 (x) × 4 (y) output voxels of one z-level: wave w does row y0 + w, its
// lanes r + 16·t (t < 2) the voxels x0 + 16·t + r. The block first copies the
// 34 × 6 × 3 input voxels its 27 taps read (x and y wrapped, zero planes
// outside z) into LDS, one 16-byte chunk of 8 channels per load, so each input
// voxel is read from memory about 4.8 times per output voxel instead of 27.
// The K loop, the MFMA lane layout and the epilogue are those of
// conv3_kernel; only the A fragments come from LDS.
// ---------------------------------------------------------------------------
template <int CIN, int COUT>
__global__ void __launch_bounds__(256) conv3_tile_kernel(const bf16 *__restrict__ in, const bf16 *__restrict__ wb,
                                                         const float *__restrict__ bias, bf16 *__restrict__ out,
                                                         int ocs, int ooff, Vol g, int relu) {
    constexpr int TX = 32, TY = 4, SX = TX + 2, SY = TY + 2, C8 = CIN / 8;
    constexpr int TN = COUT / 16, TM = TX / 16;
    constexpr int NCH = (27 * CIN + 31) / 32;
    static_assert(CIN % 8 == 0 && COUT % 16 == 0, "channel counts");
    __shared__ bf16x8 tile[3][SY][SX][C8];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int x0 = blockIdx.x * TX, y0 = blockIdx.y * TY, z = blockIdx.z;
    // the input tile: positions x0 − 1 … x0 + TX (wrapped); positions past
    // nx (or ny) feed no valid output and are zero, which keeps every read
    // inside the volume when the axis is shorter than the tile
    for (int e = tid; e < 3 * SY * SX * C8; e += 256) {
        const int c8 = e % C8;
        int rest = e / C8;
        const int sx = rest % SX;
        rest /= SX;
        const int sy = rest % SY, pz = rest / SY;
        const int xr = x0 + sx - 1, yr = y0 + sy - 1, zz = z + pz - 1;
        bf16x8 val = zero8();
        if (zz >= 0 && zz < g.nz && xr <= g.nx && yr <= g.ny) {
            const int xx = wrapi(xr, g.nx), yy = wrapi(yr, g.ny);
            val = *reinterpret_cast<const bf16x8 *>(in + ((size_t)(xx + g.nx * (yy + g.ny * zz)) * CIN + c8 * 8));
        }
        tile[pz][sy][sx][c8] = val;
    }
    __syncthreads();
    const int r = lane & 15, grp = lane >> 4;
    f32x4 acc[TM][TN];
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
        for (int u = 0; u < TN; u++) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int ch = 0; ch < NCH; ch++) {
        const int k0 = ch * 32 + grp * 8;
        const int tap = k0 / CIN, c8 = (k0 - tap * CIN) >> 3;
        bf16x8 b[TN];
#pragma unroll
        for (int u = 0; u < TN; u++)
            b[u] = *reinterpret_cast<const bf16x8 *>(wb + ((size_t)(k0 >> 3) * COUT + 16 * u + r) * 8);
        // the zero-padded last chunk (tap 27) indexes tap 26 and reads zeros
        const int tq = tap < 27 ? tap : 26;
        const int dx = tq % 3 - 1, dy = (tq / 3) % 3 - 1, dz = tq / 9 - 1;
        bf16x8 a[TM];
#pragma unroll
        for (int t = 0; t < TM; t++) a[t] = tap < 27 ? tile[dz + 1][wave + 1 + dy][16 * t + r + 1 + dx][c8] : zero8();
#pragma unroll
        for (int t = 0; t < TM; t++)
#pragma unroll
            for (int u = 0; u < TN; u++) acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], b[u], acc[t][u], 0, 0, 0);
    }
    tile_store<TM, TN>(acc, bias, out, ocs, ooff, g, relu, x0, y0 + wave, z, r, grp);
}

// The tiled convolution with the tile staged one slice of SW channels at a
// time, for the channel counts whose whole tile would leave room for fewer
// than three blocks per CU (48, 64, 96). With SW = 32 (39 KB of LDS) each tap
// is one K-chunk (k = tap·CIN + 32·slice + 8·group); with SW = 16 (20 KB) a
// K-chunk is two taps (groups 0-1 the even tap, 2-3 the odd one), and the
// missing 28th tap of the last chunk contributes zeros.
template <int CIN, int COUT, int SW>
__global__ void __launch_bounds__(256) conv3_slice_kernel(const bf16 *__restrict__ in, const bf16 *__restrict__ wb,
                                                          const float *__restrict__ bias, bf16 *__restrict__ out,
                                                          int ocs, int ooff, Vol g, int relu) {
    constexpr int TX = 32, TY = 4, SX = TX + 2, SY = TY + 2;
    constexpr int TN = COUT / 16, TM = TX / 16, NS = CIN / SW, C8 = SW / 8, NC = SW == 32 ? 27 : 14;
    static_assert((SW == 16 || SW == 32) && CIN % SW == 0 && COUT % 16 == 0, "channel counts");
    __shared__ bf16x8 tile[3][SY][SX][C8];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int x0 = blockIdx.x * TX, y0 = blockIdx.y * TY, z = blockIdx.z;
    const int r = lane & 15, grp = lane >> 4;
    f32x4 acc[TM][TN];
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
        for (int u = 0; u < TN; u++) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int sl = 0; sl < NS; sl++) {
        if (sl) __syncthreads();  // every wave has read the previous slice
        for (int e = tid; e < 3 * SY * SX * C8; e += 256) {
            const int c8 = e % C8;
            int rest = e / C8;
            const int sx = rest % SX;
            rest /= SX;
            const int sy = rest % SY, pz = rest / SY;
            const int xr = x0 + sx - 1, yr = y0 + sy - 1, zz = z + pz - 1;
            bf16x8 val = zero8();
            if (zz >= 0 && zz < g.nz && xr <= g.nx && yr <= g.ny) {
                const int xx = wrapi(xr, g.nx), yy = wrapi(yr, g.ny);
                val = *reinterpret_cast<const bf16x8 *>(in + ((size_t)(xx + g.nx * (yy + g.ny * zz)) * CIN + SW * sl +
                                                              c8 * 8));
            }
            tile[pz][sy][sx][c8] = val;
        }
        __syncthreads();
#pragma unroll 3
        for (int j = 0; j < NC; j++) {
            const int tap = SW == 32 ? j : 2 * j + (grp >> 1);
            const int c8 = SW == 32 ? grp : (grp & 1);
            const bool live = tap < 27;
            const int tq = live ? tap : 26;
            const int k0 = tq * CIN + SW * sl + c8 * 8;
            bf16x8 b[TN];
#pragma unroll
            for (int u = 0; u < TN; u++)
                b[u] = live ? *reinterpret_cast<const bf16x8 *>(wb + ((size_t)(k0 >> 3) * COUT + 16 * u + r) * 8)
                            : zero8();
            const int dx = tq % 3 - 1, dy = (tq / 3) % 3 - 1, dz = tq / 9 - 1;
            bf16x8 a[TM];
#pragma unroll
            for (int t = 0; t < TM; t++) a[t] = live ? tile[dz + 1][wave + 1 + dy][16 * t + r + 1 + dx][c8] : zero8();
#pragma unroll
            for (int t = 0; t < TM; t++)
#pragma unroll
                for (int u = 0; u < TN; u++)
                    acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], b[u], acc[t][u], 0, 0, 0);
        }
    }
    tile_store<TM, TN>(acc, bias, out, ocs, ooff, g, relu, x0, y0 + wave, z, r, grp);
}

// ---------------------------------------------------------------------------
// Weight and bias gradients of a 3³ convolution on MFMA:
//   dW[tap][c][n] = Σ_v in[nb(v, tap)][c] · dy[v][n],   db[n] = Σ_v dy[v][n]
// as 27 products of M = channels c, N = outputs n, K = voxels. The inputs are
// BF16 already, so BF16 products with FP32 accumulation lose nothing.
//
// K runs along x: lane group g of v_mfma_f32_16x16x32_bf16 takes the 8 voxels
// 8g .. 8g+7 of a 32-voxel row segment. Both operands are channels-last in
// memory and need 8 voxels of one channel per lane, so a thread loads 8
// voxels × 8 channels (eight 16-byte loads), transposes them in registers (a
// byte permute per dword) and writes [channel][voxel] rows of LDS. A row
// holds the 32 voxels, then the right and left neighbours at 32 and 39 (a row
// of 40 elements spreads 16-byte reads over the banks); the three dx taps of
// a fragment are funnel shifts of one 16-byte read and those two.
// A block marches y over the three z planes of a segment: four LDS slots per
// plane, so that row y + 2 is stored while rows y − 1 .. y + 1 are read, one
// barrier per row. Its waves share out the 9 (dy, dz) taps × channel tiles;
// dy's fragments are read once per row. The accumulators stay in registers
// over all of a block's rows; blocks write partials that wgrad_reduce_kernel
// adds in a fixed order. db is one more product, with ones for the channels.
//
// Bound: latency of a row's loads and its barrier (a row is 9 to 36 MFMAs per
// wave), hidden by the blocks of a CU. Measured at 128×128×64, the sum over
// the ten layers with their reductions: 19.8 ms on FP32 VALU products from
// FP32 LDS tiles and column sums of their own → 0.86 ms.
// ---------------------------------------------------------------------------
template <int CIN, int COUT, int CS>
__global__ void __launch_bounds__(256, COUT == 64 ? 1 : 2) wgrad_kernel(const bf16 *__restrict__ in, const bf16 *__restrict__ dy,
                                                    float *__restrict__ part, float *__restrict__ bpart, Vol g,
                                                    int ntx, int nyc, int yc) {
    constexpr int C8 = CS / 8, N8 = COUT / 8, CR = CS < 16 ? 16 : CS, CT = CR / 16, NT = COUT / 16, NG = 9 * CT,
                  GPW = (NG + 3) / 4, XW = 40;
    static_assert(CIN % CS == 0 && CS % 8 == 0 && COUT % 16 == 0 && 3 * C8 * 6 + N8 * 4 <= 256, "shapes");
    __shared__ __attribute__((aligned(16))) unsigned short sx[3][4][CR][XW];
    __shared__ __attribute__((aligned(16))) unsigned short sd[2][COUT][XW];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int r = lane & 15, grp = lane >> 4;
    const int slice = blockIdx.y;
    if constexpr (CS < 16) {  // the rows of absent channels
        for (int e = t; e < 3 * 4 * (CR - CS) * XW; e += 256) {
            const int x = e % XW, c = e / XW % (CR - CS), q = e / (XW * (CR - CS));
            sx[q >> 2][q & 3][CS + c][x] = 0;
        }
    }
    // this thread's part of a row step: 8 voxels × 8 channels of `in` (kind 0)
    // or dy (kind 2), or one edge voxel of `in` (kind 1)
    int kind = 3, pz = 0, xb = 0, c8 = 0;
    if (t < 3 * C8 * 4) {
        kind = 0;
        c8 = t % C8;
        xb = t / C8 % 4;
        pz = t / (C8 * 4);
    } else if (t < 3 * C8 * 6) {
        const int e = t - 3 * C8 * 4;
        kind = 1;
        c8 = e % C8;
        xb = e / C8 % 2;  // 0: left, 1: right
        pz = e / (C8 * 2);
    } else if (t < 3 * C8 * 6 + N8 * 4) {
        const int e = t - 3 * C8 * 6;
        kind = 2;
        c8 = e % N8;
        xb = e / N8;
    }
    f32x4 acc[GPW][3][NT], accb[NT];
#pragma unroll
    for (int u = 0; u < NT; u++) {
        accb[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < GPW; i++)
#pragma unroll
            for (int d = 0; d < 3; d++) acc[i][d][u] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const u32x4 ones = u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};  // eight BF16 ones
    const int ntask = ntx * nyc * g.nz;
    for (int task = blockIdx.x; task < ntask; task += gridDim.x) {
        const int x0 = task % ntx * 32, y0 = task / ntx % nyc * yc, z = task / (ntx * nyc);
        const int y1 = min(y0 + yc, g.ny);
        u32x4 v[8];
        // in's row ya (any, wrapped) of plane z + pz − 1, dy's row yd
        auto load = [&](int ya, int yd) {
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] = u32x4{0u, 0u, 0u, 0u};
            const int zz = z + pz - 1;
            const int yw = ya < 0 ? ya + g.ny : (ya >= g.ny ? ya - g.ny : ya);
            const bool zin = zz >= 0 && zz < g.nz;
            if (kind == 0 && zin) {
                const bf16 *p = in + (size_t)(g.nx * (yw + g.ny * zz)) * CIN + slice * CS + c8 * 8;
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const int xr = x0 + 8 * xb + q;  // one past the axis: the last voxel's right neighbour
                    if (xr <= g.nx) v[q] = *reinterpret_cast<const u32x4 *>(p + (size_t)wrapi(xr, g.nx) * CIN);
                }
            } else if (kind == 1 && zin) {
                const int xr = xb ? x0 + 32 : x0 - 1;
                if (xr <= g.nx)
                    v[0] = *reinterpret_cast<const u32x4 *>(in + (size_t)(wrapi(xr, g.nx) + g.nx * (yw + g.ny * zz)) * CIN +
                                                            slice * CS + c8 * 8);
            } else if (kind == 2 && yd < y1) {
                const bf16 *p = dy + (size_t)(g.nx * (yd + g.ny * z)) * COUT + c8 * 8;
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const int xr = x0 + 8 * xb + q;
                    if (xr < g.nx) v[q] = *reinterpret_cast<const u32x4 *>(p + (size_t)xr * COUT);
                }
            }
        };
        auto store = [&](int slot, int buf) {
            if (kind == 0 || kind == 2) {
                unsigned short *row = kind == 0 ? &sx[pz][slot][c8 * 8][8 * xb] : &sd[buf][c8 * 8][8 * xb];
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    const unsigned sel = (c & 1) ? 0x07060302u : 0x05040100u;
                    u32x4 o;
#pragma unroll
                    for (int d = 0; d < 4; d++) o[d] = __builtin_amdgcn_perm(v[2 * d + 1][c >> 1], v[2 * d][c >> 1], sel);
                    *reinterpret_cast<u32x4 *>(row + c * XW) = o;
                }
            } else if (kind == 1) {
                unsigned short *row = &sx[pz][slot][c8 * 8][xb ? 32 : 39];
#pragma unroll
                for (int c = 0; c < 8; c++)
                    row[c * XW] = (unsigned short)((c & 1) ? v[0][c >> 1] >> 16 : v[0][c >> 1] & 0xffffu);
            }
        };
        __syncthreads();  // the previous task's last row has been read
        // rows y0 − 1, y0, y0 + 1 in slots 0, 1, 2; dy's row y0 in buffer 0
        for (int q = 0; q < 3; q++) {
            load(y0 - 1 + q, y0);
            store(q, 0);
        }
        __syncthreads();
        for (int y = y0; y < y1; y++) {
            const int s = y - y0;
            const bool more = y + 1 < y1;
            if (more) load(y + 2, y + 1);
            bf16x8 b[NT];
#pragma unroll
            for (int u = 0; u < NT; u++)
                b[u] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(&sd[s & 1][16 * u + r][8 * grp]));
#pragma unroll
            for (int i = 0; i < GPW; i++) {
                const int gi = wave + 4 * i;
                if (gi < NG) {
                    const int yz = gi / CT, ct = gi % CT;
                    const unsigned short *row = &sx[yz / 3][(s + yz % 3) & 3][16 * ct + r][0];
                    const u32x4 m = *reinterpret_cast<const u32x4 *>(row + 8 * grp);
                    const unsigned lf = row[grp ? 8 * grp - 1 : 39], rt = row[8 * grp + 8];
                    const unsigned e1 = __builtin_amdgcn_alignbit(m[1], m[0], 16),
                                   e2 = __builtin_amdgcn_alignbit(m[2], m[1], 16),
                                   e3 = __builtin_amdgcn_alignbit(m[3], m[2], 16);
                    const bf16x8 a0 = __builtin_bit_cast(bf16x8, u32x4{(m[0] << 16) | lf, e1, e2, e3});
                    const bf16x8 a1 = __builtin_bit_cast(bf16x8, m);
                    const bf16x8 a2 = __builtin_bit_cast(bf16x8, u32x4{e1, e2, e3, (m[3] >> 16) | (rt << 16)});
#pragma unroll
                    for (int u = 0; u < NT; u++) {
                        acc[i][0][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b[u], acc[i][0][u], 0, 0, 0);
                        acc[i][1][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b[u], acc[i][1][u], 0, 0, 0);
                        acc[i][2][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, b[u], acc[i][2][u], 0, 0, 0);
                    }
                }
            }
            if (wave == 3 && slice == 0) {
#pragma unroll
                for (int u = 0; u < NT; u++)
                    accb[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ones), b[u], accb[u], 0, 0, 0);
            }
            if (more) {
                store((s + 3) & 3, (s + 1) & 1);
                __syncthreads();
            }
        }
    }
    // D[4·group + i][r]: channel 16·ct + 4·group + i, output 16·u + r
    float *p = part + (size_t)(slice * gridDim.x + blockIdx.x) * (27 * CS * COUT);
#pragma unroll
    for (int i = 0; i < GPW; i++) {
        const int gi = wave + 4 * i;
        if (gi < NG) {
            const int yz = gi / CT, ct = gi % CT;
#pragma unroll
            for (int d = 0; d < 3; d++)
#pragma unroll
                for (int u = 0; u < NT; u++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const int c = 16 * ct + 4 * grp + q;
                        if (CS >= 16 || c < CS) p[((size_t)(3 * yz + d) * CS + c) * COUT + 16 * u + r] = acc[i][d][u][q];
                    }
        }
    }
    if (wave == 3 && slice == 0 && grp == 0) {
#pragma unroll
        for (int u = 0; u < NT; u++) bpart[(size_t)blockIdx.x * COUT + 16 * u + r] = accb[u][0];
    }
}

// grad[tap][c][n] (c < cin, the logical input channels; cs per slice) and
// bias[n]: the sums of the nblk partials of each. A block does 16 sums, 16
// threads each over a contiguous share of the partials (FP64), then the
// shares in order.
__global__ void __launch_bounds__(256) wgrad_reduce_kernel(const float *__restrict__ part,
                                                           const float *__restrict__ bpart, float *__restrict__ grad,
                                                           float *__restrict__ bias, int nblk, int cs, int cin,
                                                           int cout) {
    __shared__ double sh[16][16];
    const int ei = threadIdx.x & 15, seg = threadIdx.x >> 4;
    const int e = blockIdx.x * 16 + ei, per = cin * cout, nw = 27 * per;
    double s = 0.0;
    if (e < nw + cout) {
        const float *p = bpart + (e - nw);
        size_t stride = cout;
        if (e < nw) {
            const int tap = e / per, rem = e - tap * per, c = rem / cout, n = rem - c * cout;
            stride = (size_t)27 * cs * cout;
            p = part + (size_t)(c / cs) * nblk * stride + ((size_t)tap * cs + c % cs) * cout + n;
        }
        const int b1 = nblk * (seg + 1) / 16;
#pragma unroll 4
        for (int b = nblk * seg / 16; b < b1; b++) s += (double)p[(size_t)b * stride];
    }
    sh[seg][ei] = s;
    __syncthreads();
    if (seg == 0 && e < nw + cout) {
        for (int q = 1; q < 16; q++) s += sh[q][ei];
        if (e < nw) grad[e] = (float)s;
        else bias[e - nw] = (float)s;
    }
}

// ---------------------------------------------------------------------------
// pooling, upsampling, skips and ReLU masks
// ---------------------------------------------------------------------------
// coarse voxel of fine voxel v (fine grid g)
__device__ __forceinline__ int parent_of(int v, Vol g) {
    const int nxy = g.nx * g.ny;
    const int z = v / nxy, rem = v - z * nxy, y = rem / g.nx, x = rem - y * g.nx;
    return (x >> 1) + (g.nx >> 1) * ((y >> 1) + (g.ny >> 1) * (z >> 1));
}
// fine voxel of child q (0..7) of coarse voxel p (fine grid g)
__device__ __forceinline__ int child_of(int p, int q, Vol g) {
    const int cx = g.nx >> 1, cy = g.ny >> 1;
    const int z = p / (cx * cy), rem = p - z * cx * cy, y = rem / cx, x = rem - y * cx;
    return (2 * x + (q & 1)) + g.nx * ((2 * y + ((q >> 1) & 1)) + g.ny * (2 * z + (q >> 2)));
}

// out[p][c] = mean of the 8 children in[child][ioff + c] (fine grid g).
// Grid (⌈(nx/2)·C/8 / 256⌉, ny/2, nz/2): a thread does 8 channels (16-byte
// loads and store) of one coarse voxel; C/8 is a power of two (lc8 = log2).
__global__ void pool_kernel(const bf16 *__restrict__ in, int ics, int ioff, bf16 *__restrict__ out, int C, int lc8,
                            Vol g) {
    const int cx = g.nx >> 1, cy = g.ny >> 1;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (cx << lc8)) return;
    const int x = e >> lc8, q = e & ((1 << lc8) - 1);
    const int y = blockIdx.y, z = blockIdx.z;
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const size_t v = (size_t)(2 * x + (k & 1)) +
                         (size_t)g.nx * ((2 * y + ((k >> 1) & 1)) + (size_t)g.ny * (2 * z + (k >> 2)));
        const bf16x8 a = *reinterpret_cast<const bf16x8 *>(in + v * ics + ioff + 8 * q);
#pragma unroll
        for (int i = 0; i < 8; i++) s[i] += (float)a[i];
    }
    bf16x8 o;
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = (bf16)(s[i] * 0.125f);
    const size_t p = (size_t)x + (size_t)cx * (y + (size_t)cy * z);
    *reinterpret_cast<bf16x8 *>(out + p * C + 8 * q) = o;
}
// out[v][ooff + c] = in[parent(v)][c] (fine grid g). Grid (⌈nx·C/8 / 256⌉,
// ny, nz): a thread does 8 channels (16 bytes); C/8 is a power of two
// (lc8 = log2), C, ocs and ooff are multiples of 8
__global__ void up_kernel(const bf16 *__restrict__ in, bf16 *__restrict__ out, int ocs, int ooff, int C, int lc8,
                          Vol g) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (g.nx << lc8)) return;
    const int x = e >> lc8, q = e & ((1 << lc8) - 1);
    const int y = blockIdx.y, z = blockIdx.z;
    const size_t v = (size_t)x + (size_t)g.nx * (y + (size_t)g.ny * z);
    const size_t p = (size_t)(x >> 1) + (size_t)(g.nx >> 1) * ((y >> 1) + (size_t)(g.ny >> 1) * (z >> 1));
    *reinterpret_cast<bf16x8 *>(out + v * ocs + ooff + 8 * q) = *reinterpret_cast<const bf16x8 *>(in + p * C + 8 * q);
}
// out[v][c] = y[v][yoff + c] > 0 ? gin[v][goff + c] : 0
__global__ void relu_mask_kernel(const bf16 *gin, int gcs, int goff, const bf16 *__restrict__ y, int ycs,
                                 int yoff, bf16 *out, int C, int nvox) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)nvox * C) return;
    const int v = (int)(e / C), c = (int)(e - (size_t)v * C);
    out[e] = (float)y[(size_t)v * ycs + yoff + c] > 0.f ? gin[(size_t)v * gcs + goff + c] : (bf16)0.f;
}
// the upsampling's backward with the ReLU mask of its input (coarse y [p][C]):
// out[p][c] = y[p][c] > 0 ? Σ_children gcat[child][goff + c] : 0 (fine grid g)
__global__ void up_back_kernel(const bf16 *__restrict__ gcat, int gcs, int goff, const bf16 *__restrict__ y,
                               bf16 *__restrict__ out, int C, Vol g) {
    const int nc = (g.nx >> 1) * (g.ny >> 1) * (g.nz >> 1);
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)nc * C) return;
    const int p = (int)(e / C), c = (int)(e - (size_t)p * C);
    float s = 0.f;
    for (int q = 0; q < 8; q++) s += (float)gcat[(size_t)child_of(p, q, g) * gcs + goff + c];
    out[e] = (float)y[e] > 0.f ? (bf16)s : (bf16)0.f;
}
// the skip's gradient: the pooling's backward plus the concatenation's slice,
// masked by the skip's ReLU: out[v][c] = y[v][off + c] > 0 ? gp[parent][c]/8 + gcat[v][off + c] : 0
__global__ void skip_back_kernel(const bf16 *__restrict__ gp, const bf16 *__restrict__ gcat,
                                 const bf16 *__restrict__ cat, int cs, int off, bf16 *__restrict__ out, int C, Vol g) {
    const int nf = g.nx * g.ny * g.nz;
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)nf * C) return;
    const int v = (int)(e / C), c = (int)(e - (size_t)v * C);
    const size_t s = (size_t)v * cs + off + c;
    const float gv = (float)gp[(size_t)parent_of(v, g) * C + c] * 0.125f + (float)gcat[s];
    out[e] = (float)cat[s] > 0.f ? (bf16)gv : (bf16)0.f;
}

// ---------------------------------------------------------------------------
// input, head, loss
// ---------------------------------------------------------------------------
// Σ x² per block (FP64)
__global__ void sumsq64_kernel(const double *__restrict__ x, int n, double *__restrict__ part) {
    __shared__ double sh[UB];
    double s = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) s += x[i] * x[i];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = UB / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}
// scal[0] = 1/rms (0 when the input is zero), scal[1] = rms
__global__ void rms_finalize_kernel(const double *__restrict__ part, int nb, int n, double *__restrict__ scal) {
    if (threadIdx.x != 0) return;
    double s = 0.0;
    for (int b = 0; b < nb; b++) s += part[b];
    const double rms = sqrt(s / n);
    scal[0] = rms > 0 ? 1.0 / rms : 0.0;
    scal[1] = rms;
}
// x0[v][0] = src·s, x0[v][1] = mask (when given), other channels 0
__global__ void pack_kernel(const double *__restrict__ src, const double *__restrict__ mask,
                            const double *__restrict__ scal, bf16 *__restrict__ x0, int nvox) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nvox) return;
    const double s = scal[0];
    bf16x8 o = zero8();
    o[0] = (bf16)(float)(src[v] * s);
    if (mask) o[1] = (bf16)(float)mask[v];
    *reinterpret_cast<bf16x8 *>(x0 + (size_t)v * 8) = o;
}
// out[v] = (bh + Σ_c wh[c]·a[v][c]) · rms  (FP64 output, the source's scale restored)
__global__ void head_kernel(const bf16 *__restrict__ a, const float *__restrict__ wh, const double *__restrict__ scal,
                            double *__restrict__ out, float *__restrict__ yout, int nvox) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nvox) return;
    const bf16x8 a0 = *reinterpret_cast<const bf16x8 *>(a + (size_t)v * 16);
    const bf16x8 a1 = *reinterpret_cast<const bf16x8 *>(a + (size_t)v * 16 + 8);
    float y = wh[16];
#pragma unroll
    for (int c = 0; c < 8; c++) y = fmaf(wh[c], (float)a0[c], y);
#pragma unroll
    for (int c = 0; c < 8; c++) y = fmaf(wh[8 + c], (float)a1[c], y);
    if (yout) yout[v] = y;
    if (out) out[v] = (double)y * scal[1];
}
// loss = mean((y − t·s)²); dy = 2 (y − t·s) / n; head gradients and g9 = dy·wh ⊙ (a > 0)
__global__ void __launch_bounds__(256) head_back_kernel(const float *__restrict__ y, const double *__restrict__ tgt,
                                                        const double *__restrict__ scal, const bf16 *__restrict__ a,
                                                        const float *__restrict__ wh, bf16 *__restrict__ g9,
                                                        double *__restrict__ part, int nvox) {
    // part per block: [0] Σ loss terms, [1..16] Σ dy·a[c], [17] Σ dy
    __shared__ double sh[18][256];
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    double acc[18];
    for (int q = 0; q < 18; q++) acc[q] = 0.0;
    if (v < nvox) {
        const float d = y[v] - (float)(tgt[v] * scal[0]);
        const float dy = 2.f * d / (float)nvox;
        acc[0] = (double)d * d;
        acc[17] = dy;
        bf16x8 o0 = zero8(), o1 = zero8();
        for (int c = 0; c < 16; c++) {
            const float ac = (float)a[(size_t)v * 16 + c];
            acc[1 + c] = (double)dy * ac;
            const float gv = ac > 0.f ? dy * wh[c] : 0.f;
            if (c < 8) o0[c] = (bf16)gv; else o1[c - 8] = (bf16)gv;
        }
        *reinterpret_cast<bf16x8 *>(g9 + (size_t)v * 16) = o0;
        *reinterpret_cast<bf16x8 *>(g9 + (size_t)v * 16 + 8) = o1;
    }
    for (int q = 0; q < 18; q++) sh[q][threadIdx.x] = acc[q];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w)
            for (int q = 0; q < 18; q++) sh[q][threadIdx.x] += sh[q][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x < 18) part[(size_t)blockIdx.x * 18 + threadIdx.x] = sh[threadIdx.x][0];
}
// loss (scal[2]) and the head gradients (grad: wh[16], bh): block q sums
// partial q over the nb blocks of head_back_kernel, strided over its 256
// threads, then a fixed-order tree (deterministic)
__global__ void __launch_bounds__(256) head_reduce_kernel(const double *__restrict__ part, int nb, int nvox,
                                                          double *__restrict__ scal, float *__restrict__ ghead) {
    __shared__ double sh[256];
    const int q = blockIdx.x;
    double s = 0.0;
    for (int b = threadIdx.x; b < nb; b += 256) s += part[(size_t)b * 18 + q];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    if (q == 0) scal[2] = sh[0] / nvox;
    else ghead[q - 1] = (float)sh[0];  // q-1 = 0..15: wh, 16: bh
}

// ---------------------------------------------------------------------------
// parameters: Adam and the BF16 weight layouts
// ---------------------------------------------------------------------------
__global__ void adam_kernel(float *__restrict__ w, float *__restrict__ m, float *__restrict__ v,
                            const float *__restrict__ g, int n, float lr, float b1, float b2, float c1, float c2,
                            float eps) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}
// forward B layout: wf[k/8][n][k%8], k = tap·cinp + c (c < cin, else 0; rows past 27·cinp 0)
// backward-data B layout (the flipped, transposed kernel, a conv cout → cinp):
// wt[k'/8][c][k'%8], k' = tap'·cout + n, value W[26 − tap'][c][n]
__global__ void wlayout_kernel(const float *__restrict__ W, bf16 *__restrict__ wf, bf16 *__restrict__ wt, int cin,
                               int cinp, int cout, int kf, int kt) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < kf * cout) {
        const int k = e / cout, n = e - k * cout;
        const int tap = k / cinp, c = k - tap * cinp;
        const float val = (tap < 27 && c < cin) ? W[(tap * cin + c) * cout + n] : 0.f;
        wf[((size_t)(k >> 3) * cout + n) * 8 + (k & 7)] = (bf16)val;
    }
    if (wt && e < kt * cinp) {
        const int k = e / cinp, c = e - k * cinp;
        const int tap = k / cout, n = k - tap * cout;
        const float val = (tap < 27 && c < cin) ? W[((26 - tap) * cin + c) * cout + n] : 0.f;
        wt[((size_t)(k >> 3) * cinp + c) * 8 + (k & 7)] = (bf16)val;
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct UConv {
    int cin, cinp, cout;
    size_t woff, boff;  // offsets in the FP32 parameter vector
    bf16 *wf = nullptr, *wt = nullptr;
    int kf, kt;  // K rows (padded to chunks of 32) of the two layouts
};

struct UNet {
    int nx, ny, nz, inc;
    Vol g0, g1, g2;
    int n0, n1, n2;
    UConv L[10];
    size_t nparam, headoff;
    float *W = nullptr, *G = nullptr, *M = nullptr, *V = nullptr;
    int step = 0;
    // activations (BF16, channels-last)
    bf16 *x0, *a0, *cat0, *a8, *a9, *p0, *a2, *cat1, *a6, *a7, *p1, *a4, *a5;
    // gradients
    bf16 *g0b16, *g1b16, *gcat0, *g1l, *g2l, *gcat1, *gl2a, *gl2b, *gp1, *gp0;
    float *y;           // head output (scaled space)
    double *scal;       // [0] 1/rms, [1] rms, [2] loss
    double *dpart;      // reduction partials (FP64)
    float *fpart;       // weight-gradient partials (FP32, WGRAD_PART)
};

#define UCHK(x)                                  \
    do {                                         \
        if ((x) != hipSuccess) return -2;        \
    } while (0)

static int nblk(size_t n, int b = UB) { return (int)((n + b - 1) / b); }

template <int CIN, int COUT>
static void conv_launch(hipStream_t st, const bf16 *in, const bf16 *wb, const float *bias, bf16 *out, int ocs,
                        int ooff, Vol g, int relu) {
    if constexpr (CIN == 48) {
        const dim3 grid((g.nx + 31) / 32, (g.ny + 3) / 4, g.nz);
        hipLaunchKernelGGL((conv3_slice_kernel<CIN, COUT, 16>), grid, dim3(256), 0, st, in, wb, bias, out, ocs, ooff,
                           g, relu);
    } else if constexpr (CIN <= 32) {
        // the whole LDS tile (3 · 6 · 34 · CIN · 2 bytes: 39 KB at 32 channels)
        const dim3 grid((g.nx + 31) / 32, (g.ny + 3) / 4, g.nz);
        hipLaunchKernelGGL((conv3_tile_kernel<CIN, COUT>), grid, dim3(256), 0, st, in, wb, bias, out, ocs, ooff, g,
                           relu);
    } else if constexpr (CIN % 32 == 0) {
        const dim3 grid((g.nx + 31) / 32, (g.ny + 3) / 4, g.nz);
        hipLaunchKernelGGL((conv3_slice_kernel<CIN, COUT, 32>), grid, dim3(256), 0, st, in, wb, bias, out, ocs, ooff,
                           g, relu);
    } else {
        const int nv = g.nx * g.ny * g.nz;
        hipLaunchKernelGGL((conv3_kernel<CIN, COUT>), dim3((nv + 255) / 256), dim3(256), 0, st, in, wb, bias, out, ocs,
                           ooff, g, relu);
    }
}

// dispatch on (cin, cout) to the instantiated convolutions
static int conv_run(hipStream_t st, int cin, int cout, const bf16 *in, const bf16 *wb, const float *bias, bf16 *out,
                    int ocs, int ooff, Vol g, int relu) {
#define CASE(a, b)                                                              \
    if (cin == a && cout == b) {                                                \
        conv_launch<a, b>(st, in, wb, bias, out, ocs, ooff, g, relu);           \
        return 0;                                                               \
    }
    CASE(8, 16) CASE(16, 16) CASE(16, 32) CASE(32, 32) CASE(32, 64) CASE(64, 64) CASE(96, 32) CASE(48, 16)
    CASE(32, 16) CASE(64, 32) CASE(32, 96) CASE(16, 48)
#undef CASE
    return -1;
}

// CS: the input channels of a block (with 16 or 32 the accumulators of a
// wave's taps stay within 144 registers; 48 needs 84 with 16 outputs)
// part: the partials' room; plan: takes the rows, tasks and blocks when given
constexpr size_t WGRAD_PART = (size_t)768 * (27 * 1024 + 64);  // blocks × (taps × (channels · outputs) + outputs)
template <int CIN, int COUT, int CS>
static int wgrad_launch(hipStream_t st, float *part, const bf16 *in, const bf16 *dy, Vol g, float *grad, float *bias,
                        int cin, int *plan) {
    constexpr int NS = CIN / CS;
    const int ntx = (g.nx + 31) / 32;
    // rows per block: few (a row's start costs three rows of loads) until the
    // blocks fill the chip, 256 CUs × 2
    int yc = 32;
    while (yc > 8 && (long long)ntx * g.nz * ((g.ny + yc - 1) / yc) * NS < 512) yc /= 2;
    const int nyc = (g.ny + yc - 1) / yc;
    long long nb = (long long)ntx * nyc * g.nz;
    if (nb > 768 / NS) nb = 768 / NS;
    if (plan) {
        plan[0] = yc;
        plan[1] = ntx * nyc * g.nz;
        plan[2] = (int)nb;
    }
    const size_t wpart = (size_t)NS * nb * 27 * CS * COUT;
    if (wpart + nb * COUT > WGRAD_PART) return -1;
    hipLaunchKernelGGL((wgrad_kernel<CIN, COUT, CS>), dim3((unsigned)nb, NS), dim3(256), 0, st, in, dy, part,
                       part + wpart, g, ntx, nyc, yc);
    hipLaunchKernelGGL(wgrad_reduce_kernel, dim3(nblk((size_t)27 * cin * COUT + COUT, 16)), dim3(256), 0, st, part,
                       part + wpart, grad, bias, (int)nb, CS, cin, COUT);
    return 0;
}
static int wgrad_run(hipStream_t st, float *part, int cinp, int cin, int cout, const bf16 *in, const bf16 *dy, Vol g,
                     float *grad, float *bias, int *plan = nullptr) {
#define CASE(a, b, cs) \
    if (cinp == a && cout == b) return wgrad_launch<a, b, cs>(st, part, in, dy, g, grad, bias, cin, plan);
    CASE(8, 16, 8) CASE(16, 16, 16) CASE(16, 32, 16) CASE(32, 32, 32) CASE(32, 64, 16) CASE(64, 64, 16)
    CASE(96, 32, 32) CASE(48, 16, 48)
#undef CASE
    return -1;
}

int conv3_wgrad(hipStream_t st, int cin, int cout, int nx, int ny, int nz, const void *in, const void *dy, float *dw,
                float *db, int *plan) {
    float *part = nullptr;
    if (hipMalloc(&part, WGRAD_PART * 4) != hipSuccess) return -2;
    int rc = wgrad_run(st, part, cin, cin, cout, (const bf16 *)in, (const bf16 *)dy, Vol{nx, ny, nz}, dw, db, plan);
    if (rc == 0 && (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess)) rc = -2;
    hipFree(part);
    return rc;
}

static int refresh_layouts(UNet *N, hipStream_t st) {
    for (int l = 0; l < 10; l++) {
        UConv &c = N->L[l];
        const int n = (c.kf * c.cout > c.kt * c.cinp) ? c.kf * c.cout : c.kt * c.cinp;
        hipLaunchKernelGGL(wlayout_kernel, dim3(nblk(n)), dim3(UB), 0, st, (const float *)(N->W + c.woff), c.wf, c.wt,
                           c.cin, c.cinp, c.cout, c.kf, c.kt);
    }
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

void unet_destroy(UNet *N) {
    if (!N) return;
    void *ptrs[] = {N->W, N->G, N->M, N->V, N->x0, N->a0, N->cat0, N->a8, N->a9, N->p0, N->a2, N->cat1, N->a6,
                    N->a7, N->p1, N->a4, N->a5, N->g0b16, N->g1b16, N->gcat0, N->g1l, N->g2l, N->gcat1, N->gl2a,
                    N->gl2b, N->gp1, N->gp0, N->y, N->scal, N->dpart, N->fpart};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    for (auto &c : N->L) {
        if (c.wf) (void)hipFree(c.wf);
        if (c.wt) (void)hipFree(c.wt);
    }
    delete N;
}

// He-normal initial weights from a seeded splitmix64 + Box–Muller stream, zero biases
static void init_params(UNet *N, std::vector<float> &w, uint64_t seed) {
    uint64_t s = seed ? seed : 0x9E3779B97F4A7C15ull;
    auto next = [&]() {
        uint64_t z = (s += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    };
    auto unif = [&]() { return ((next() >> 11) + 0.5) * (1.0 / 9007199254740992.0); };
    auto gauss = [&]() { return sqrt(-2.0 * log(unif())) * cos(6.283185307179586 * unif()); };
    w.assign(N->nparam, 0.f);
    for (auto &c : N->L) {
        const double sd = sqrt(2.0 / (27.0 * c.cin));
        for (size_t i = 0; i < (size_t)27 * c.cin * c.cout; i++) w[c.woff + i] = (float)(sd * gauss());
    }
    const double sdh = sqrt(1.0 / 16.0);
    for (int c = 0; c < 16; c++) w[N->headoff + c] = (float)(sdh * gauss());
}

UNet *unet_create(int nx, int ny, int nz, int inc, uint64_t seed, char *err, size_t errlen) {
    if (nx % 4 || ny % 4 || nz % 4 || nx < 4 || ny < 4 || nz < 4) {
        snprintf(err, errlen, "the U-Net needs every axis divisible by 4 (got %d x %d x %d)", nx, ny, nz);
        return nullptr;
    }
    if (inc != 1 && inc != 2) {
        snprintf(err, errlen, "in_channels must be 1 (source) or 2 (source and mask)");
        return nullptr;
    }
    // voxel indices are int (channel offsets are size_t products): nvox < 2^30
    if ((size_t)nx * ny * nz >= ((size_t)1 << 30)) {
        snprintf(err, errlen, "grid too large for the U-Net (at most 2^30 voxels)");
        return nullptr;
    }
    UNet *N = new UNet();
    N->nx = nx; N->ny = ny; N->nz = nz; N->inc = inc;
    N->g0 = Vol{nx, ny, nz}; N->g1 = Vol{nx / 2, ny / 2, nz / 2}; N->g2 = Vol{nx / 4, ny / 4, nz / 4};
    N->n0 = nx * ny * nz; N->n1 = N->n0 / 8; N->n2 = N->n1 / 8;
    const int spec[10][3] = {{inc, 8, 16}, {16, 16, 16}, {16, 16, 32}, {32, 32, 32}, {32, 32, 64},
                             {64, 64, 64}, {96, 96, 32}, {32, 32, 32}, {48, 48, 16}, {16, 16, 16}};
    size_t off = 0;
    for (int l = 0; l < 10; l++) {
        UConv &c = N->L[l];
        c.cin = spec[l][0]; c.cinp = spec[l][1]; c.cout = spec[l][2];
        c.woff = off; off += (size_t)27 * c.cin * c.cout;
        c.boff = off; off += c.cout;
        c.kf = ((27 * c.cinp + 31) / 32) * 32;
        c.kt = ((27 * c.cout + 31) / 32) * 32;
    }
    N->headoff = off;
    off += 17;
    N->nparam = off;
    bool ok = true;
    auto A = [&](void **p, size_t bytes) {
        if (hipMalloc(p, bytes) != hipSuccess) ok = false;
        else (void)zero_dev(*p, bytes);
    };
    const size_t b2 = sizeof(bf16);
    A((void **)&N->W, off * 4); A((void **)&N->G, off * 4); A((void **)&N->M, off * 4); A((void **)&N->V, off * 4);
    for (int l = 0; l < 10; l++) {
        UConv &c = N->L[l];
        A((void **)&c.wf, (size_t)c.kf * c.cout * b2);
        if (l > 0) A((void **)&c.wt, (size_t)c.kt * c.cinp * b2);
    }
    const size_t n0 = N->n0, n1 = N->n1, n2 = N->n2;
    A((void **)&N->x0, n0 * 8 * b2); A((void **)&N->a0, n0 * 16 * b2); A((void **)&N->cat0, n0 * 48 * b2);
    A((void **)&N->a8, n0 * 16 * b2); A((void **)&N->a9, n0 * 16 * b2);
    A((void **)&N->p0, n1 * 16 * b2); A((void **)&N->a2, n1 * 32 * b2); A((void **)&N->cat1, n1 * 96 * b2);
    A((void **)&N->a6, n1 * 32 * b2); A((void **)&N->a7, n1 * 32 * b2);
    A((void **)&N->p1, n2 * 32 * b2); A((void **)&N->a4, n2 * 64 * b2); A((void **)&N->a5, n2 * 64 * b2);
    A((void **)&N->g0b16, n0 * 16 * b2); A((void **)&N->g1b16, n0 * 16 * b2); A((void **)&N->gcat0, n0 * 48 * b2);
    A((void **)&N->g1l, n1 * 32 * b2); A((void **)&N->g2l, n1 * 32 * b2); A((void **)&N->gcat1, n1 * 96 * b2);
    A((void **)&N->gl2a, n2 * 64 * b2); A((void **)&N->gl2b, n2 * 64 * b2); A((void **)&N->gp1, n2 * 32 * b2);
    A((void **)&N->gp0, n1 * 16 * b2);
    A((void **)&N->y, n0 * 4);
    A((void **)&N->scal, 8 * 8);
    const int nbh = nblk(n0);
    A((void **)&N->dpart, (size_t)(nbh > 4096 ? nbh : 4096) * 18 * 8);
    A((void **)&N->fpart, WGRAD_PART * 4);
    if (!ok) {
        snprintf(err, errlen, "hipMalloc failed for the U-Net buffers");
        unet_destroy(N);
        return nullptr;
    }
    std::vector<float> w;
    init_params(N, w, seed);
    if (upload_dev(N->W, w.data(), off * 4) != hipSuccess || refresh_layouts(N, 0) != 0 ||
        hipDeviceSynchronize() != hipSuccess) {
        snprintf(err, errlen, "U-Net initialisation failed");
        unet_destroy(N);
        return nullptr;
    }
    return N;
}

size_t unet_num_params(const UNet *N) { return N->nparam; }
int unet_dims_match(const UNet *N, int nx, int ny, int nz) { return N->nx == nx && N->ny == ny && N->nz == nz; }
int unet_get_params(UNet *N, float *host) {
    return hipMemcpy(host, N->W, N->nparam * 4, hipMemcpyDeviceToHost) == hipSuccess ? 0 : -2;
}
int unet_set_params(UNet *N, hipStream_t st, const float *host) {
    if (upload_dev(N->W, host, N->nparam * 4) != hipSuccess) return -2;
    (void)zero_dev(N->M, N->nparam * 4);
    (void)zero_dev(N->V, N->nparam * 4);
    N->step = 0;
    return refresh_layouts(N, st);
}

// the forward pass; the source's RMS into scal, the head output into N->y and (if out) out
int unet_forward(UNet *N, hipStream_t st, const double *src, const double *mask, double *out) {
    const int n0 = N->n0;
    hipLaunchKernelGGL(sumsq64_kernel, dim3(256), dim3(UB), 0, st, src, n0, N->dpart);
    hipLaunchKernelGGL(rms_finalize_kernel, dim3(1), dim3(64), 0, st, N->dpart, 256, n0, N->scal);
    hipLaunchKernelGGL(pack_kernel, dim3(nblk(n0)), dim3(UB), 0, st, src, N->inc == 2 ? mask : nullptr, N->scal, N->x0,
                       n0);
    UConv *L = N->L;
    const float *W = N->W;
    int rc = 0;
    rc |= conv_run(st, 8, 16, N->x0, L[0].wf, W + L[0].boff, N->a0, 16, 0, N->g0, 1);
    rc |= conv_run(st, 16, 16, N->a0, L[1].wf, W + L[1].boff, N->cat0, 48, 32, N->g0, 1);  // skip0
    hipLaunchKernelGGL(pool_kernel, dim3(nblk((size_t)(N->g0.nx / 2) * 2), N->g0.ny / 2, N->g0.nz / 2), dim3(UB), 0, st,
                       N->cat0, 48, 32, N->p0, 16, 1, N->g0);
    rc |= conv_run(st, 16, 32, N->p0, L[2].wf, W + L[2].boff, N->a2, 32, 0, N->g1, 1);
    rc |= conv_run(st, 32, 32, N->a2, L[3].wf, W + L[3].boff, N->cat1, 96, 64, N->g1, 1);  // skip1
    hipLaunchKernelGGL(pool_kernel, dim3(nblk((size_t)(N->g1.nx / 2) * 4), N->g1.ny / 2, N->g1.nz / 2), dim3(UB), 0, st,
                       N->cat1, 96, 64, N->p1, 32, 2, N->g1);
    rc |= conv_run(st, 32, 64, N->p1, L[4].wf, W + L[4].boff, N->a4, 64, 0, N->g2, 1);
    rc |= conv_run(st, 64, 64, N->a4, L[5].wf, W + L[5].boff, N->a5, 64, 0, N->g2, 1);
    static_assert(64 % 8 == 0 && 96 % 8 == 0 && 32 % 8 == 0 && 48 % 8 == 0, "up_kernel moves 8 channels");
    hipLaunchKernelGGL(up_kernel, dim3(nblk((size_t)N->g1.nx * 8), N->g1.ny, N->g1.nz), dim3(UB), 0, st, N->a5, N->cat1,
                       96, 0, 64, 3, N->g1);
    rc |= conv_run(st, 96, 32, N->cat1, L[6].wf, W + L[6].boff, N->a6, 32, 0, N->g1, 1);
    rc |= conv_run(st, 32, 32, N->a6, L[7].wf, W + L[7].boff, N->a7, 32, 0, N->g1, 1);
    hipLaunchKernelGGL(up_kernel, dim3(nblk((size_t)N->g0.nx * 4), N->g0.ny, N->g0.nz), dim3(UB), 0, st, N->a7, N->cat0,
                       48, 0, 32, 2, N->g0);
    rc |= conv_run(st, 48, 16, N->cat0, L[8].wf, W + L[8].boff, N->a8, 16, 0, N->g0, 1);
    rc |= conv_run(st, 16, 16, N->a8, L[9].wf, W + L[9].boff, N->a9, 16, 0, N->g0, 1);
    hipLaunchKernelGGL(head_kernel, dim3(nblk(n0)), dim3(UB), 0, st, N->a9, W + N->headoff, N->scal, out, N->y, n0);
    return rc ? -1 : (hipGetLastError() == hipSuccess ? 0 : -2);
}

// the loss of one sample and the gradient of every parameter into N->G
int unet_backward(UNet *N, hipStream_t st, const double *target) {
    const int n0 = N->n0, n1 = N->n1, n2 = N->n2;
    UConv *L = N->L;
    float *G = N->G;
    int rc = 0;
    const int nbh = nblk(n0);
    hipLaunchKernelGGL(head_back_kernel, dim3(nbh), dim3(256), 0, st, N->y, target, N->scal, N->a9, N->W + N->headoff,
                       N->g0b16, N->dpart, n0);
    hipLaunchKernelGGL(head_reduce_kernel, dim3(18), dim3(256), 0, st, N->dpart, nbh, n0, N->scal, G + N->headoff);
    // layer 9 (16 → 16 at full resolution): g9 in g0b16
    auto layer_grads = [&](int l, const bf16 *in, const bf16 *g, Vol gv) {
        rc |= wgrad_run(st, N->fpart, L[l].cinp, L[l].cin, L[l].cout, in, g, gv, G + L[l].woff, G + L[l].boff);
    };
    layer_grads(9, N->a8, N->g0b16, N->g0);
    rc |= conv_run(st, 16, 16, N->g0b16, L[9].wt, nullptr, N->g1b16, 16, 0, N->g0, 0);
    hipLaunchKernelGGL(relu_mask_kernel, dim3(nblk((size_t)n0 * 16)), dim3(UB), 0, st, N->g1b16, 16, 0, N->a8, 16, 0,
                       N->g1b16, 16, n0);
    // layer 8 (cat0 48 → 16)
    layer_grads(8, N->cat0, N->g1b16, N->g0);
    rc |= conv_run(st, 16, 48, N->g1b16, L[8].wt, nullptr, N->gcat0, 48, 0, N->g0, 0);
    // up (a7 → cat0[0:32)) backward with a7's mask → g7 (level 1, 32)
    hipLaunchKernelGGL(up_back_kernel, dim3(nblk((size_t)n1 * 32)), dim3(UB), 0, st, N->gcat0, 48, 0, N->a7, N->g1l, 32,
                       N->g0);
    // layer 7 (32 → 32 at 1/2)
    layer_grads(7, N->a6, N->g1l, N->g1);
    rc |= conv_run(st, 32, 32, N->g1l, L[7].wt, nullptr, N->g2l, 32, 0, N->g1, 0);
    hipLaunchKernelGGL(relu_mask_kernel, dim3(nblk((size_t)n1 * 32)), dim3(UB), 0, st, N->g2l, 32, 0, N->a6, 32, 0,
                       N->g2l, 32, n1);
    // layer 6 (cat1 96 → 32)
    layer_grads(6, N->cat1, N->g2l, N->g1);
    rc |= conv_run(st, 32, 96, N->g2l, L[6].wt, nullptr, N->gcat1, 96, 0, N->g1, 0);
    // up (a5 → cat1[0:64)) backward with a5's mask → g5 (level 2, 64)
    hipLaunchKernelGGL(up_back_kernel, dim3(nblk((size_t)n2 * 64)), dim3(UB), 0, st, N->gcat1, 96, 0, N->a5, N->gl2a, 64,
                       N->g1);
    // layer 5 (64 → 64 at 1/4)
    layer_grads(5, N->a4, N->gl2a, N->g2);
    rc |= conv_run(st, 64, 64, N->gl2a, L[5].wt, nullptr, N->gl2b, 64, 0, N->g2, 0);
    hipLaunchKernelGGL(relu_mask_kernel, dim3(nblk((size_t)n2 * 64)), dim3(UB), 0, st, N->gl2b, 64, 0, N->a4, 64, 0,
                       N->gl2b, 64, n2);
    // layer 4 (p1 32 → 64)
    layer_grads(4, N->p1, N->gl2b, N->g2);
    rc |= conv_run(st, 64, 32, N->gl2b, L[4].wt, nullptr, N->gp1, 32, 0, N->g2, 0);
    // skip1: pool backward + cat1[64:96) slice, masked by skip1 → g3 (level 1, 32)
    hipLaunchKernelGGL(skip_back_kernel, dim3(nblk((size_t)n1 * 32)), dim3(UB), 0, st, N->gp1, N->gcat1, N->cat1, 96, 64,
                       N->g1l, 32, N->g1);
    // layer 3 (a2 32 → 32)
    layer_grads(3, N->a2, N->g1l, N->g1);
    rc |= conv_run(st, 32, 32, N->g1l, L[3].wt, nullptr, N->g2l, 32, 0, N->g1, 0);
    hipLaunchKernelGGL(relu_mask_kernel, dim3(nblk((size_t)n1 * 32)), dim3(UB), 0, st, N->g2l, 32, 0, N->a2, 32, 0,
                       N->g2l, 32, n1);
    // layer 2 (p0 16 → 32)
    layer_grads(2, N->p0, N->g2l, N->g1);
    rc |= conv_run(st, 32, 16, N->g2l, L[2].wt, nullptr, N->gp0, 16, 0, N->g1, 0);
    // skip0: pool backward + cat0[32:48) slice, masked by skip0 → g1 (full, 16)
    hipLaunchKernelGGL(skip_back_kernel, dim3(nblk((size_t)n0 * 16)), dim3(UB), 0, st, N->gp0, N->gcat0, N->cat0, 48, 32,
                       N->g0b16, 16, N->g0);
    // layer 1 (a0 16 → 16)
    layer_grads(1, N->a0, N->g0b16, N->g0);
    rc |= conv_run(st, 16, 16, N->g0b16, L[1].wt, nullptr, N->g1b16, 16, 0, N->g0, 0);
    hipLaunchKernelGGL(relu_mask_kernel, dim3(nblk((size_t)n0 * 16)), dim3(UB), 0, st, N->g1b16, 16, 0, N->a0, 16, 0,
                       N->g1b16, 16, n0);
    // layer 0 (x0 → 16)
    layer_grads(0, N->x0, N->g1b16, N->g0);
    return rc ? -1 : (hipGetLastError() == hipSuccess ? 0 : -2);
}

int unet_loss(UNet *N, hipStream_t st, float *loss) {
    double l = 0;
    if (hipMemcpyAsync(&l, N->scal + 2, 8, hipMemcpyDeviceToHost, st) != hipSuccess) return -2;
    if (hipStreamSynchronize(st) != hipSuccess) return -2;
    *loss = (float)l;
    return 0;
}

int unet_gradients(UNet *N, hipStream_t st, const double *src, const double *mask, const double *target,
                   float *grad_host, float *loss) {
    int rc = unet_forward(N, st, src, mask, nullptr);
    if (rc) return rc;
    rc = unet_backward(N, st, target);
    if (rc) return rc;
    if (grad_host && hipMemcpyAsync(grad_host, N->G, N->nparam * 4, hipMemcpyDeviceToHost, st) != hipSuccess) return -2;
    return unet_loss(N, st, loss);
}

int unet_train_step(UNet *N, hipStream_t st, const double *src, const double *mask, const double *target, float lr,
                    float *loss) {
    int rc = unet_forward(N, st, src, mask, nullptr);
    if (rc) return rc;
    rc = unet_backward(N, st, target);
    if (rc) return rc;
    N->step++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - powf(b1, (float)N->step), c2 = 1.f - powf(b2, (float)N->step);
    hipLaunchKernelGGL(adam_kernel, dim3(nblk(N->nparam)), dim3(UB), 0, st, N->W, N->M, N->V, (const float *)N->G,
                       (int)N->nparam, lr, b1, b2, c1, c2, 1e-8f);
    rc = refresh_layouts(N, st);
    if (rc) return rc;
    return loss ? unet_loss(N, st, loss) : 0;
}

// ---------------------------------------------------------------------------
// Flexible CG (Notay, SIAM J. Sci. Comput. 22 (2000) 1444; truncation 1) on
// the FP64 operator of a multigrid plan, with the network as initial guess
// and as (part of) the preconditioner. The network is nonlinear, so the
// preconditioner varies between iterations: the new direction is
// orthogonalised against the previous one, β = −(z·w)/(p·w) with w = A p,
// and α = (p·r)/(p·w). The operator is singular (constants): b's mean is
// removed and every z and the solution are projected to zero mean.
//   mode 0: z = N(r)
//   mode 1: z = N(r) + V(r − A N(r))   (a V-cycle on what the network leaves)
//   mode 2: z = V(r)
// ---------------------------------------------------------------------------
__global__ void fcg_sums_kernel(const double *__restrict__ a, const double *__restrict__ b,
                                const double *__restrict__ c, const double *__restrict__ d, int n,
                                double *__restrict__ part) {
    // part[blk] = (Σ a·b, Σ c·d, Σ a, Σ c)   (b or d null: 1)
    __shared__ double sh[4][UB];
    double s0 = 0, s1 = 0, s2 = 0, s3 = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const double ai = a[i], ci = c ? c[i] : 0.0;
        s0 += ai * (b ? b[i] : 1.0);
        s2 += ai;
        if (c) { s1 += ci * (d ? d[i] : 1.0); s3 += ci; }
    }
    sh[0][threadIdx.x] = s0; sh[1][threadIdx.x] = s1; sh[2][threadIdx.x] = s2; sh[3][threadIdx.x] = s3;
    __syncthreads();
    for (int w = UB / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w)
            for (int q = 0; q < 4; q++) sh[q][threadIdx.x] += sh[q][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x < 4) part[blockIdx.x * 4 + threadIdx.x] = sh[threadIdx.x][0];
}
// the four sums over nb block partials: 64 threads per component, each over
// every 64th block, then a tree in LDS (a fixed order)
__global__ void __launch_bounds__(256) fcg_finalize_kernel(const double *__restrict__ part, int nb,
                                                           double *__restrict__ out) {
    __shared__ double sh[4][64];
    const int q = threadIdx.x & 3, t = threadIdx.x >> 2;
    double s = 0;
    for (int b = t; b < nb; b += 64) s += part[b * 4 + q];
    sh[q][t] = s;
    __syncthreads();
    for (int w = 32; w > 0; w >>= 1) {
        if (t < w) sh[q][t] += sh[q][t + w];
        __syncthreads();
    }
    if (threadIdx.x < 4) out[threadIdx.x] = sh[threadIdx.x][0];
}
// y = a·x + b·y − m   (x may be null: y = b·y − m)
__global__ void fcg_axpby_kernel(double *__restrict__ y, const double *__restrict__ x, double a, double b, double m,
                                 int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    y[i] = (x ? a * x[i] : 0.0) + b * y[i] - m;
}
// x += α p; r −= α w
__global__ void fcg_update_kernel(double *__restrict__ x, double *__restrict__ r, const double *__restrict__ p,
                                  const double *__restrict__ w, double alpha, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    x[i] += alpha * p[i];
    r[i] -= alpha * w[i];
}

struct FCGState {
    int n = 0;
    FCGOp op;  // the operator A (default: the multigrid plan's fine operator)
    double *b = nullptr, *x = nullptr, *r = nullptr, *z = nullptr, *p = nullptr, *w = nullptr, *t = nullptr;
    double *part = nullptr, *sc = nullptr;
};

FCGState *fcg_create(int n, FCGOp op) {
    FCGState *F = new FCGState();
    F->n = n;
    F->op = op;
    bool ok = true;
    for (double **q : {&F->b, &F->x, &F->r, &F->z, &F->p, &F->w, &F->t})
        if (hipMalloc(q, sizeof(double) * n) != hipSuccess) ok = false;
    if (hipMalloc(&F->part, sizeof(double) * 4 * 1024) != hipSuccess) ok = false;
    if (hipMalloc(&F->sc, sizeof(double) * 4) != hipSuccess) ok = false;
    if (!ok) {
        fcg_destroy(F);
        return nullptr;
    }
    return F;
}
void fcg_destroy(FCGState *F) {
    if (!F) return;
    for (double *q : {F->b, F->x, F->r, F->z, F->p, F->w, F->t, F->part, F->sc})
        if (q) (void)hipFree(q);
    delete F;
}

// (Σ a·b, Σ c·d, Σ a, Σ c) to the host
static void fcg_sums(FCGState *F, hipStream_t st, const double *a, const double *b, const double *c, const double *d,
                     double out[4]) {
    const int nb = 1024;
    hipLaunchKernelGGL(fcg_sums_kernel, dim3(nb), dim3(UB), 0, st, a, b, c, d, F->n, F->part);
    hipLaunchKernelGGL(fcg_finalize_kernel, dim3(1), dim3(256), 0, st, F->part, nb, F->sc);
    hipMemcpyAsync(out, F->sc, sizeof(double) * 4, hipMemcpyDeviceToHost, st);
    hipStreamSynchronize(st);
}
static void fcg_project(FCGState *F, hipStream_t st, double *y) {
    double s[4];
    fcg_sums(F, st, y, nullptr, nullptr, nullptr, s);
    hipLaunchKernelGGL(fcg_axpby_kernel, dim3(nblk(F->n)), dim3(UB), 0, st, y, (const double *)nullptr, 0.0, 1.0,
                       s[2] / F->n, F->n);
}
// z = M(r), mean-free
static void fcg_apply(FCGState *F, MGPlan *P, hipStream_t st, double *out, const double *x) {
    if (F->op.apply) F->op.apply(F->op.ctx, st, out, x);
    else mg_apply(P, st, out, x);
}

static int fcg_precond(FCGState *F, MGPlan *P, UNet *N, const double *mask, int mode, hipStream_t st) {
    if (mode == 2) {
        mg_precond_apply(P, st, F->z, F->r);
    } else {
        int rc = unet_forward(N, st, F->r, mask, F->z);
        if (rc) return rc;
        if (mode == 1) {
            fcg_apply(F, P, st, F->t, F->z);  // t = A z1
            hipLaunchKernelGGL(fcg_axpby_kernel, dim3(nblk(F->n)), dim3(UB), 0, st, F->t, (const double *)F->r, 1.0,
                               -1.0, 0.0, F->n);  // t = r − A z1
            mg_precond_apply(P, st, F->t, F->t);
            hipLaunchKernelGGL(fcg_axpby_kernel, dim3(nblk(F->n)), dim3(UB), 0, st, F->z, (const double *)F->t, 1.0,
                               1.0, 0.0, F->n);  // z = z1 + V(t)
        }
    }
    fcg_project(F, st, F->z);
    return 0;
}

int fcg_solve(FCGState *F, MGPlan *P, UNet *N, const double *mask, int mode, int use_guess, hipStream_t st,
              double *xout, const double *bin, double tol, int maxit, int *iters_out, double *resid_out,
              double *bnorm_out) {
    const int n = F->n;
    const int nb = nblk(n);
    double s[4];
    // b' = b − mean(b)
    hipMemcpyAsync(F->b, bin, sizeof(double) * n, hipMemcpyDeviceToDevice, st);
    fcg_project(F, st, F->b);
    fcg_sums(F, st, F->b, F->b, nullptr, nullptr, s);
    const double bnorm = sqrt(s[0]);
    *bnorm_out = bnorm;
    if (bnorm == 0) {
        hipMemsetAsync(xout, 0, sizeof(double) * n, st);
        *iters_out = 0;
        *resid_out = 0;
        return 3;
    }
    // x0 = N(b') (projected) and r = b' − A x0, or x0 = 0 and r = b'
    if (use_guess && N) {
        int rc = unet_forward(N, st, F->b, mask, F->x);
        if (rc) return -1;
        fcg_project(F, st, F->x);
        fcg_apply(F, P, st, F->w, F->x);
        hipMemcpyAsync(F->r, F->b, sizeof(double) * n, hipMemcpyDeviceToDevice, st);
        hipLaunchKernelGGL(fcg_axpby_kernel, dim3(nb), dim3(UB), 0, st, F->r, (const double *)F->w, -1.0, 1.0, 0.0, n);
    } else {
        hipMemsetAsync(F->x, 0, sizeof(double) * n, st);
        hipMemcpyAsync(F->r, F->b, sizeof(double) * n, hipMemcpyDeviceToDevice, st);
    }
    fcg_sums(F, st, F->r, F->r, nullptr, nullptr, s);
    double rnorm = sqrt(s[0]);
    int iters = 0, status = rnorm <= tol * bnorm ? 0 : 1;
    if (status != 0) {
        if (fcg_precond(F, P, N, mask, mode, st)) return -1;
        hipMemcpyAsync(F->p, F->z, sizeof(double) * n, hipMemcpyDeviceToDevice, st);
    }
    while (status != 0 && iters < maxit) {
        fcg_apply(F, P, st, F->w, F->p);
        fcg_sums(F, st, F->p, F->w, F->p, F->r, s);  // p·w, p·r
        const double pw = s[0], pr = s[1];
        // breakdown relative to the step's numerator, as pcg!'s |p·Ap| > eps·|r·z| (issue #132)
        if (!(fabs(pw) > DBL_EPSILON * fabs(pr)) || !std::isfinite(pw)) { status = 2; break; }
        const double alpha = pr / pw;
        hipLaunchKernelGGL(fcg_update_kernel, dim3(nb), dim3(UB), 0, st, F->x, F->r, (const double *)F->p,
                           (const double *)F->w, alpha, n);
        iters++;
        fcg_sums(F, st, F->r, F->r, nullptr, nullptr, s);
        rnorm = sqrt(s[0]);
        if (rnorm <= tol * bnorm) { status = 0; break; }
        if (fcg_precond(F, P, N, mask, mode, st)) return -1;
        fcg_sums(F, st, F->z, F->w, nullptr, nullptr, s);
        const double beta = -s[0] / pw;
        hipLaunchKernelGGL(fcg_axpby_kernel, dim3(nb), dim3(UB), 0, st, F->p, (const double *)F->z, 1.0, beta, 0.0, n);
    }
    hipMemcpyAsync(xout, F->x, sizeof(double) * n, hipMemcpyDeviceToDevice, st);
    fcg_project(F, st, xout);
    *iters_out = iters;
    *resid_out = rnorm;
    return status;
}

}  // namespace aeo
